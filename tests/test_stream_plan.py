"""How a matrix-core kNN pass is cut (StreamPlan in csrc/knn_stream.h), on the
host: the candidate buffers of one launch stay within their bound for every
number of queries, train rows, neighbours and columns, and a launch covers at
least one block of queries."""
import os
import subprocess

from conftest import ROOT

PROGRAM = r"""
#include <cstdio>
#include "knn_stream.h"
using namespace kodama_hip;
int main() {
  const int rows[] = {1, 63, 64, 256, 257, 4096, 100000, 524288, 524544, 1000000, 1048832, 20000000, 2000000000};
  for (int queries : rows) for (int train : rows) for (int k : {1, 32, 33, 128}) for (int list : {8, 16}) {
    if (list == 8 && k > 32) continue;
    for (int steps = 1; steps <= kStreamMaxSteps; ++steps) {
      const StreamPlan plan(queries, train, k, list, steps);
      const bool ok = plan.slices >= 1 && plan.slices <= kStreamMaxSlices && plan.max_slices >= 1 &&
                      plan.max_slices <= kStreamMaxSlices && 32 * plan.max_slices > 2 * k &&
                      plan.query_bytes >= static_cast<size_t>(plan.slices) * stream_capacity(list) * 8 &&
                      plan.query_bytes >= static_cast<size_t>(plan.max_slices) * 128 &&
                      plan.batch() >= kStreamBlockRows && plan.batch() % kStreamBlockRows == 0 &&
                      plan.batch() * plan.query_bytes <= kStreamCandBytes;
      if (!ok) {
        std::printf("queries %d train %d k %d list %d steps %d: slices %d / %d, batch %d, %zu bytes a query\n", queries,
                    train, k, list, steps, plan.slices, plan.max_slices, plan.batch(), plan.query_bytes);
        return 1;
      }
    }
  }
  return 0;
}
"""


def test_buffers_of_a_launch_are_bounded(tmp_path):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=gnu++17", "-O1", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(os.environ.get("ROCM", "/opt/rocm"), "include"),
                    "-I", os.path.join(ROOT, "kodama_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
