"""Exceptions in the parallel loops of the batch calls (csrc/loop_errors.h): the
first one comes out after the region, as a status of the call and not as the
end of the process."""
import os
import subprocess

from conftest import ROOT

CSRC = os.path.join(ROOT, "kodama_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <new>
#include <stdexcept>
#include "loop_errors.h"
int main() {
  for (int bad : {-1, 0, 37, 99}) {
    kodama_hip::LoopErrors errors;
    int done = 0;
    bool threw = false;
#pragma omp parallel for schedule(dynamic, 4) reduction(+ : done) num_threads(4)
    for (int r = 0; r < 100; ++r) {
      errors.run([&] {
        if (r == bad) throw std::bad_alloc();
        ++done;
      });
    }
    try { errors.rethrow(); } catch (const std::bad_alloc&) { threw = true; }
    if (threw != (bad >= 0) || done != (bad >= 0 ? 99 : 100)) { std::printf("%d %d %d\n", bad, threw, done); return 1; }
  }
  return 0;
}
"""


def test_the_first_exception_comes_out_after_the_loop(tmp_path):
    src, exe = tmp_path / "loop.cpp", tmp_path / "loop"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=gnu++17", "-O1", "-fopenmp", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
