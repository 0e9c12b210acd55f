// Kernels of the KODAMA.matrix orchestration (matrix_kernels.hip): the Lloyd
// steps of the reference k-means in its own float order, and the projection of
// non-landmark rows through the global graph.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>

namespace kodama_hip {

// out[r] = dot(x_r, x_r) in the reference's float order (see matrix_kernels.hip);
// *norm_max (may be null; the caller cleared it) = their largest.
hipError_t launch_sse_norms(const float* x, int rows, int p, float* out, float* norm_max, hipStream_t s);

// Nearest centroid of every row (smallest (|x|^2 + |c|^2) - 2 x.c, first
// cluster on ties); rows whose assignment changes are counted in *changed.
// With runs > 1, `runs` problems of n rows and k clusters each, laid out one
// after another (x, x_norm, centroids, c_norm, assign, changed strided by
// problem), solved by one launch; active (may be null) skips problems whose
// entry is 0. row_op / centroid_op: score operands (knn_stream.h) of the rows
// and the centroids, Euclidean, `parts` parts, each problem's rows padded to
// pad_n (a multiple of 16) and its centroids to pad_k (a multiple of 64).
struct KmeansAssignParams {
  const float* x = nullptr;
  int n = 0, p = 0;
  const float* x_norm = nullptr;
  const float* centroids = nullptr;
  const float* c_norm = nullptr;
  int k = 0;
  int* assign = nullptr;
  int* changed = nullptr;
  const int* active = nullptr;
  const void* row_op = nullptr;
  const void* centroid_op = nullptr;
  const float* norm2_max = nullptr;  // [3]: the largest row norm, 0, 0
  const float* c_norm_max = nullptr; // largest of c_norm over all problems
  int parts = 1, pad_n = 0, pad_k = 0;
};
hipError_t launch_kmeans_assign(const KmeansAssignParams& prm, hipStream_t s, int runs = 1);

// Per cluster: member rows summed in ascending row order, then scaled by
// 1 / count (clusters without members stay zero); sizes as float counts.
// Batched as launch_kmeans_assign. Workspaces: offsets [runs x k x
// kmeans_segments(n)], members [runs x n].
int kmeans_segments(int n);
hipError_t launch_kmeans_update(const float* x, int n, int p, const int* assign, int k, int* offsets, int* members,
                                float* centroids, float* sizes, hipStream_t s, int runs = 1,
                                const int* active = nullptr);

// Entries per row of the projection's table: a power of two up to 32 runs, whole
// 64-lane groups beyond. And the most landmarks whose positions fit 16 bits.
inline int project_run_stride(int runs) {
  if (runs > 32) return (runs + 63) / 64 * 64;
  int stride = 1;
  while (stride < runs) stride *= 2;
  return stride;
}
constexpr int kProjectNarrow = 65535;
size_t project_local_bytes(int n, int runs, int max_landmarks);

struct ProjectParams {
  const int* graph = nullptr;        // [n x neighbors] 0-based ids, -1 = none
  int n = 0;
  int neighbors = 0;
  const int* landmarks = nullptr;    // per run, ascending data rows, concatenated
  const int* run_offsets = nullptr;  // [runs + 1]
  const int* clbest = nullptr;       // per landmark, same indexing as landmarks
  int runs = 0;
  int votes = 0;                     // most landmark neighbours that vote (1..64)
  int max_landmarks = 0;             // largest run's landmark count
  void* local = nullptr;             // workspace [n x run_stride], project_local_bytes: landmark position or -1
  int run_stride = 0;                // project_run_stride(runs)
  int* res = nullptr;                // [runs x n]
};

// res[r][i]: the landmark's own label, else the majority label (smallest on
// ties) of the first `votes` landmarks in row i's graph neighbours, else the
// run's first landmark label. Fills prm.local first (row and run -> position in
// the run's landmark list).
hipError_t launch_project(const ProjectParams& prm, hipStream_t s);

}  // namespace kodama_hip
