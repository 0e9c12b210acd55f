// Exact kNN on device-resident rows: the host driver (knn_search.cpp) of the
// matrix-core candidates (knn_stream.h) and the register scan (launch.h), and
// the row kernels they share (knn_kernels.hip).
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <vector>

namespace kodama_hip {

// Merged lists of listed rows [count x k] (run-local ids, distances) -> the
// padded vote layout.
hipError_t launch_publish_listed(const int* idx, const float* dist, const int* qlist, const int* qrun,
                                 const int* pad_offsets, int pad_total, int count, int k, int* out_index,
                                 float* out_score, hipStream_t s);
// Rows rows[i] of src [* x p] (null: row i) -> dst, `stride` floats apart (0:
// p), zeros past p; and the inverse scatter of [count x k] results.
hipError_t launch_gather_rows(const float* src, const int* rows, int count, int p, float* dst, hipStream_t s,
                              int stride = 0);
hipError_t launch_scatter_results(const int* src_idx, const float* src_dist, const int* rows, int count, int k,
                                  int* dst_idx, float* dst_dist, hipStream_t s);

// Exact kNN of device-resident rows (internal distances, (distance, index)
// order, -1 / +inf beyond the available rows), bit-identical to the register
// scan: FP16 matrix-core candidates with the exact rerank (knn_stream.h) when
// k <= 128 and train_rows >= 4096 (beyond 64 dimensions also query_rows >=
// 1024), otherwise the register scan. Queries the first pass cannot certify
// take a second one with three operand parts and 256 candidates, and what that
// leaves the scan; *mfma_fallbacks counts those (-1: the scan ran alone).
void device_exact_knn(const float* d_train, int train_rows, const float* d_query, int query_rows, int dims, int k,
                      int metric, const int* d_exclude, int* d_idx, float* d_dist, hipStream_t s,
                      int* mfma_fallbacks = nullptr);
// Cosine rows as native_knn.cpp:1005-1035 prepares them (prepare_rows, variant
// 1): the row times 1 / sqrt of its float sum of squares in column order.
hipError_t launch_normalize_rows(float* x, int rows, int p, hipStream_t s);

// Schedule of a per-fold table build: path 1 scan, 2 matrix cores with 16 x
// `list` candidates per query and slice; 0 = by rule. `waves` is accepted and
// reported, and chooses nothing.
struct TableSchedule {
  int path = 0;
  int list = 0;
  int waves = 0;
};
void set_fold_table_schedule(const TableSchedule& t);
TableSchedule last_fold_table_schedule();

// Per-fold kNN tables of a batch of runs (precompute_knn_cv_cuda,
// core.cpp:694-782, for all runs at once) into the transposed padded vote
// layout [k x pad_total] (padded row ids, scores = minus the internal
// distance; -1 / -inf past the available rows). Two paths give identical
// tables: 1 the register scan, 2 matrix-core candidates with the exact rerank
// (the rows those cannot certify rescanned). path 0 follows the process-wide
// setting (set_fold_table_path), whose 0 chooses by the size of the largest
// run. Returns the path used.
struct FoldTableJob {
  const float* d_x = nullptr;       // prepared rows [n x p]
  int p = 0, k = 0, metric = 0;
  const int* d_rows = nullptr;      // concatenated data rows of the runs
  const int* d_folds = nullptr;     // fold of each concatenated row
  std::vector<int> run_offsets;     // host copy, [runs + 1]
  const int* d_run_offsets = nullptr;
  const int* d_pad_offsets = nullptr;
  const int* d_block_run = nullptr; // run of each 256 padded rows
  int pad_total = 0, max_rows = 0;
  int path = 0;
  int* d_nbr = nullptr;
  float* d_score = nullptr;
  int* fallbacks = nullptr;         // rows the matrix-core path rescanned (may be null)
};
int device_fold_tables(const FoldTableJob& job, hipStream_t s);
void set_fold_table_path(int path);
int fold_table_path();
int last_fold_table_path();

}  // namespace kodama_hip
