// Exact kNN through FP16 matrix-core candidates with a threshold from class maxima
// (knn_stream.hip): parameter blocks and launchers.
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstddef>

namespace kodama_hip {

constexpr int kStreamMaxSteps = 9;     // 32-deep MFMA steps per pair (operand width / 32)
constexpr int kStreamMaxK = 128;       // neighbours served
constexpr int kStreamBlockRows = 256;  // operand rows are padded to this multiple per set or run
constexpr int kStreamMerge = 512;      // candidates the rerank holds per query (all slices)
constexpr int kStreamMaxSlices = 16;

// Operand width of one pair: `parts` 1 (FP16 of the rows) or 3 (high and low
// FP16 parts, hi.hi + hi.lo + lo.hi) of p columns and, for Euclidean
// distances, the FP16 parts of -|t|^2 / 2.
inline int stream_width(int p, int parts, bool euclid) { return parts * p + (euclid ? (parts == 1 ? 2 : 3) : 0); }
inline int stream_steps(int p, int parts, bool euclid) { return (stream_width(p, parts, euclid) + 31) / 32; }
// Candidates kept per query and slice (list 8, k <= 32: 128; list 16: 256).
inline int stream_capacity(int list) { return 16 * list; }
// Queries per wave of the maxima and candidates: two 32-query tiles, one where
// the operands are wide.
inline int stream_queries_per_wave(int steps) { return steps <= 4 ? 64 : 32; }
// Slices of the maxima at least: 2.1 k class maxima place the k-th largest of
// them at about the 1.4 k-th largest score.
inline int stream_min_max_slices(int k) { return (21 * k / 10 + 31) / 32; }
// Sampled chunks for the threshold, about 1000 k rows: scoring a row twice
// costs as much as 1 / (1000 k) of an append per query, so past this many the
// appends that a longer sample saves no longer pay for it.
inline int stream_sample_chunks(int k) { return 16 * k; }

struct KnnStreamParams {
  // Rows for the exact re-score; train_stride is a multiple of 4 floats, train
  // 16-byte aligned.
  const float* train = nullptr;
  const float* query = nullptr;
  int train_stride = 0, query_stride = 0;
  const void* train_op = nullptr;   // operand fragments (launch_stream_operands)
  const void* query_op = nullptr;
  const float* query_norm2 = nullptr;  // [query rows]
  const float* norm2_max = nullptr;    // [3], see StreamNormsJob
  int train_rows = 0, query_rows = 0, dims = 0, k = 0;
  int parts = 1, euclid = 0;
  const int* exclude = nullptr;     // [query rows] train row to skip, may be null
  // Per-fold tables of a batch of runs: operands in the padded layout (each
  // run's rows start at a multiple of 256), results and rows concatenated.
  const int* block_run = nullptr;   // run of each 256 padded rows
  const int* run_offsets = nullptr;
  const int* pad_offsets = nullptr;
  const int* folds = nullptr;       // [rows], concatenated
  int pad_rows = 0;
  // For tables query_rows padded rows from query_begin on (a multiple of 256),
  // and the buffers below start at query_begin; otherwise 0.
  int query_begin = 0;
  // Class maxima: sampled 64-row chunks (all rows when at least as many),
  // dealt to max_slices workgroups per query block; 32 values per query and slice.
  int sample_chunks = 1, max_slices = 1;
  float* maxima = nullptr;          // [query rows][max_slices][32]; may share cand
  float* threshold = nullptr;       // [query rows]
  int slices = 1;                   // the candidates' train rows are cut into this many ranges
  int list = 8;                     // capacity / 16
  uint2* cand = nullptr;            // [query rows][slices][capacity] (score bits, row)
  int* cand_count = nullptr;        // [query rows][slices], -1 = overflowed
  float* cand_bound = nullptr;      // [query rows][slices] scores below it were dropped
  int* flags = nullptr;             // [query rows] 1 = needs another path; tables: [rows], concatenated
  int* out_index = nullptr;         // [query rows x k]; tables: the vote layout [k x pad_rows]
  float* out_dist = nullptr;        // internal distances; tables: scores (minus the distance)
};

// How one pass is cut: slices of the candidates and of the maxima towards eight
// workgroups per CU, at most kStreamMaxSlices of at least kStreamSliceRows
// train rows each (so a few hundred queries leave most CUs idle), and launches
// of batch() queries whose candidate buffers stay within kStreamCandBytes.
constexpr int kStreamTargetBlocks = 2048;
constexpr int kStreamSliceRows = 256;
constexpr size_t kStreamCandBytes = size_t(1) << 30;
struct StreamPlan {
  int slices, max_slices, list, k;
  size_t query_bytes;  // buffer of one query: its candidates, before them its maxima
  StreamPlan(int query_rows, int train_rows, int k_, int list_, int steps) : list(list_), k(k_) {
    const int per_block = 4 * stream_queries_per_wave(steps);
    const int blocks = (query_rows + per_block - 1) / per_block;
    const int want = std::min((kStreamTargetBlocks + blocks - 1) / blocks,
                              std::min(kStreamMaxSlices, std::max(1, train_rows / kStreamSliceRows)));
    const size_t list_bytes = static_cast<size_t>(stream_capacity(list)) * sizeof(uint2);
    const size_t fit = kStreamCandBytes / (list_bytes * blocks * per_block);
    slices = std::max(1, std::min(want, static_cast<int>(std::min<size_t>(fit, kStreamMaxSlices))));
    max_slices = std::min(kStreamMaxSlices, std::max(stream_min_max_slices(k), want));
    query_bytes = std::max(list_bytes * slices, static_cast<size_t>(max_slices) * 32 * sizeof(float));
  }
  // Query rows per launch, whole blocks of kStreamBlockRows.
  int batch() const {
    const size_t blocks = std::max<size_t>(1, kStreamCandBytes / query_bytes / kStreamBlockRows);
    return static_cast<int>(std::min<size_t>(blocks, (1 << 30) / kStreamBlockRows)) * kStreamBlockRows;
  }
  void apply(KnnStreamParams& m, unsigned char* buffer) const {
    m.slices = slices;
    m.list = list;
    m.sample_chunks = stream_sample_chunks(k);
    m.max_slices = max_slices;
    m.maxima = reinterpret_cast<float*>(buffer);  // read before the candidates are written
    m.cand = reinterpret_cast<uint2*>(buffer);
  }
};

// The operands are the rows less a centre: the error of a score grows with the
// norms, and data away from the origin would otherwise be certified by little
// but its offset. Euclidean distances do not change when every row is moved;
// inner products change by q.centre, the same for all of a query's train rows,
// when the train rows alone are. centre [p]: the mean of up to kStreamCenterRows
// rows spread evenly (any centre gives the same results), finite values only, 0
// where there is none.
constexpr int kStreamCenterRows = 1024;
hipError_t launch_stream_center(const float* x, int rows, int p, int stride, float* center, hipStream_t s);
// Squared norms [rows] of the rows less the centre and of the rows as given
// (either may be null), and their maxima. norm2_max of the searches is three
// floats that the caller clears to 0: the largest of the train rows as their
// operands have them, of the queries likewise, and (inner product) of the train
// rows as given, unless the queries are the same rows.
struct StreamNormsJob {
  const float* x = nullptr;
  int rows = 0, p = 0, stride = 0;
  const float* center = nullptr;    // [p] (null: 0)
  float* norm2 = nullptr;
  float* norm2_max = nullptr;
  float* given_norm2 = nullptr;
  float* given_norm2_max = nullptr; // may be null
};
hipError_t launch_stream_norms(const StreamNormsJob& job, hipStream_t s);
inline int stream_row_stride(int p) { return (p + 3) / 4 * 4; }
// Rows -> operand fragments of `steps` x 32 columns, rows padded with zeros to
// pad_rows; either output may be null. norm2_max scales them. `tile` rows a
// fragment: 32 (x 16 columns, v_mfma_f32_32x32x16_f16) or 16 (x 32 columns,
// v_mfma_f32_16x16x32_f16).
// For the padded table layout pass block_run / run_offsets / pad_offsets.
struct StreamOperandJob {
  const float* x = nullptr;
  int stride = 0;                   // floats between rows (0: p)
  const float* train_center = nullptr;  // [p], of the rows as train rows / as queries (null: 0)
  const float* query_center = nullptr;
  const float* norm2 = nullptr;     // Euclidean train rows: of the centred rows
  const float* norm2_max = nullptr;
  int rows = 0, p = 0, parts = 1, euclid = 0;
  int tile = 32;
  int pad_rows = 0;                 // multiple of tile
  int group_rows = 0, group_pad = 0;  // equal groups of group_rows rows, padded to group_pad (0: one group)
  const int* block_run = nullptr;   // tables: run of each 256 padded rows
  const int* run_offsets = nullptr;
  const int* pad_offsets = nullptr;
  void* train_op = nullptr;
  void* query_op = nullptr;
};
hipError_t launch_stream_operands(const StreamOperandJob& job, hipStream_t s);
inline size_t stream_operand_bytes(size_t pad_rows, int steps) { return pad_rows * steps * 64; }

// Candidates of every query, then the rerank (certified queries get their k
// nearest, the others flags = 1).
hipError_t launch_knn_stream(const KnnStreamParams& prm, hipStream_t s);

}  // namespace kodama_hip
