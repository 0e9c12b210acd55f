// Host driver of the exact kNN on the device: matrix-core candidates with the
// exact rerank where they apply, the register scan otherwise and for the
// queries the rerank flags.
#include <algorithm>
#include <atomic>
#include <functional>
#include <vector>

#include "../../include/kodama_hip.h"
#include "device.h"
#include "knn_search.h"
#include "knn_stream.h"
#include "launch.h"

namespace kodama_hip {

namespace {

constexpr int kScanBlock = 256;          // queries per register-scan block
constexpr int kScanTargetBlocks = 512;   // two blocks per CU
constexpr int kMaxSlices = 64;           // lists one merge wave combines
constexpr int kSliceAlign = 64;          // LDS tile rows of the scan
constexpr int kTableTargetBlocks = 2048; // sliced rescans of flagged table rows
constexpr int kStreamMinTrain = 4096;     // smaller train sets use the register scan
constexpr int kStreamWideQueries = 1024;  // queries beyond 64 dimensions for the matrix cores

}  // namespace

void device_exact_knn(const float* d_train, int train_rows, const float* d_query, int query_rows, int dims, int k,
                      int metric, const int* d_exclude, int* d_idx, float* d_dist, hipStream_t s, int* mfma_fallbacks) {
  const bool euclid = metric == KODAMA_HIP_EUCLIDEAN;
  if (mfma_fallbacks) *mfma_fallbacks = -1;  // -1: the MFMA path was not used
  // Register scan. Few queries (one block per 256) would leave most CUs idle,
  // so the train rows are cut into slices scanned by separate blocks, whose
  // lists are merged after: about 512 blocks in all, at most 64 slices.
  auto scan = [&](const float* q, int rows, const int* ex, int* idx, float* dist) {
    KnnTopkParams prm;
    prm.train = d_train;
    prm.query = q;
    prm.train_rows = train_rows;
    prm.query_rows = rows;
    prm.dims = dims;
    prm.k = k;
    prm.exclude = ex;
    prm.out_index = idx;
    prm.out_dist = dist;
    const int gx = (rows + kScanBlock - 1) / kScanBlock;
    int slices = std::min(kMaxSlices, std::max(1, (kScanTargetBlocks + gx - 1) / gx));
    int slice_rows = (train_rows + slices - 1) / slices;
    slice_rows = std::max(kSliceAlign, (slice_rows + kSliceAlign - 1) / kSliceAlign * kSliceAlign);
    slices = (train_rows + slice_rows - 1) / slice_rows;
    if (slices <= 1) {
      check(launch_knn_topk(prm, 0, euclid, rows, 1, s), "knn_topk launch");
      return;
    }
    DeviceBuffer<int> part_idx(static_cast<size_t>(slices) * rows * k);
    DeviceBuffer<float> part_dist(part_idx.size());
    prm.slice_rows = slice_rows;
    prm.out_index = part_idx.get();
    prm.out_dist = part_dist.get();
    check(launch_knn_topk(prm, 0, euclid, rows, slices, s), "knn_topk launch");
    check(launch_knn_merge_slices(part_idx.get(), part_dist.get(), slices, rows, k, idx, dist, s),
          "knn_merge_slices launch");
    check(hipStreamSynchronize(s), "knn scan sync");  // the partial lists are freed on return
  };
  const int narrow = stream_steps(dims, 1, euclid);
  if (k > kStreamMaxK || train_rows < kStreamMinTrain || query_rows == 0 || narrow > kStreamMaxSteps ||
      (dims > 64 && query_rows < kStreamWideQueries)) {
    scan(d_query, query_rows, d_exclude, d_idx, d_dist);
    return;
  }
  // Matrix-core candidates in one FP16 part (three where that is as wide) and
  // the buffer the width of k needs; the queries it cannot certify take three
  // parts and the larger buffer, and only what is left the scan.
  const bool same = d_query == d_train;
  // Norms: Euclidean, of the centred rows on both sides; inner product, the
  // train rows' centred and as given, the queries' as given.
  DeviceBuffer<float> center(static_cast<size_t>(dims)), t_n2(static_cast<size_t>(train_rows)), n2_max(3);
  check(launch_stream_center(d_train, train_rows, dims, dims, center.get(), s), "stream_center launch");
  check(hipMemsetAsync(n2_max.get(), 0, 3 * sizeof(float), s), "memset");
  const float* const query_center = euclid ? center.get() : nullptr;
  StreamNormsJob tn;
  tn.x = d_train;
  tn.rows = train_rows;
  tn.p = tn.stride = dims;
  tn.center = center.get();
  tn.norm2_max = n2_max.get();
  (euclid ? tn.norm2 : tn.given_norm2) = t_n2.get();
  if (!euclid) tn.given_norm2_max = n2_max.get() + (same ? 1 : 2);
  check(launch_stream_norms(tn, s), "stream_norms launch");
  // The rerank's 16-byte loads need rows of whole ones: a padded copy where
  // the columns are not a multiple of four (0.1 ms per million rows of 50).
  const int stride = stream_row_stride(dims);
  DeviceBuffer<float> padded(stride != dims ? static_cast<size_t>(train_rows) * stride : 0);
  if (stride != dims) {
    check(launch_gather_rows(d_train, nullptr, train_rows, dims, padded.get(), s, stride), "gather_rows launch");
  }
  // One pass over `rows` queries; returns the flagged ones.
  auto pass = [&](const float* q, int rows, const int* ex, int parts, int list, bool self, int* idx, float* dist) {
    const int steps = stream_steps(dims, parts, euclid);
    const int t_pad = (train_rows + kStreamBlockRows - 1) / kStreamBlockRows * kStreamBlockRows;
    const int q_pad = (rows + kStreamBlockRows - 1) / kStreamBlockRows * kStreamBlockRows;
    DeviceBuffer<unsigned char> t_op(stream_operand_bytes(static_cast<size_t>(t_pad), steps)),
      q_op(stream_operand_bytes(static_cast<size_t>(q_pad), steps));
    DeviceBuffer<float> q_n2;
    if (!self) {
      q_n2.resize(static_cast<size_t>(rows));
      StreamNormsJob qn;
      qn.x = q;
      qn.rows = rows;
      qn.p = qn.stride = dims;
      qn.center = query_center;
      qn.norm2 = q_n2.get();
      qn.norm2_max = n2_max.get() + 1;
      check(launch_stream_norms(qn, s), "stream_norms launch");
    }
    StreamOperandJob op;
    op.x = d_train;
    op.train_center = center.get();
    op.query_center = query_center;
    op.norm2 = t_n2.get();
    op.norm2_max = n2_max.get();
    op.rows = train_rows;
    op.p = dims;
    op.parts = parts;
    op.euclid = euclid ? 1 : 0;
    op.pad_rows = t_pad;
    op.train_op = t_op.get();
    op.query_op = self ? q_op.get() : nullptr;
    check(launch_stream_operands(op, s), "stream_operands launch");
    if (!self) {
      op.x = q;
      op.norm2 = q_n2.get();
      op.rows = rows;
      op.pad_rows = q_pad;
      op.train_op = nullptr;
      op.query_op = q_op.get();
      check(launch_stream_operands(op, s), "stream_operands launch");
    }
    const StreamPlan plan(rows, train_rows, k, list, steps);
    const int batch = std::min(q_pad, plan.batch());
    DeviceBuffer<unsigned char> cand(static_cast<size_t>(batch) * plan.query_bytes);
    DeviceBuffer<float> threshold(static_cast<size_t>(batch));
    DeviceBuffer<int> count(static_cast<size_t>(batch) * plan.slices), flags(static_cast<size_t>(rows));
    DeviceBuffer<float> bound(count.size());
    KnnStreamParams m;
    m.train = stride != dims ? padded.get() : d_train;
    m.train_stride = stride;
    m.query_stride = dims;
    m.train_op = t_op.get();
    m.norm2_max = n2_max.get();
    m.train_rows = train_rows;
    m.dims = dims;
    m.k = k;
    m.parts = parts;
    m.euclid = euclid ? 1 : 0;
    plan.apply(m, cand.get());
    m.threshold = threshold.get();
    m.cand_count = count.get();
    m.cand_bound = bound.get();
    for (int q0 = 0; q0 < rows; q0 += batch) {
      m.query = q + static_cast<size_t>(q0) * dims;
      m.query_op = q_op.get() + stream_operand_bytes(static_cast<size_t>(q0), steps);
      m.query_norm2 = (self ? t_n2.get() : q_n2.get()) + q0;
      m.query_rows = std::min(batch, rows - q0);
      m.exclude = ex ? ex + q0 : nullptr;
      m.flags = flags.get() + q0;
      m.out_index = idx + static_cast<size_t>(q0) * k;
      m.out_dist = dist + static_cast<size_t>(q0) * k;
      check(launch_knn_stream(m, s), "knn_stream launch");
    }
    std::vector<int> h_flags(static_cast<size_t>(rows)), redo;
    flags.download(h_flags.data(), h_flags.size(), s);
    check(hipStreamSynchronize(s), "knn_stream sync");
    for (int i = 0; i < rows; ++i) if (h_flags[i]) redo.push_back(i);
    return redo;
  };
  const int parts = stream_steps(dims, 3, euclid) == narrow ? 3 : 1;
  const int list = k <= 32 ? 8 : 16;
  const std::vector<int> redo = pass(d_query, query_rows, d_exclude, parts, list, same, d_idx, d_dist);
  if (mfma_fallbacks) *mfma_fallbacks = static_cast<int>(redo.size());
  if (redo.empty()) return;
  // Gathers the listed rows of a query set and runs `find` on them.
  auto on_rows = [&](const std::vector<int>& list_rows, const float* q, int all, const int* ex, int* idx, float* dist,
                     const std::function<void(const float*, int, const int*, int*, float*)>& find) {
    const int nr = static_cast<int>(list_rows.size());
    DeviceBuffer<int> d_rows(static_cast<size_t>(nr)), r_idx(static_cast<size_t>(nr) * k), ex_sub;
    DeviceBuffer<float> q_sub(static_cast<size_t>(nr) * dims), r_dist(static_cast<size_t>(nr) * k);
    std::vector<int> sub;
    d_rows.upload(list_rows.data(), list_rows.size(), s);
    check(launch_gather_rows(q, d_rows.get(), nr, dims, q_sub.get(), s), "gather_rows launch");
    if (ex) {
      std::vector<int> h_ex(static_cast<size_t>(all));
      check(hipMemcpyAsync(h_ex.data(), ex, h_ex.size() * sizeof(int), hipMemcpyDeviceToHost, s), "download");
      check(hipStreamSynchronize(s), "exclusion sync");
      for (int i : list_rows) sub.push_back(h_ex[i]);
      ex_sub.resize(sub.size());
      ex_sub.upload(sub.data(), sub.size(), s);
    }
    find(q_sub.get(), nr, ex ? ex_sub.get() : nullptr, r_idx.get(), r_dist.get());
    check(launch_scatter_results(r_idx.get(), r_dist.get(), d_rows.get(), nr, k, idx, dist, s),
          "scatter_results launch");
    check(hipStreamSynchronize(s), "fallback sync");
  };
  const int wide = stream_steps(dims, 3, euclid) <= kStreamMaxSteps ? 3 : 1;
  on_rows(redo, d_query, query_rows, d_exclude, d_idx, d_dist,
          [&](const float* q, int rows, const int* ex, int* idx, float* dist) {
            if (wide == parts && list == 16) {
              scan(q, rows, ex, idx, dist);
              return;
            }
            const std::vector<int> redo2 = pass(q, rows, ex, wide, 16, false, idx, dist);
            if (mfma_fallbacks) *mfma_fallbacks = static_cast<int>(redo2.size());
            if (!redo2.empty()) on_rows(redo2, q, rows, ex, idx, dist, scan);
          });
}

namespace {

// From this many rows in the largest run the matrix-core path builds the
// tables: its ten launches cost about what the scan (a serial chain of one
// distance after the other per query) needs for so many rows.
constexpr int kTableStreamRows = 64;
// Flagged rows that rerun the tables with three operand parts and the larger
// buffers, in place of the scan.
constexpr int kTableRerunShare = 16;
std::atomic<int> g_table_path{0}, g_table_list{0}, g_table_waves{0};
thread_local TableSchedule g_last_table;

}  // namespace

void set_fold_table_path(int path) { set_fold_table_schedule(TableSchedule{path, 0, 0}); }
int fold_table_path() { return g_table_path.load(); }
int last_fold_table_path() { return g_last_table.path; }
void set_fold_table_schedule(const TableSchedule& t) {
  g_table_path.store(t.path);
  g_table_list.store(t.list);
  g_table_waves.store(t.waves);
}
TableSchedule last_fold_table_schedule() { return g_last_table; }

int device_fold_tables(const FoldTableJob& job, hipStream_t s) {
  const bool euclid = job.metric == KODAMA_HIP_EUCLIDEAN;
  if (job.fallbacks) *job.fallbacks = -1;  // -1: the register scan served every row
  const int runs = static_cast<int>(job.run_offsets.size()) - 1;
  const int total = job.run_offsets[runs];
  const int forced = g_table_list.load();
  const int narrow = stream_steps(job.p, 1, euclid);
  // A forced list of 8 leaves k > 32 to the scan.
  const bool stream_ok = narrow <= kStreamMaxSteps && job.k <= kStreamMaxK && !(forced == 8 && job.k > 32);
  int path = job.path != 0 ? job.path : g_table_path.load();
  if (path == 0) path = job.max_rows >= kTableStreamRows ? 2 : 1;
  if (path == 2 && !stream_ok) path = 1;

  KnnTopkParams scan;
  scan.train = job.d_x;
  scan.dims = job.p;
  scan.k = job.k;
  scan.rows = job.d_rows;
  scan.folds = job.d_folds;
  scan.run_offsets = job.d_run_offsets;
  scan.pad_offsets = job.d_pad_offsets;
  scan.pad_total = job.pad_total;
  scan.out_index = job.d_nbr;
  scan.out_dist = job.d_score;
  if (path == 1) {
    check(launch_knn_topk(scan, 1, euclid, job.max_rows, runs, s), "knn_topk launch");
    g_last_table = TableSchedule{1, 0, 0};
    return 1;
  }

  const int stride = stream_row_stride(job.p);
  DeviceBuffer<float> xc(static_cast<size_t>(total) * stride), center(static_cast<size_t>(job.p)),
    n2(static_cast<size_t>(total)), n2_max(3);
  DeviceBuffer<int> flags(static_cast<size_t>(total));
  check(launch_gather_rows(job.d_x, job.d_rows, total, job.p, xc.get(), s, stride), "gather_rows launch");
  // Norms and centre as in device_exact_knn for a set searched in itself.
  check(launch_stream_center(xc.get(), total, job.p, stride, center.get(), s), "stream_center launch");
  check(hipMemsetAsync(n2_max.get(), 0, 3 * sizeof(float), s), "memset");
  StreamNormsJob norms;
  norms.x = xc.get();
  norms.rows = total;
  norms.p = job.p;
  norms.stride = stride;
  norms.center = center.get();
  norms.norm2_max = n2_max.get();
  (euclid ? norms.norm2 : norms.given_norm2) = n2.get();
  if (!euclid) norms.given_norm2_max = n2_max.get() + 1;
  check(launch_stream_norms(norms, s), "stream_norms launch");
  std::vector<int> h_flags(static_cast<size_t>(total));
  auto pass = [&](int parts, int list) {
    const int steps = stream_steps(job.p, parts, euclid);
    DeviceBuffer<unsigned char> t_op(stream_operand_bytes(static_cast<size_t>(job.pad_total), steps)), q_op(t_op.size());
    StreamOperandJob op;
    op.x = xc.get();
    op.stride = stride;
    op.train_center = center.get();
    op.query_center = euclid ? center.get() : nullptr;
    op.norm2 = n2.get();
    op.norm2_max = n2_max.get();
    op.rows = total;
    op.p = job.p;
    op.parts = parts;
    op.euclid = euclid ? 1 : 0;
    op.pad_rows = job.pad_total;
    op.block_run = job.d_block_run;
    op.run_offsets = job.d_run_offsets;
    op.pad_offsets = job.d_pad_offsets;
    op.train_op = t_op.get();
    op.query_op = q_op.get();
    check(launch_stream_operands(op, s), "stream_operands launch");
    const StreamPlan plan(job.pad_total, job.max_rows, job.k, list, steps);
    const int batch = std::min(job.pad_total, plan.batch());
    DeviceBuffer<unsigned char> cand(static_cast<size_t>(batch) * plan.query_bytes);
    DeviceBuffer<int> count(static_cast<size_t>(batch) * plan.slices);
    DeviceBuffer<float> bound(count.size()), threshold(static_cast<size_t>(batch));
    KnnStreamParams m;
    m.train = m.query = xc.get();
    m.train_stride = m.query_stride = stride;
    m.train_op = t_op.get();
    m.query_op = q_op.get();
    m.query_norm2 = n2.get();
    m.norm2_max = n2_max.get();
    m.train_rows = total;
    m.dims = job.p;
    m.k = job.k;
    m.parts = parts;
    m.euclid = euclid ? 1 : 0;
    m.block_run = job.d_block_run;
    m.run_offsets = job.d_run_offsets;
    m.pad_offsets = job.d_pad_offsets;
    m.folds = job.d_folds;
    m.pad_rows = job.pad_total;
    plan.apply(m, cand.get());
    m.threshold = threshold.get();
    m.cand_count = count.get();
    m.cand_bound = bound.get();
    m.flags = flags.get();
    m.out_index = job.d_nbr;
    m.out_dist = job.d_score;
    for (m.query_begin = 0; m.query_begin < job.pad_total; m.query_begin += batch) {
      m.query_rows = std::min(batch, job.pad_total - m.query_begin);
      check(launch_knn_stream(m, s), "knn_stream launch");
    }
    flags.download(h_flags.data(), h_flags.size(), s);
    check(hipStreamSynchronize(s), "fold tables sync");
  };
  int parts = stream_steps(job.p, 3, euclid) == narrow ? 3 : 1;
  int list = forced != 0 ? forced : job.k <= 32 ? 8 : 16;
  g_last_table = TableSchedule{2, list, g_table_waves.load() != 0 ? g_table_waves.load() : 4};
  pass(parts, list);
  const long long first = std::count(h_flags.begin(), h_flags.end(), 1);
  const int wide = stream_steps(job.p, 3, euclid) <= kStreamMaxSteps ? 3 : 1;
  if (first > total / kTableRerunShare && (wide != parts || list != 16)) pass(wide, 16);

  std::vector<int> qlist, qrun, qoff(static_cast<size_t>(runs) + 1, 0);
  int max_q = 0;
  for (int r = 0; r < runs; ++r) {
    for (int i = job.run_offsets[r]; i < job.run_offsets[r + 1]; ++i) {
      if (h_flags[i]) {
        qlist.push_back(i - job.run_offsets[r]);
        qrun.push_back(r);
      }
    }
    qoff[r + 1] = static_cast<int>(qlist.size());
    max_q = std::max(max_q, qoff[r + 1] - qoff[r]);
  }
  const int nflag = static_cast<int>(qlist.size());
  if (job.fallbacks) *job.fallbacks = nflag;
  if (nflag == 0) return 2;
  DeviceBuffer<int> d_ql(qlist.size()), d_qo(qoff.size()), d_qr(qrun.size());
  d_ql.upload(qlist.data(), qlist.size(), s);
  d_qo.upload(qoff.data(), qoff.size(), s);
  d_qr.upload(qrun.data(), qrun.size(), s);
  // A few flagged rows per run would leave one block per run scanning the
  // whole run; their train rows are cut into slices (about 2048 blocks in
  // all, at most 64 slices) whose lists are merged.
  const int gx = (max_q + kScanBlock - 1) / kScanBlock;
  int slices = std::min(kMaxSlices, std::max(1, (kTableTargetBlocks + gx * runs - 1) / (gx * runs)));
  int slice_rows = (job.max_rows + slices - 1) / slices;
  slice_rows = std::max(kSliceAlign, (slice_rows + kSliceAlign - 1) / kSliceAlign * kSliceAlign);
  slices = (job.max_rows + slice_rows - 1) / slice_rows;
  scan.qlist = d_ql.get();
  scan.qlist_offsets = d_qo.get();
  if (slices <= 1) {
    check(launch_knn_topk(scan, 1, euclid, max_q, runs, s), "knn_topk launch");
    check(hipStreamSynchronize(s), "fold tables sync");
    return 2;
  }
  DeviceBuffer<int> part_idx(static_cast<size_t>(slices) * nflag * job.k), m_idx(static_cast<size_t>(nflag) * job.k);
  DeviceBuffer<float> part_dist(part_idx.size()), m_dist(m_idx.size());
  scan.list_total = nflag;
  scan.slice_rows = slice_rows;
  scan.out_index = part_idx.get();
  scan.out_dist = part_dist.get();
  check(launch_knn_topk(scan, 1, euclid, max_q, runs, s, slices), "knn_topk launch");
  check(launch_knn_merge_slices(part_idx.get(), part_dist.get(), slices, nflag, job.k, m_idx.get(), m_dist.get(), s),
        "knn_merge_slices launch");
  check(launch_publish_listed(m_idx.get(), m_dist.get(), d_ql.get(), d_qr.get(), job.d_pad_offsets, job.pad_total,
                              nflag, job.k, job.d_nbr, job.d_score, s),
        "publish_listed launch");
  check(hipStreamSynchronize(s), "fold tables sync");
  return 2;
}

}  // namespace kodama_hip
