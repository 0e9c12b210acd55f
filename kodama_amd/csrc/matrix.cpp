// KODAMA.matrix building blocks on the host: the reference's random streams
// (libstdc++ mt19937 / mt19937_64, std::shuffle, std::generate_canonical,
// std::sample, called in the reference's order so the draws coincide) and the
// k-means driver whose Lloyd steps run on the device (matrix_kernels.hip).
#include "matrix.h"

#include <algorithm>
#include <map>
#include <cmath>
#include <iterator>
#include <limits>
#include <numeric>
#include <stdexcept>

#include "device.h"
#include "knn_stream.h"
#include "matrix_launch.h"

namespace kodama_hip {

namespace {

// mt19937 seeded with the low 32 bits: integers by modulo, floats as
// draw / 2^32-1 in float (kodama_matrix.cpp:535-549).
class FaissStream {
 public:
  explicit FaissStream(std::uint64_t seed) : g_(static_cast<std::uint32_t>(seed)) {}
  int below(int m) { return static_cast<int>(g_() % static_cast<std::uint32_t>(m)); }
  float unit() { return static_cast<float>(g_()) / static_cast<float>(std::mt19937::max()); }

 private:
  std::mt19937 g_;
};

// Fisher-Yates from the front (kodama_matrix.cpp:551-564).
IVec seed_order(int n, std::uint64_t seed) {
  IVec order(static_cast<size_t>(n));
  std::iota(order.begin(), order.end(), 0);
  FaissStream r(seed);
  for (int i = 0; i + 1 < n; ++i) std::swap(order[i], order[i + r.below(n - i)]);
  return order;
}

// Float prefix-sum tree over the donor weights, updated in place
// (kodama_matrix.cpp:566-603): the same float additions in the same order.
class DonorTree {
 public:
  explicit DonorTree(const std::vector<float>& w) : t_(w.size() + 1, 0.0f), w_(w.size(), 0.0f) {
    for (size_t i = 0; i < w.size(); ++i) set(i, w[i]);
  }
  void set(size_t i, float v) {
    const float delta = v - w_[i];
    w_[i] = v;
    for (size_t j = i + 1; j < t_.size(); j += j & (~j + 1)) t_[j] += delta;
  }
  float total() const {
    float acc = 0.0f;
    for (size_t j = w_.size(); j > 0; j -= j & (~j + 1)) acc += t_[j];
    return acc;
  }
  // Largest prefix whose float sum stays <= target; -1 past the end.
  int find(float target) const {
    size_t pos = 0, step = 1;
    float prefix = 0.0f;
    while ((step << 1) < t_.size()) step <<= 1;
    for (; step > 0; step >>= 1) {
      const size_t nx = pos + step;
      if (nx < t_.size() && prefix + t_[nx] <= target) {
        pos = nx;
        prefix += t_[nx];
      }
    }
    return pos < w_.size() ? static_cast<int>(pos) : -1;
  }

 private:
  std::vector<float> t_, w_;
};

// Each empty cluster takes half of a donor drawn by weight max(0, size - 1)
// (the largest cluster if every weight is zero); the two centroids are pushed
// apart by a relative 1/1024 with alternating signs (kodama_matrix.cpp:605-662).
void split_empty_clusters(int rows, int p, int k, std::vector<float>& sizes, std::vector<float>& cent) {
  if (rows <= k) return;
  const float eps = 1.0f / 1024.0f;
  FaissStream r(1234u);
  std::vector<float> w(static_cast<size_t>(k));
  for (int c = 0; c < k; ++c) w[c] = std::max(0.0f, sizes[c] - 1.0f);
  DonorTree tree(w);
  for (int e = 0; e < k; ++e) {
    if (sizes[e] != 0.0f) continue;
    const float total = tree.total();
    int donor = total > 0.0f ? tree.find(r.unit() * total) : -1;
    if (donor < 0) donor = static_cast<int>(std::max_element(sizes.begin(), sizes.end()) - sizes.begin());
    float* ce = cent.data() + static_cast<size_t>(e) * p;
    float* cd = cent.data() + static_cast<size_t>(donor) * p;
    std::copy_n(cd, p, ce);
    for (int j = 0; j < p; ++j) {
      const bool even = (j & 1) == 0;
      ce[j] *= even ? 1.0f + eps : 1.0f - eps;
      cd[j] *= even ? 1.0f - eps : 1.0f + eps;
    }
    sizes[e] = sizes[donor] / 2.0f;
    sizes[donor] -= sizes[e];
    tree.set(static_cast<size_t>(e), std::max(0.0f, sizes[e] - 1.0f));
    tree.set(static_cast<size_t>(donor), std::max(0.0f, sizes[donor] - 1.0f));
  }
}

}  // namespace

namespace {

// Device state of `runs` k-means problems of n rows and k clusters: the score
// operands of the rows are made once, those of the centroids per assignment.
struct DeviceLloyd {
  const float* d_x;
  int runs, n, p, k, parts, steps, pad_n, pad_k;
  hipStream_t s;
  DeviceBuffer<float> xn, cent, cn, sizes, norm2_max;
  DeviceBuffer<int> asg, changed, offsets, members;  // changed: per run, then the largest centroid norm
  DeviceBuffer<unsigned char> row_op, cent_op;

  DeviceLloyd(const float* x, int runs_, int n_, int p_, int k_, hipStream_t stream)
      : d_x(x), runs(runs_), n(n_), p(p_), k(k_), s(stream), xn(static_cast<size_t>(runs) * n),
        cent(static_cast<size_t>(runs) * k * p), cn(static_cast<size_t>(runs) * k), sizes(cn.size()), norm2_max(3),
        asg(xn.size()), changed(static_cast<size_t>(runs) + 1),
        offsets(static_cast<size_t>(runs) * k * kmeans_segments(n)), members(xn.size()) {
    // Three FP16 parts where they are as wide as one.
    parts = stream_steps(p, 3, true) == stream_steps(p, 1, true) ? 3 : 1;
    steps = stream_steps(p, parts, true);
    pad_n = (n + 15) / 16 * 16;
    pad_k = (k + 63) / 64 * 64;
    row_op.resize(stream_operand_bytes(static_cast<size_t>(runs) * pad_n, steps));
    cent_op.resize(stream_operand_bytes(static_cast<size_t>(runs) * pad_k, steps));
    check(hipMemsetAsync(asg.get(), 0xFF, sizeof(int) * asg.size(), s), "memset");  // -1: unassigned
    check(hipMemsetAsync(norm2_max.get(), 0, 3 * sizeof(float), s), "memset");
    check(launch_sse_norms(d_x, runs * n, p, xn.get(), norm2_max.get(), s), "sse_norms launch");
    StreamOperandJob op = operand_job(d_x, xn.get(), n, pad_n);
    op.query_op = row_op.get();
    check(launch_stream_operands(op, s), "stream_operands launch");
  }
  StreamOperandJob operand_job(const float* x, const float* norm2, int rows, int pad) const {
    StreamOperandJob op;
    op.tile = 16;
    op.x = x;
    op.norm2 = norm2;
    op.norm2_max = norm2_max.get();
    op.p = p;
    op.parts = parts;
    op.euclid = 1;
    op.pad_rows = runs * pad;
    op.group_rows = rows;
    op.group_pad = pad;
    return op;
  }
  // Assignment to the centroids in `cent`; counts the changes.
  void assign(const int* active) {
    check(hipMemsetAsync(changed.get(), 0, sizeof(int) * changed.size(), s), "memset");
    float* const cn_max = reinterpret_cast<float*>(changed.get() + runs);
    check(launch_sse_norms(cent.get(), runs * k, p, cn.get(), cn_max, s), "sse_norms launch");
    StreamOperandJob op = operand_job(cent.get(), cn.get(), k, pad_k);
    op.train_op = cent_op.get();
    check(launch_stream_operands(op, s), "stream_operands launch");
    KmeansAssignParams a;
    a.x = d_x;
    a.n = n;
    a.p = p;
    a.x_norm = xn.get();
    a.centroids = cent.get();
    a.c_norm = cn.get();
    a.k = k;
    a.assign = asg.get();
    a.changed = changed.get();
    a.active = active;
    a.row_op = row_op.get();
    a.centroid_op = cent_op.get();
    a.norm2_max = norm2_max.get();
    a.c_norm_max = cn_max;
    a.parts = parts;
    a.pad_n = pad_n;
    a.pad_k = pad_k;
    check(launch_kmeans_assign(a, s, runs), "kmeans_assign launch");
  }
  void update(const int* active) {
    check(launch_kmeans_update(d_x, n, p, asg.get(), k, offsets.get(), members.get(), cent.get(), sizes.get(), s, runs,
                               active),
          "kmeans_update launch");
  }
};

// Whether split_empty_clusters would change anything.
bool has_empty(const float* sizes, int rows, int k) {
  return rows > k && std::find(sizes, sizes + k, 0.0f) != sizes + k;
}

}  // namespace

IVec device_kmeans(const float* h_x, const float* d_x, int n, int p, int k, std::mt19937_64& rng, int max_iter,
                   hipStream_t s) {
  k = std::max(1, std::min(k, n));
  const std::uint64_t kseed = rng() & 0x7fffffffULL;
  const IVec order = seed_order(n, kseed + 1u);
  std::vector<float> cent(static_cast<size_t>(k) * p), sizes(static_cast<size_t>(k));
  for (int c = 0; c < k; ++c) std::copy_n(h_x + static_cast<size_t>(order[c]) * p, p, cent.data() + static_cast<size_t>(c) * p);
  DeviceLloyd dev(d_x, 1, n, p, k, s);
  dev.cent.upload(cent.data(), cent.size(), s);
  for (int it = 0; it < std::max(1, max_iter); ++it) {
    dev.assign(nullptr);
    dev.update(nullptr);
    int changed = 0;
    dev.changed.download(&changed, 1, s);
    dev.sizes.download(sizes.data(), sizes.size(), s);
    check(hipStreamSynchronize(s), "kmeans sync");
    // The centroids stay on the device unless an empty cluster must be split.
    if (has_empty(sizes.data(), n, k)) {
      dev.cent.download(cent.data(), cent.size(), s);
      check(hipStreamSynchronize(s), "kmeans sync");
      split_empty_clusters(n, p, k, sizes, cent);
      dev.cent.upload(cent.data(), cent.size(), s);
    }
    if (changed == 0) break;
  }
  dev.assign(nullptr);
  IVec labels(static_cast<size_t>(n));
  dev.asg.download(labels.data(), labels.size(), s);
  check(hipStreamSynchronize(s), "kmeans sync");  // cent is read until here
  for (int& l : labels) ++l;
  return labels;
}

std::vector<IVec> device_kmeans_batch(const float* h_x, const int* rows, const float* d_rows, int runs, int n, int p,
                                      int k, std::vector<std::mt19937_64>& rngs, int max_iter, hipStream_t s) {
  k = std::max(1, std::min(k, n));
  const size_t kp = static_cast<size_t>(k) * p;
  std::vector<float> cent(static_cast<size_t>(runs) * kp), sizes(static_cast<size_t>(runs) * k);
#pragma omp parallel for schedule(dynamic)
  for (int r = 0; r < runs; ++r) {
    const std::uint64_t kseed = rngs[r]() & 0x7fffffffULL;
    const IVec order = seed_order(n, kseed + 1u);
    for (int c = 0; c < k; ++c) {
      const int data_row = rows[static_cast<size_t>(r) * n + order[c]];
      std::copy_n(h_x + static_cast<size_t>(data_row) * p, p, cent.data() + r * kp + static_cast<size_t>(c) * p);
    }
  }
  DeviceLloyd dev(d_rows, runs, n, p, k, s);
  DeviceBuffer<int> d_active(2 * static_cast<size_t>(runs));
  dev.cent.upload(cent.data(), cent.size(), s);
  // Phase of each problem: Lloyd rounds (assign, update, split), then one
  // final assignment with the last centroids, then done.
  enum Phase { kLoop, kFinal, kDone };
  std::vector<int> phase(static_cast<size_t>(runs), kLoop), rounds(static_cast<size_t>(runs), 0),
    act(2 * static_cast<size_t>(runs)), changed(static_cast<size_t>(runs));
  for (;;) {
    bool any = false, update = false;
    for (int r = 0; r < runs; ++r) {
      act[r] = phase[r] != kDone ? 1 : 0;
      act[runs + r] = phase[r] == kLoop ? 1 : 0;
      any = any || act[r];
      update = update || act[runs + r];
    }
    if (!any) break;
    d_active.upload(act.data(), act.size(), s);
    dev.assign(d_active.get());
    dev.changed.download(changed.data(), changed.size(), s);
    if (update) {
      dev.update(d_active.get() + runs);
      dev.sizes.download(sizes.data(), sizes.size(), s);
    }
    check(hipStreamSynchronize(s), "kmeans sync");  // act is reused
    if (update) {
      // The centroids stay on the device, but for runs with an empty cluster.
      std::vector<int> split;
      for (int r = 0; r < runs; ++r) {
        if (act[runs + r] && has_empty(sizes.data() + static_cast<size_t>(r) * k, n, k)) split.push_back(r);
      }
      for (int r : split) dev.cent.download(cent.data() + r * kp, kp, s, r * kp);
      if (!split.empty()) check(hipStreamSynchronize(s), "kmeans sync");
#pragma omp parallel for schedule(dynamic)
      for (size_t i = 0; i < split.size(); ++i) {
        const int r = split[i];
        std::vector<float> sz(sizes.begin() + static_cast<size_t>(r) * k, sizes.begin() + static_cast<size_t>(r + 1) * k);
        std::vector<float> ce(cent.begin() + r * kp, cent.begin() + (r + 1) * kp);
        split_empty_clusters(n, p, k, sz, ce);
        std::copy(ce.begin(), ce.end(), cent.begin() + r * kp);
      }
      for (int r : split) dev.cent.upload(cent.data() + r * kp, kp, s, r * kp);
    }
    for (int r = 0; r < runs; ++r) {
      if (phase[r] == kFinal) {
        phase[r] = kDone;
      } else if (phase[r] == kLoop) {
        ++rounds[r];
        if (changed[r] == 0 || rounds[r] >= std::max(1, max_iter)) phase[r] = kFinal;
      }
    }
  }
  std::vector<int> flat(static_cast<size_t>(runs) * n);
  dev.asg.download(flat.data(), flat.size(), s);
  check(hipStreamSynchronize(s), "kmeans sync");
  std::vector<IVec> labels(static_cast<size_t>(runs));
  for (int r = 0; r < runs; ++r) {
    labels[r].assign(flat.begin() + static_cast<size_t>(r) * n, flat.begin() + static_cast<size_t>(r + 1) * n);
    for (int& l : labels[r]) ++l;
  }
  return labels;
}

void index_strata(const IVec& labels, int strata, IVec& offsets, IVec& rows) {
  if (strata < 1) throw InvalidArgument("landmark strata count must be positive.");
  offsets.assign(static_cast<size_t>(strata) + 1, 0);
  for (int l : labels) {
    if (l < 1 || l > strata) throw InvalidArgument("landmark stratum label is out of range.");
    ++offsets[l];
  }
  std::partial_sum(offsets.begin(), offsets.end(), offsets.begin());
  rows.assign(labels.size(), 0);
  IVec cursor(offsets.begin(), offsets.end() - 1);
  for (size_t i = 0; i < labels.size(); ++i) rows[cursor[labels[i] - 1]++] = static_cast<int>(i);
}

IVec quota_sample_landmarks(const IVec& offsets, const IVec& rows, int target, std::mt19937_64& rng) {
  const int total = static_cast<int>(rows.size());
  target = std::max(1, std::min(target, total));
  const int strata = static_cast<int>(offsets.size()) - 1;
  // Proportional quotas: floor of target * count / total (long double), the
  // fractions kept for the residual slots.
  IVec quota(static_cast<size_t>(strata), 0), live;
  std::vector<long double> rest(static_cast<size_t>(strata), 0.0L);
  int given = 0;
  for (int st = 0; st < strata; ++st) {
    const int count = offsets[st + 1] - offsets[st];
    if (count <= 0) continue;
    live.push_back(st);
    const long double share =
      static_cast<long double>(target) * static_cast<long double>(count) / static_cast<long double>(total);
    quota[st] = std::min(count, static_cast<int>(std::floor(share)));
    rest[st] = share - static_cast<long double>(quota[st]);
    given += quota[st];
  }
  std::shuffle(live.begin(), live.end(), rng);
  const int residual = target - given;
  if (residual > 0) {
    // Systematic draw: one uniform offset, then every unit step of the running
    // fraction sum over the shuffled strata takes one more row.
    const long double start = std::generate_canonical<long double, 64>(rng);
    long double running = 0.0L;
    int taken = 0;
    std::vector<char> bumped(static_cast<size_t>(strata), 0);
    for (int st : live) {
      running += rest[st];
      if (taken < residual && start + static_cast<long double>(taken) < running) {
        ++quota[st];
        bumped[st] = 1;
        ++taken;
      }
    }
    // A last boundary lost to rounding goes to the largest remaining fraction.
    while (taken < residual) {
      int pick = -1;
      long double best = -1.0L;
      for (int st : live) {
        if (!bumped[st] && rest[st] > best) {
          best = rest[st];
          pick = st;
        }
      }
      if (pick < 0) throw DeviceError("landmark quota allocation could not be completed.");
      ++quota[pick];
      bumped[pick] = 1;
      ++taken;
    }
  }
  IVec out;
  out.reserve(static_cast<size_t>(target));
  for (int st = 0; st < strata; ++st) {
    if (quota[st] <= 0) continue;
    std::sample(rows.cbegin() + offsets[st], rows.cbegin() + offsets[st + 1], std::back_inserter(out), quota[st],
                rng);
  }
  if (static_cast<int>(out.size()) != target) throw DeviceError("landmark quota allocation gave the wrong size.");
  std::sort(out.begin(), out.end());
  return out;
}

IVec normalize_constrain(const int32_t* constrain, int n) {
  IVec out(static_cast<size_t>(n));
  if (constrain == nullptr) {
    std::iota(out.begin(), out.end(), 1);
    return out;
  }
  std::map<int, int> ids;
  for (int i = 0; i < n; ++i) out[i] = ids.emplace(constrain[i], static_cast<int>(ids.size()) + 1).first->second;
  return out;
}

bool is_identity_constrain(const IVec& groups) {
  for (size_t i = 0; i < groups.size(); ++i) {
    if (groups[i] != static_cast<int>(i + 1)) return false;
  }
  return true;
}

IVec factor_subset(const IVec& values, const IVec& rows) {
  std::map<int, int> ids;
  IVec out(rows.size());
  for (size_t i = 0; i < rows.size(); ++i) {
    out[i] = ids.emplace(values[rows[i]], static_cast<int>(ids.size()) + 1).first->second;
  }
  return out;
}

int majority_label(const IVec& labels) {
  std::map<int, int> counts;
  for (int v : labels) ++counts[v];
  int best = counts.begin()->first, best_n = counts.begin()->second;
  for (const auto& kv : counts) {
    if (kv.second > best_n) {  // ascending keys: a tie keeps the smaller label
      best = kv.first;
      best_n = kv.second;
    }
  }
  return best;
}

IVec constrained_majority(const IVec& labels, const IVec& groups) {
  std::map<int, IVec> members;
  for (size_t i = 0; i < labels.size(); ++i) members[groups[i]].push_back(labels[i]);
  std::map<int, int> label_of;
  for (const auto& kv : members) label_of[kv.first] = majority_label(kv.second);
  IVec out(labels.size());
  for (size_t i = 0; i < labels.size(); ++i) out[i] = label_of[groups[i]];
  return out;
}

}  // namespace kodama_hip
