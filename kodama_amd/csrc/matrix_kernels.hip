// KODAMA.matrix orchestration kernels for gfx950.
//
// k-means (kodama_matrix.cpp:664-799). The reference's portable x86-64 build
// computes every dot product in SSE registers without FMA
// (kodama_matrix.cpp:91-124): 16 running partials over blocks of 16 dimensions
// (each product rounded, then added), the lane sums (s[l] + s[4+l]) +
// (s[8+l] + s[12+l]), then ((l0 + l1) + l2) + l3, then the remaining
// dimensions one product at a time. The kernels keep that order. A product and
// its sum round once here, though: __fmul_rn and __fadd_rn are plain operators
// in HIP's headers, where contraction is on, and the compiler makes FMAs of
// them. So norms and distances can differ from that build in the last bit, and
// an assignment where two distances are that close; the centroid sums have no
// products and are bit-identical.
//
// kmeans_assign_kernel: the nearest centroid is the largest score q.c - |c|^2 /
// 2 up to the bound of score_device.h, so FP16 matrix-core scores pick the
// candidates (64 rows per wave as B operands, centroids through LDS 64 at a
// time, once for each row's largest score T, once to queue the pairs scoring
// at least T - 2E) and only those, about 1.3 per row, are evaluated in the
// reference's order, one pair per lane; the smallest (distance, cluster) wins
// as in the reference loop. One thread per row over every centroid was bound
// by 118 vector operations and 13 LDS reads per pair: 0.64 ms on average for
// 100k rows and 100 x 3000 rows against 300 centroids of 50 columns, now 0.07.
// kmeans_update_kernel: one workgroup per cluster, one thread per feature; the
// members come from a stable counting sort of the assignment, so they are
// added in ascending row order, the order of the reference's sequential sum,
// sixteen rows in flight. Every workgroup searching all rows for its members
// took 0.39 ms on the same shapes; the sort takes 0.10 and the sums 0.05.
//
// project_kernel: one wave per row and 64 runs, a lane per run: the position
// of each neighbour in every run's landmark list is one coalesced row of the
// table filled by local_fill_kernel and local_scatter_kernel; the votes of up
// to 64 landmark neighbours sit in the lane's LDS slice, the results leave
// through LDS as whole lines. A thread per (row, run) read the graph row once
// per run, uncoalesced: 8.2 ms for 100k rows, 100 neighbours and 100 runs.
// project_few_kernel: up to 32 runs the table has as many entries a row as the
// next power of two, and as many lanes work on a row. 64 lanes and 128 bytes a
// row for one run cost 1M rows 11 ms (and 128 MB) that the call's projection
// does not take now (74.6 -> 63.4 ms, most of it the caller's graph; 32 runs
// 77.8 -> 74.1).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "knn_stream.h"
#include "matrix_launch.h"
#include "score_device.h"

namespace kodama_hip {

namespace {

constexpr int kBlock = 256;
constexpr int kMaxVotes = 64;

// Reference-order dot of two rows.
__device__ __forceinline__ float sse_dot_rows(const float* __restrict__ a, const float* __restrict__ b, int p) {
#pragma clang fp contract(off)
  float s[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) s[j] = 0.0f;
  int i = 0;
  for (; i + 15 < p; i += 16) {
#pragma unroll
    for (int j = 0; j < 16; ++j) s[j] = __fadd_rn(s[j], __fmul_rn(a[i + j], b[i + j]));
  }
  float lane[4];
#pragma unroll
  for (int l = 0; l < 4; ++l) lane[l] = __fadd_rn(__fadd_rn(s[l], s[4 + l]), __fadd_rn(s[8 + l], s[12 + l]));
  float sum = __fadd_rn(__fadd_rn(__fadd_rn(lane[0], lane[1]), lane[2]), lane[3]);
  for (; i < p; ++i) sum = __fadd_rn(sum, __fmul_rn(a[i], b[i]));
  return sum;
}

// Reference-order squared norm of a row.
__device__ __forceinline__ float sse_norm(const float* __restrict__ a, int p) {
  float s[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) s[j] = 0.0f;
  int i = 0;
  for (; i + 15 < p; i += 16) {
#pragma unroll
    for (int j = 0; j < 16; ++j) s[j] = __fadd_rn(s[j], __fmul_rn(a[i + j], a[i + j]));
  }
  float lane[4];
#pragma unroll
  for (int l = 0; l < 4; ++l) lane[l] = __fadd_rn(__fadd_rn(s[l], s[4 + l]), __fadd_rn(s[8 + l], s[12 + l]));
  float sum = __fadd_rn(__fadd_rn(__fadd_rn(lane[0], lane[1]), lane[2]), lane[3]);
  for (; i < p; ++i) sum = __fadd_rn(sum, __fmul_rn(a[i], a[i]));
  return sum;
}

}  // namespace

// norm_max (may be null): raised to the block's largest norm (>= 0, so their
// bits order as integers; NaN excluded).
__global__ void __launch_bounds__(kBlock) sse_norms_kernel(const float* __restrict__ x, int rows, int p,
                                                            float* __restrict__ out, float* __restrict__ norm_max) {
  __shared__ uint32_t s_max;
  if (threadIdx.x == 0) s_max = 0u;
  __syncthreads();
  const int r = blockIdx.x * kBlock + threadIdx.x;
  if (r < rows) {
    const float sum = sse_norm(x + static_cast<size_t>(r) * p, p);
    out[r] = sum;
    if (sum > 0.0f) atomicMax(&s_max, __float_as_uint(sum));
  }
  __syncthreads();
  if (threadIdx.x == 0 && norm_max != nullptr && s_max != 0u) {
    atomicMax(reinterpret_cast<uint32_t*>(norm_max), s_max);
  }
}

// Roundings of the reference's (|x|^2 + |c|^2) - 2 x.c in units of its norms: 16
// block sums, 15 tail products and the lane sums, two roundings each, for the
// dot and the norms.
constexpr float kAssignRoundings = 160.0f;

// KS: 32-deep MFMA steps; NQ: 16-row tiles per wave.
template <int KS, int NQ>
__global__ void __launch_bounds__(kBlock, KS <= 8 ? 2 : 1) kmeans_assign_kernel(KmeansAssignParams prm) {
  constexpr int kWaveRows = NQ * 16;
  constexpr int kQueue = 64 + 16 * kWaveRows;  // what is left below 64, and one 16-centroid tile
  __shared__ u32x4 s_t[2][KS * kBlock];        // 64 centroids x KS x 64 bytes
  __shared__ uint32_t s_queue[4][kQueue];      // centroid << 6 | row of the wave
  __shared__ int s_n[4];
  __shared__ unsigned long long s_best[4][kWaveRows];
  // Problem blockIdx.y of a batch of equal-sized ones (rows n, clusters k).
  const int run = blockIdx.y;
  if (prm.active != nullptr && !prm.active[run]) return;  // whole block
  const int n = prm.n, p = prm.p, k = prm.k;
  const float* x = prm.x + static_cast<size_t>(run) * n * p;
  const float* x_norm = prm.x_norm + static_cast<size_t>(run) * n;
  const float* centroids = prm.centroids + static_cast<size_t>(run) * k * p;
  const float* c_norm = prm.c_norm + static_cast<size_t>(run) * k;
  int* assign = prm.assign + static_cast<size_t>(run) * n;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int grp = lane >> 4, col = lane & 15;
  const int row0 = static_cast<int>(blockIdx.x) * (4 * kWaveRows) + wave * kWaveRows;

  const u32x4* qop = reinterpret_cast<const u32x4*>(prm.row_op) +
                     (static_cast<size_t>(run) * prm.pad_n + row0) / 16 * (KS * 64) + lane;
  const u32x4* cop = reinterpret_cast<const u32x4*>(prm.centroid_op) + static_cast<size_t>(run) * prm.pad_k / 16 * (KS * 64);
  f16x8 bq[NQ][KS];
  float th[NQ];
#pragma unroll
  for (int t = 0; t < NQ; ++t) {
    const bool tile = row0 + t * 16 < n;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) bq[t][ks] = as_f16x8(tile ? qop[(t * KS + ks) * 64] : u32x4{0, 0, 0, 0});
    th[t] = -INFINITY;
  }
  if (lane < kWaveRows) s_best[wave][lane] = ~0ull;
  if (lane == 0) s_n[wave] = 0;

  // Evaluates the queued pairs, one per lane.
  auto flush = [&]() {
#pragma clang fp contract(off)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int count = __builtin_amdgcn_readfirstlane(s_n[wave]);
    for (int e = lane; e < count; e += 64) {
      const uint32_t pair = s_queue[wave][e];
      const int local = static_cast<int>(pair & 63u), c = static_cast<int>(pair >> 6);
      const float* a = x + static_cast<size_t>(row0 + local) * p;
      const float* b = centroids + static_cast<size_t>(c) * p;
      const float dist = __fsub_rn(__fadd_rn(x_norm[row0 + local], c_norm[c]), __fmul_rn(2.0f, sse_dot_rows(a, b, p)));
      if (dist < INFINITY) {
        atomicMin(&s_best[wave][local],
                  static_cast<unsigned long long>(order_key(dist)) << 32 | static_cast<unsigned long long>(c));
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) s_n[wave] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

  // Both passes over the centroids: 0 keeps the largest score, 1 queues.
  auto stream = [&](auto pass) {
    u32x4 pre[KS];
    auto fetch = [&](int c0) {
      const u32x4* src = cop + static_cast<size_t>(c0 / 16) * (KS * 64);
#pragma unroll
      for (int i = 0; i < KS; ++i) pre[i] = src[static_cast<int>(threadIdx.x) + i * kBlock];
    };
    auto store = [&](int b) {
#pragma unroll
      for (int i = 0; i < KS; ++i) s_t[b][static_cast<int>(threadIdx.x) + i * kBlock] = pre[i];
    };
    fetch(0);
    store(0);
    __builtin_amdgcn_s_waitcnt(0);  // the row operands too
    __syncthreads();
    int buf = 0;
    for (int c0 = 0; c0 < k; c0 += 64, buf ^= 1) {
      const bool more = c0 + 64 < k;
      if (more) fetch(c0 + 64);
#pragma unroll 1
      for (int sub = 0; sub < 4; ++sub) {
        f32x4 acc[NQ];
#pragma unroll
        for (int t = 0; t < NQ; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const f16x8 a = as_f16x8(s_t[buf][(sub * KS + ks) * 64 + lane]);
#pragma unroll
          for (int t = 0; t < NQ; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bq[t][ks], acc[t], 0, 0, 0);
        }
        const int c = c0 + sub * 16 + 4 * grp;  // this lane's first centroid
        if constexpr (decltype(pass)::value == 0) {
#pragma unroll
          for (int t = 0; t < NQ; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r) th[t] = fmaxf(th[t], c + r < k ? acc[t][r] : -INFINITY);
          }
        } else {
          bool any = false;
#pragma unroll
          for (int t = 0; t < NQ; ++t) {
            // Not below: a NaN score is evaluated (and never wins).
            bool hit[4];
            int count = 0;
            const bool live = row0 + t * 16 + col < n;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              hit[r] = live && c + r < k && !(acc[t][r] < th[t]);
              count += hit[r] ? 1 : 0;
            }
            if (count > 0) {
              int slot = atomicAdd(&s_n[wave], count);
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                if (hit[r]) s_queue[wave][slot++] = static_cast<uint32_t>(c + r) << 6 | static_cast<uint32_t>(t * 16 + col);
              }
            }
            any = any || count > 0;
          }
          if (__ballot(any) != 0ull) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (__builtin_amdgcn_readfirstlane(s_n[wave]) >= 64) flush();
          }
        }
      }
      if (more) store(buf ^ 1);
      __syncthreads();
    }
  };
  stream(std::integral_constant<int, 0>{});
  const float scale = operand_scale(prm.norm2_max);
  // The largest centroid of this assignment: repeated splits of one donor and
  // long float sums take centroids past the largest row. The scale is the
  // rows', and FP16 holds the norm column up to 2^15.
  const float cmax = sqrtf(*prm.c_norm_max) * scale * 1.0001f;
  const bool usable = norms_usable(prm.norm2_max) && cmax < 30000.0f;
#pragma unroll
  for (int t = 0; t < NQ; ++t) {
    float m = th[t];
    m = fmaxf(m, __shfl_xor(m, 16));
    m = fmaxf(m, __shfl_xor(m, 32));
    const int row = row0 + t * 16 + col;
    const float qn = row < n ? sqrtf(x_norm[row]) * scale * 1.0001f : 0.0f;
    const float err = pair_error(qn, cmax, p, prm.parts, prm.parts * p + 3, qn * qn + cmax * cmax, kAssignRoundings);
    th[t] = usable ? drop_bound(m, 2.0f * err) : -INFINITY;
  }
  stream(std::integral_constant<int, 1>{});
  flush();
  bool moved = false;
  const int row = row0 + lane;
  if (lane < kWaveRows && row < n) {
    const unsigned long long key = s_best[wave][lane];
    const int best = key == ~0ull ? 0 : static_cast<int>(static_cast<uint32_t>(key));
    moved = assign[row] != best;
    if (moved) assign[row] = best;
  }
  const int count = __popcll(__ballot(moved));
  if (lane == 0 && count > 0) atomicAdd(&prm.changed[run], count);
}

// Stable counting sort of the rows by cluster, in segments of 1024 rows. One
// thread per cluster reads the segment's assignment from LDS (the same address
// in every lane): PLACE = false counts into offsets[c * segments + segment],
// PLACE = true writes the members, in ascending row order, from there.
constexpr int kSegment = 1024;
template <bool PLACE>
__global__ void __launch_bounds__(kBlock) kmeans_members_kernel(const int* __restrict__ assign, int n, int k,
                                                                int* __restrict__ offsets, int* __restrict__ members,
                                                                const int* __restrict__ active) {
  __shared__ int4 s_a[kSegment / 4];
  const int run = blockIdx.y;
  if (active != nullptr && !active[run]) return;  // whole block
  const int segments = gridDim.x, seg = blockIdx.x;
  assign += static_cast<size_t>(run) * n;
  offsets += static_cast<size_t>(run) * k * segments;
  if (PLACE) members += static_cast<size_t>(run) * n;
  for (int i = threadIdx.x; i < kSegment; i += kBlock) {
    const int row = seg * kSegment + i;
    reinterpret_cast<int*>(s_a)[i] = row < n ? assign[row] : -1;
  }
  __syncthreads();
  for (int c = threadIdx.x; c < k; c += kBlock) {
    int at = PLACE ? offsets[static_cast<size_t>(c) * segments + seg] : 0;
#pragma unroll 4
    for (int i = 0; i < kSegment / 4; ++i) {
      const int4 a = s_a[i];
      if constexpr (PLACE) {
        if (a.x != c && a.y != c && a.z != c && a.w != c) continue;
        const int row = seg * kSegment + 4 * i;
        if (a.x == c) members[at++] = row;
        if (a.y == c) members[at++] = row + 1;
        if (a.z == c) members[at++] = row + 2;
        if (a.w == c) members[at++] = row + 3;
      } else {
        at += (a.x == c) + (a.y == c) + (a.z == c) + (a.w == c);
      }
    }
    if (!PLACE) offsets[static_cast<size_t>(c) * segments + seg] = at;
  }
}

// Exclusive prefix sum of each run's `count` entries, in place.
__global__ void __launch_bounds__(1024) kmeans_offsets_kernel(int* __restrict__ offsets, int count,
                                                              const int* __restrict__ active) {
  __shared__ int s_wave[16];
  const int run = blockIdx.x;
  if (active != nullptr && !active[run]) return;  // whole block
  offsets += static_cast<size_t>(run) * count;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int base = 0;
  for (int e0 = 0; e0 < count; e0 += 1024) {
    const int e = e0 + static_cast<int>(threadIdx.x);
    const int v = e < count ? offsets[e] : 0;
    int sum = v;  // inclusive over the wave
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(sum, d);
      if (lane >= d) sum += up;
    }
    if (lane == 63) s_wave[wave] = sum;
    __syncthreads();
    int before = 0, total = 0;
    for (int w = 0; w < 16; ++w) {
      if (w < wave) before += s_wave[w];
      total += s_wave[w];
    }
    if (e < count) offsets[e] = base + before + sum - v;
    base += total;
    __syncthreads();
  }
}

__global__ void __launch_bounds__(kBlock) kmeans_update_kernel(const float* __restrict__ x, int n, int p,
                                                                const int* __restrict__ offsets, int segments,
                                                                const int* __restrict__ members, int k,
                                                                float* __restrict__ centroids,
                                                                float* __restrict__ sizes,
                                                                const int* __restrict__ active) {
  constexpr int kInFlight = 16;
  const int run = blockIdx.y;
  if (active != nullptr && !active[run]) return;  // whole block
  x += static_cast<size_t>(run) * n * p;
  offsets += static_cast<size_t>(run) * k * segments;
  members += static_cast<size_t>(run) * n;
  const int c = blockIdx.x;
  const int begin = offsets[static_cast<size_t>(c) * segments];
  const int end = c + 1 < k ? offsets[static_cast<size_t>(c + 1) * segments] : n;
  const int f = threadIdx.x;
  // A float count by ones stops at 2^24.
  const float count = static_cast<float>(min(end - begin, 1 << 24));
  if (f < p) {
    float acc = 0.0f;
    int m = begin;
    for (; m + kInFlight <= end; m += kInFlight) {
      float v[kInFlight];
#pragma unroll
      for (int i = 0; i < kInFlight; ++i) v[i] = x[static_cast<size_t>(members[m + i]) * p + f];
#pragma unroll
      for (int i = 0; i < kInFlight; ++i) acc = __fadd_rn(acc, v[i]);
    }
    if (m < end) {
      float v[kInFlight];
#pragma unroll
      for (int i = 0; i < kInFlight; ++i) v[i] = x[static_cast<size_t>(members[min(m + i, end - 1)]) * p + f];
#pragma unroll
      for (int i = 0; i < kInFlight; ++i) {
        if (m + i < end) acc = __fadd_rn(acc, v[i]);
      }
    }
    if (count != 0.0f) acc = __fmul_rn(acc, __fdiv_rn(1.0f, count));
    centroids[(static_cast<size_t>(run) * k + c) * p + f] = acc;
  }
  if (threadIdx.x == 0) sizes[static_cast<size_t>(run) * k + c] = count;
}

__global__ void __launch_bounds__(kBlock) local_fill_kernel(uint32_t* __restrict__ local, size_t words) {
  for (size_t e = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x; e < words;
       e += static_cast<size_t>(gridDim.x) * kBlock) {
    local[e] = 0xFFFFFFFFu;
  }
}

// local[landmark row][r] = its position in run r's landmark list (rows are
// distinct within a run, so no two threads write one entry).
template <class T>
__global__ void __launch_bounds__(kBlock) local_scatter_kernel(ProjectParams prm) {
  const int j = blockIdx.x * kBlock + threadIdx.x;
  const int r = blockIdx.y;
  const int begin = prm.run_offsets[r];
  if (j >= prm.run_offsets[r + 1] - begin) return;
  static_cast<T*>(prm.local)[static_cast<size_t>(prm.landmarks[begin + j]) * prm.run_stride + r] = static_cast<T>(j);
}

// The result of row i in a run: `local` is the run's column of the table, `row`
// the graph row, `votes` this lane's LDS slice (an entry per 64 lanes). Whole
// waves; `mine` is false in lanes without a row or run.
template <class T>
__device__ __forceinline__ int project_row(const ProjectParams& prm, const int* row, const T* local, int i,
                                           const int* lab, bool mine, int* votes) {
  constexpr T kNone = static_cast<T>(-1);
  const T self = mine ? local[static_cast<size_t>(i) * prm.run_stride] : kNone;
  int nv = 0;
  bool open = mine && self == kNone;  // still collects votes
  for (int j0 = 0; j0 < prm.neighbors && __ballot(open) != 0ull; j0 += 8) {
    // Eight neighbours' table rows in flight.
    T pos[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int g = j0 + u < prm.neighbors ? row[j0 + u] : -1;
      pos[u] = g >= 0 && g < prm.n ? local[static_cast<size_t>(g) * prm.run_stride] : kNone;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (open && pos[u] != kNone) {
        votes[nv * 64] = static_cast<int>(pos[u]);
        open = ++nv < prm.votes;
      }
    }
  }
  if (!mine) return 0;
  if (self != kNone) return lab[self];
  if (nv == 0) return lab[0];
  // Labels only now: their loads wait once, not per neighbour.
  for (int a = 0; a < nv; ++a) votes[a * 64] = lab[votes[a * 64]];
  int best = 0, best_count = 0;
  for (int a = 0; a < nv; ++a) {
    const int va = votes[a * 64];
    int cnt = 0;
    for (int b = 0; b < nv; ++b) cnt += votes[b * 64] == va ? 1 : 0;
    if (cnt > best_count || (cnt == best_count && va < best)) {
      best = va;
      best_count = cnt;
    }
  }
  return best;
}

// blockIdx.x: 64 rows, sixteen per wave; blockIdx.y: 64 runs, one per lane.
template <class T>
__global__ void __launch_bounds__(kBlock) project_kernel(ProjectParams prm) {
  __shared__ int s_out[64][65];               // [run][row]
  extern __shared__ int votes_lds[];          // [4 waves][votes][64 lanes]
  // The wave is uniform: its graph rows come through scalar loads.
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6), lane = threadIdx.x & 63;
  const int r = static_cast<int>(blockIdx.y) * 64 + lane;
  const bool mine = r < prm.runs;
  const int* lab = prm.clbest + (mine ? prm.run_offsets[r] : 0);
  const T* local = static_cast<const T*>(prm.local) + static_cast<size_t>(blockIdx.y) * 64 + lane;
  int* votes = votes_lds + wave * prm.votes * 64 + lane;
  for (int q = 0; q < 16; ++q) {
    const int i = static_cast<int>(blockIdx.x) * 64 + wave * 16 + q;
    if (i >= prm.n) break;
    const int* row = prm.graph + static_cast<size_t>(i) * prm.neighbors;
    s_out[lane][wave * 16 + q] = project_row<T>(prm, row, local, i, lab, mine, votes);
  }
  __syncthreads();
  const int i = static_cast<int>(blockIdx.x) * 64 + lane;
  for (int u = wave; u < 64; u += 4) {
    const int run = static_cast<int>(blockIdx.y) * 64 + u;
    if (run < prm.runs && i < prm.n) prm.res[static_cast<size_t>(run) * prm.n + i] = s_out[u][lane];
  }
}

// Up to 32 runs: run_stride (a power of two) lanes per row, 64 / run_stride
// rows a wave.
template <class T>
__global__ void __launch_bounds__(kBlock) project_few_kernel(ProjectParams prm) {
  extern __shared__ int votes_lds[];          // [4 waves][votes][64 lanes]
  const size_t t = static_cast<size_t>(blockIdx.x) * kBlock + threadIdx.x;
  const size_t at = t / static_cast<unsigned>(prm.run_stride);
  const int r = static_cast<int>(t & static_cast<unsigned>(prm.run_stride - 1));
  const bool mine = at < static_cast<size_t>(prm.n) && r < prm.runs;
  const int i = mine ? static_cast<int>(at) : 0;
  const int* lab = prm.clbest + (mine ? prm.run_offsets[r] : 0);
  const T* local = static_cast<const T*>(prm.local) + (mine ? r : 0);
  int* votes = votes_lds + (threadIdx.x >> 6) * prm.votes * 64 + (threadIdx.x & 63);
  const int out =
      project_row<T>(prm, prm.graph + static_cast<size_t>(i) * prm.neighbors, local, i, lab, mine, votes);
  if (mine) prm.res[static_cast<size_t>(r) * prm.n + i] = out;
}

// ---- launchers --------------------------------------------------------------

hipError_t launch_sse_norms(const float* x, int rows, int p, float* out, float* norm_max, hipStream_t s) {
  if (rows == 0) return hipSuccess;
  hipLaunchKernelGGL(sse_norms_kernel, dim3((rows + kBlock - 1) / kBlock), dim3(kBlock), 0, s, x, rows, p, out,
                     norm_max);
  return hipGetLastError();
}

template <int KS>
static void launch_assign_steps(const KmeansAssignParams& prm, int runs, hipStream_t s) {
  constexpr int NQ = KS <= 4 ? 4 : 2;
  const int rows = 4 * NQ * 16;
  hipLaunchKernelGGL((kmeans_assign_kernel<KS, NQ>), dim3((prm.n + rows - 1) / rows, runs), dim3(kBlock), 0, s, prm);
}

hipError_t launch_kmeans_assign(const KmeansAssignParams& prm, hipStream_t s, int runs) {
  const int steps = stream_steps(prm.p, prm.parts, true);
  if (prm.p < 1 || prm.p > 256 || prm.k < 1 || prm.k > (1 << 25) || runs < 1 || runs > 65535 || steps < 1 || steps > 9 ||
      prm.pad_n % 16 != 0 || prm.pad_n < prm.n || prm.pad_k % 64 != 0 || prm.pad_k < prm.k || prm.c_norm_max == nullptr) {
    return hipErrorInvalidValue;
  }
  if (prm.n == 0) return hipSuccess;
  switch (steps) {
    case 1: launch_assign_steps<1>(prm, runs, s); break;
    case 2: launch_assign_steps<2>(prm, runs, s); break;
    case 3: launch_assign_steps<3>(prm, runs, s); break;
    case 4: launch_assign_steps<4>(prm, runs, s); break;
    case 5: launch_assign_steps<5>(prm, runs, s); break;
    case 6: launch_assign_steps<6>(prm, runs, s); break;
    case 7: launch_assign_steps<7>(prm, runs, s); break;
    case 8: launch_assign_steps<8>(prm, runs, s); break;
    default: launch_assign_steps<9>(prm, runs, s); break;
  }
  return hipGetLastError();
}

int kmeans_segments(int n) { return (n + kSegment - 1) / kSegment; }

hipError_t launch_kmeans_update(const float* x, int n, int p, const int* assign, int k, int* offsets, int* members,
                                float* centroids, float* sizes, hipStream_t s, int runs, const int* active) {
  if (p < 1 || p > kBlock || k < 1 || runs < 1) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  const int segments = kmeans_segments(n);
  const dim3 sort_grid(segments, runs);
  hipLaunchKernelGGL((kmeans_members_kernel<false>), sort_grid, dim3(kBlock), 0, s, assign, n, k, offsets, members,
                     active);
  hipLaunchKernelGGL(kmeans_offsets_kernel, dim3(runs), dim3(1024), 0, s, offsets, k * segments, active);
  hipLaunchKernelGGL((kmeans_members_kernel<true>), sort_grid, dim3(kBlock), 0, s, assign, n, k, offsets, members,
                     active);
  hipLaunchKernelGGL(kmeans_update_kernel, dim3(k, runs), dim3((p + 63) / 64 * 64), 0, s, x, n, p, offsets, segments,
                     members, k, centroids, sizes, active);
  return hipGetLastError();
}

template <class T>
static hipError_t launch_project_t(const ProjectParams& prm, hipStream_t s) {
  const bool few = prm.run_stride < 64;
  const size_t votes = 4 * 64 * sizeof(int) * static_cast<size_t>(prm.votes);
  const hipError_t e = hipFuncSetAttribute(
      few ? reinterpret_cast<const void*>(&project_few_kernel<T>) : reinterpret_cast<const void*>(&project_kernel<T>),
      hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(votes));
  if (e != hipSuccess) return e;
  const size_t words = project_local_bytes(prm.n, prm.runs, prm.max_landmarks) / sizeof(uint32_t);
  const size_t fill_blocks = std::min<size_t>((words + kBlock - 1) / kBlock, 8192);
  hipLaunchKernelGGL(local_fill_kernel, dim3(static_cast<unsigned>(fill_blocks)), dim3(kBlock), 0, s,
                     static_cast<uint32_t*>(prm.local), words);
  hipLaunchKernelGGL((local_scatter_kernel<T>), dim3((prm.max_landmarks + kBlock - 1) / kBlock, prm.runs),
                     dim3(kBlock), 0, s, prm);
  if (few) {
    const size_t threads = static_cast<size_t>(prm.n) * prm.run_stride;
    hipLaunchKernelGGL((project_few_kernel<T>), dim3(static_cast<unsigned>((threads + kBlock - 1) / kBlock)),
                       dim3(kBlock), votes, s, prm);
  } else {
    hipLaunchKernelGGL((project_kernel<T>), dim3((prm.n + 63) / 64, (prm.runs + 63) / 64), dim3(kBlock), votes, s, prm);
  }
  return hipGetLastError();
}

// Whole words.
size_t project_local_bytes(int n, int runs, int max_landmarks) {
  const size_t bytes =
      static_cast<size_t>(n) * project_run_stride(runs) * (max_landmarks <= kProjectNarrow ? 2 : 4);
  return (bytes + 3) / 4 * 4;
}

hipError_t launch_project(const ProjectParams& prm, hipStream_t s) {
  if (prm.votes < 1 || prm.votes > kMaxVotes || prm.neighbors < 0 || prm.runs < 1 || prm.local == nullptr ||
      prm.max_landmarks < 1 || prm.run_stride != project_run_stride(prm.runs)) {
    return hipErrorInvalidValue;
  }
  if (prm.n == 0) return hipSuccess;
  if (prm.max_landmarks <= kProjectNarrow) return launch_project_t<uint16_t>(prm, s);
  return launch_project_t<uint32_t>(prm, s);
}

}  // namespace kodama_hip
