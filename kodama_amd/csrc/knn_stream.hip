// Exact kNN through FP16 matrix-core candidates with a threshold from class maxima, and
// an exact FP32 rerank.
//
// Score of a (query, train row) pair: s = q.t - |t|^2 / 2 (Euclidean) or q.t
// (inner product, cosine rows); the nearest rows have the largest scores. The
// train rows, and for Euclidean distances the queries, are taken less a sample's
// mean, which moves no distance (or all of a query's inner products alike): the
// error below follows the spread of the data and not their offset (50k x 128,
// k = 30, at a mean of 10 standard deviations: 3.9 ms; without, every row was
// flagged twice and scanned, 193 ms). All rows are scaled by one power of two
// that brings the largest norm to at most 2^14, rounded to FP16 (parts = 1) or
// split into two FP16 parts (parts = 3: hi.hi + hi.lo + lo.hi along K), and the
// norm term rides in spare K columns (2^13 on the query side, the FP16 parts of
// -|t|^2 / 2^14 on the train side), so one v_mfma_f32_32x32x16_f16 chain gives s for 32 x 32 pairs. Each
// s differs from the exact distance's by at most E (pair_error below).
//
// Three kernels stream the train rows (a wave owns 32 NQ queries as B operands
// in registers; train rows go through LDS 64 at a time in the fragment order
// of the A operand, so staging and reads are linear; output lane l holds query
// l % 32 against train rows 8 (r / 4) + 4 (l / 32) + r % 4, r = 0..15). The
// 32 x 32 products reach 1.8 PFLOP/s here on random operands (2.45 on zeros),
// the 16 x 16 ones 1.25 (1.36), measured with operands held in registers.
//
// knn_maxima_kernel, over all rows or a sample of about 1000 k: each lane
// keeps the largest score of each of its 16 row classes (half a three-way
// maximum per pair, no branch). A query has 32 classes per slice of the
// sample, at least 2.1 k in all.
// knn_threshold_kernel: T = the k-th largest of a query's class maxima (all of
// distinct rows, so at least k rows reach T; it is about the 1.4 k-th largest
// score), threshold T - 2E: the k-th best exact distance belongs to a
// score >= T - E, so every row of the true k nearest scores >= T - 2E.
// knn_candidates_kernel, over all rows: a pair below its query's threshold is
// dropped with one maximum per two pairs and one compare per 16; the others are
// appended to the query's candidate buffer. Where the sample was a part of the
// rows the buffer may run full; the wave then tightens T from the buffer
// itself (bisection over ballots) and drops what falls below.
// At 1M rows the matrix cores are busy 47 % of the cycles at 1.9 GHz (the
// maxima: 71 % at 1.5; the card holds 1.7 of its 2.4 GHz under bare products
// of such operands, so power is the outer limit); the rest is a wave with
// pairs to append, nearly every stage, holding the other three at its barrier.
// 128 queries per wave, half the LDS traffic and half the waves: 161 ms
// against 134. The pairs queued in LDS and drained 64 at a time: 507 ms (the
// queue's code spills registers in the loop).
// Two passes of MFMAs with 1.4 k appends per query cost less than one
// pass with lists or a running threshold (k ln(n / k) appends): an append
// takes as long as the MFMAs of some 1000 pairs.
//
// knn_stream_rerank_kernel: one wave per query merges the slices'
// candidates, applies the same bound once more, re-scores what is left in the
// reference's FP32 summation order (one candidate per lane) and writes the k
// smallest by (distance, index): the rows and values of the exact scan. Its
// time is the gathered rows (a lane's own row, 16 bytes a load: the copy is
// padded to 4 columns) and the ranking of n ~ k candidates against each other,
// so that the second bound is only taken where it saves a round of 64
// distances, and distance and row are one 64-bit key, read two at a time.
// Rows staged through LDS for coalesced loads left fewer waves in flight:
// 1.9 ms against 1.5 at k = 100.
// Queries whose bound kept more than the buffer holds (many near-equal
// distances) are flagged for another path.
//
// Measured on one MI355X: the self graph of 1M x 50, k = 30, maxima 3.6 ms,
// candidates 134 ms (7.5e12 pairs/s, 0.95 PFLOP/s of FP16 with the padding to
// 64 columns), rerank 4.1 ms (5.4 with 4-byte loads, a bound for every query and
// keys of two words); split-BF16 products with sorted lists per lane
// column took 871 + 34 ms for the candidates. 100k x 50, k = 100: 1.05 + 2.55
// (3.0 with 16 x 16 products, which take as long at 1M rows) + 1.06 ms (1.5) against 26.6 + 18.9 (scan of the queries the lists could not
// certify) + 1.3. 10007 x 30011 x 100, k = 30: 0.33 ms against 23.1 ms of the
// register scan. A running threshold without the maxima appended 3.5 times as
// much: 316 ms at 1M rows, 18.3 ms at 100k.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "knn_stream.h"
#include "score_device.h"

namespace kodama_hip {

namespace {

constexpr int kWave = 64;
constexpr int kTile = 32;   // rows of an operand fragment and of an MFMA
constexpr int kChunk = 64;  // train rows per LDS stage
// Train row, in its tile of 32, of output register r in the wave's half h.
constexpr int tile_row(int r) { return 8 * (r / 4) + r % 4; }  // + 4 h

// A key that at least k of the wave's keys (R per lane, 0 = empty, at least k
// non-empty) reach and at most k + 2 unless ties or `exact`: bisection on
// ballot counts. Uniform.
template <int R>
__device__ __forceinline__ uint32_t kth_largest(const uint32_t (&key)[R], int used, int k) {
  uint32_t hi = 0, lo = 0;
#pragma unroll
  for (int i = 0; i < R; ++i) hi = max(hi, key[i]);
  {
    uint32_t inv = 0;  // smallest non-empty key, as the largest complement
#pragma unroll
    for (int i = 0; i < R; ++i) inv = max(inv, key[i] != 0u ? ~key[i] : 0u);
    lo = ~wave_max(inv);
  }
  hi = wave_max(hi);  // count(>= lo) >= k; the answer is in [lo, hi]
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo + 1u) / 2u;  // lo < mid <= hi
    int c = 0;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (i < used) c += __popcll(__ballot(key[i] >= mid));
    }
    if (c >= k) {
      lo = mid;
      if (c <= k + 2) break;
    } else {
      hi = mid - 1u;
    }
  }
  return lo;
}

}  // namespace

// Mean of a sample of the rows. 16 columns a block, 64 threads a column with all
// their loads in flight: one round trip to memory (four times as many in turn
// added some 15 us to a call).
__global__ void __launch_bounds__(1024) stream_center_kernel(const float* __restrict__ x, int rows, int p, int stride,
                                                             float* __restrict__ center) {
  constexpr int kParts = 64, kLoads = kStreamCenterRows / kParts;
  __shared__ float s_sum[kParts][17];
  __shared__ int s_count[kParts][17];
  const int sub = threadIdx.x & 15, part = threadIdx.x >> 4;
  const int c = static_cast<int>(blockIdx.x) * 16 + sub;
  float v[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int e = part + i * kParts;
    const size_t row = rows > kStreamCenterRows ? static_cast<size_t>(e) * static_cast<size_t>(rows) / kStreamCenterRows
                                                : static_cast<size_t>(e);
    v[i] = c < p && row < static_cast<size_t>(rows) ? x[row * stride + c] : INFINITY;
  }
  float sum = 0.0f;
  int count = 0;
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const bool use = isfinite(v[i]);
    sum += use ? v[i] : 0.0f;
    count += use ? 1 : 0;
  }
  s_sum[part][sub] = sum;
  s_count[part][sub] = count;
  __syncthreads();
  if (part != 0 || c >= p) return;
#pragma unroll 8
  for (int i = 1; i < kParts; ++i) {
    sum += s_sum[i][sub];
    count += s_count[i][sub];
  }
  const float mean = sum / static_cast<float>(max(count, 1));
  center[c] = isfinite(mean) ? mean : 0.0f;
}

// 16 lanes per row; block maxima, one atomic each per block (norms are >= 0, so
// their bits order as integers; a NaN norm does not enter).
__global__ void stream_norms_kernel(StreamNormsJob job) {
  __shared__ uint32_t s_max[2];
  if (threadIdx.x < 2) s_max[threadIdx.x] = 0u;
  __syncthreads();
  const int sub = threadIdx.x & 15;
  for (size_t r = static_cast<size_t>(blockIdx.x) * 16 + (threadIdx.x >> 4); r < static_cast<size_t>(job.rows);
       r += static_cast<size_t>(gridDim.x) * 16) {
    const float* src = job.x + r * job.stride;
    float s = 0.0f, given = 0.0f;
    for (int d = sub; d < job.p; d += 16) {
      const float g = src[d], v = g - (job.center != nullptr ? job.center[d] : 0.0f);
      s = fmaf(v, v, s);
      given = fmaf(g, g, given);
    }
#pragma unroll
    for (int m = 1; m < 16; m <<= 1) {
      s += __shfl_xor(s, m);
      given += __shfl_xor(given, m);
    }
    if (sub == 0) {
      if (job.norm2 != nullptr) job.norm2[r] = s;
      if (s >= 0.0f) atomicMax(&s_max[0], __float_as_uint(s));
      if (job.given_norm2 != nullptr) job.given_norm2[r] = given;
      if (given >= 0.0f) atomicMax(&s_max[1], __float_as_uint(given));
    }
  }
  __syncthreads();
  if (threadIdx.x == 0 && s_max[0] != 0u) atomicMax(reinterpret_cast<uint32_t*>(job.norm2_max), s_max[0]);
  if (threadIdx.x == 1 && s_max[1] != 0u && job.given_norm2_max != nullptr) {
    atomicMax(reinterpret_cast<uint32_t*>(job.given_norm2_max), s_max[1]);
  }
}

// One thread per 16-byte fragment piece: with fragments of T rows (32 or 16)
// and 512 / T columns, piece ((tile * (steps T / 16) + step) * 64 + lane)
// holds row tile * T + lane % T, columns step * 512 / T + 8 (lane / T) .. + 7.
// Blocks cover 256 pieces; reads are 8 consecutive floats a lane.
__global__ void stream_operands_kernel(StreamOperandJob job, int steps) {
  const size_t e = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const size_t total = static_cast<size_t>(job.pad_rows) / 16 * steps * 64;
  if (e >= total) return;
  const int lane = static_cast<int>(e & 63);
  const int tile = job.tile, fragments = steps * tile / 16;
  const size_t ts = e >> 6;
  const int step = static_cast<int>(ts % fragments);
  const int prow = static_cast<int>(ts / fragments) * tile + (lane & (tile - 1));
  int row = prow;
  bool live = prow < job.rows;
  if (job.group_pad > 0) {
    const int group = prow / job.group_pad, local = prow - group * job.group_pad;
    live = local < job.group_rows;
    row = group * job.group_rows + local;
  }
  if (job.block_run != nullptr) {
    const int run = job.block_run[prow / kStreamBlockRows];
    const int local = prow - job.pad_offsets[run];
    live = local < job.run_offsets[run + 1] - job.run_offsets[run];
    row = job.run_offsets[run] + local;
  }
  const float scale = operand_scale(job.norm2_max);
  const int p = job.p;
  const int c0 = step * (512 / tile) + 8 * (lane / tile);
  _Float16 tv[8], qv[8];
  const float* src = job.x + static_cast<size_t>(live ? row : 0) * (job.stride != 0 ? job.stride : p);
  const float nt = live && job.euclid ? -(job.norm2[row] * scale) * scale * 0x1p-14f : 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int c = c0 + i;
    _Float16 a = static_cast<_Float16>(0.0f), b = static_cast<_Float16>(0.0f);
    if (live) {
      if (c < job.parts * p) {
        const int seg = c / p, d = c - seg * p;
        const float v = src[d];
        const float t = (v - (job.train_center != nullptr ? job.train_center[d] : 0.0f)) * scale;
        const float q = (v - (job.query_center != nullptr ? job.query_center[d] : 0.0f)) * scale;
        const _Float16 th = static_cast<_Float16>(t), qh = static_cast<_Float16>(q);
        a = seg == 1 ? static_cast<_Float16>(t - static_cast<float>(th)) : th;  // train: hi, lo, hi
        b = seg == 2 ? static_cast<_Float16>(q - static_cast<float>(qh)) : qh;  // query: hi, hi, lo
      } else if (job.euclid) {
        const int j = c - job.parts * p;
        const _Float16 h = static_cast<_Float16>(nt);
        const float r1 = nt - static_cast<float>(h);
        const _Float16 m = static_cast<_Float16>(r1);
        const _Float16 l = static_cast<_Float16>(r1 - static_cast<float>(m));
        const int parts = job.parts == 1 ? 2 : 3;
        if (j < parts) {
          a = j == 0 ? h : j == 1 ? m : l;
          b = static_cast<_Float16>(8192.0f);
        }
      }
    }
    tv[i] = a;
    qv[i] = b;
  }
  if (job.train_op != nullptr) {
    f16x8 w;
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = tv[i];
    reinterpret_cast<u32x4*>(job.train_op)[e] = __builtin_bit_cast(u32x4, w);
  }
  if (job.query_op != nullptr) {
    f16x8 w;
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = qv[i];
    reinterpret_cast<u32x4*>(job.query_op)[e] = __builtin_bit_cast(u32x4, w);
  }
}

// The queries and train rows of one workgroup.
struct StreamRange {
  int t_begin, t_end, q_end;  // operand rows
  int delta;                  // operand row -> row of x (tables: concatenated)
};
__device__ __forceinline__ StreamRange stream_range(const KnnStreamParams& prm, int q_block) {
  StreamRange g{0, prm.train_rows, prm.query_rows, 0};
  if (prm.block_run != nullptr) {
    const int run = prm.block_run[q_block / kStreamBlockRows];
    g.t_begin = prm.pad_offsets[run];
    g.t_end = g.q_end = g.t_begin + (prm.run_offsets[run + 1] - prm.run_offsets[run]);
    g.delta = prm.run_offsets[run] - g.t_begin;
  }
  return g;
}

// Roundings of the kNN distances (p <= 256: at most 8 block sums, the lane tree
// of 5 and 31 tail terms in sequence, one rounding each: 50) and of a centred
// row (2^-24 of it, which moves half a squared distance by at most
// 2^-23 (q^2 + t^2)).
constexpr float kDistanceRoundings = 52.0f;

// 2E for a query of squared norm norm2, scaled. A Euclidean value is computed
// from differences, which the centre does not enter; an inner product from the
// rows as given.
__device__ __forceinline__ float drop_error(const KnnStreamParams& prm, float norm2) {
  const float scale = operand_scale(prm.norm2_max) * 1.0001f;
  const float q = sqrtf(norm2) * scale;
  const float t = sqrtf(prm.norm2_max[0]) * scale;
  const float given = prm.euclid ? t : sqrtf(fmaxf(prm.norm2_max[1], prm.norm2_max[2])) * scale;
  const int width = prm.parts * prm.dims + (prm.euclid ? 3 : 0);
  return 2.0f * pair_error(q, t, prm.dims, prm.parts, width, q * q + given * given, kDistanceRoundings);
}

// LDS staging of 64 train rows: the next chunk is loaded into registers while
// this one is scored; two buffers, one barrier per chunk.
constexpr int kThreads = 256;
template <int KS, bool FOLDS>
__device__ __forceinline__ void fetch_chunk(const KnnStreamParams& prm, const StreamRange& g, int c0, u32x4 (&pre)[KS],
                                            int& pre_grp) {
  const u32x4* src = reinterpret_cast<const u32x4*>(prm.train_op) + static_cast<size_t>(c0 / kTile) * (2 * KS * 64);
#pragma unroll
  for (int i = 0; i < KS; ++i) pre[i] = src[static_cast<int>(threadIdx.x) + i * kThreads];
  if (FOLDS && threadIdx.x < kChunk) {
    const int j = c0 + static_cast<int>(threadIdx.x);
    pre_grp = j < g.t_end ? prm.folds[j + g.delta] : -2;
  }
}
template <int KS, bool FOLDS>
__device__ __forceinline__ void store_chunk(const KnnStreamParams& prm, const u32x4 (&pre)[KS], int pre_grp, u32x4* s_t,
                                            int* s_grp) {
#pragma unroll
  for (int i = 0; i < KS; ++i) s_t[static_cast<int>(threadIdx.x) + i * kThreads] = pre[i];
  if (FOLDS && threadIdx.x < kChunk) s_grp[threadIdx.x] = pre_grp;
}

template <int KS, int NQ>
__device__ __forceinline__ void load_queries(const KnnStreamParams& prm, int q_wave, int q_end, int lane,
                                             f16x8 (&bq)[NQ][2 * KS]) {
#pragma unroll
  for (int t = 0; t < NQ; ++t) {
    // Operand tiles exist for the padded rows; a wave past them reads none.
    const u32x4* src =
        reinterpret_cast<const u32x4*>(prm.query_op) + (static_cast<size_t>(q_wave / kTile + t) * (2 * KS)) * 64 + lane;
    const bool tile = q_wave + t * kTile < q_end;
#pragma unroll
    for (int ks = 0; ks < 2 * KS; ++ks) bq[t][ks] = as_f16x8(tile ? src[ks * 64] : u32x4{0, 0, 0, 0});
  }
}

// Scores of one tile of train rows against the wave's queries.
template <int KS, int NQ>
__device__ __forceinline__ void score_tile(const u32x4* s_tile, int lane, const f16x8 (&bq)[NQ][2 * KS],
                                           f32x16 (&acc)[NQ]) {
  const f32x16 zero = {};
#pragma unroll
  for (int ks = 0; ks < 2 * KS; ++ks) {
    const f16x8 a = as_f16x8(s_tile[ks * 64 + lane]);
#pragma unroll
    for (int t = 0; t < NQ; ++t) {
      acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, bq[t][ks], ks == 0 ? zero : acc[t], 0, 0, 0);
    }
  }
}

// KS: 32 columns of the operands each. NQ: 32-query tiles per wave. blockIdx.x: query block,
// blockIdx.y: share of the sampled chunks.
template <int KS, int NQ, bool FOLDS>
__global__ void __launch_bounds__(256, KS <= 2 ? 3 : 2) knn_maxima_kernel(KnnStreamParams prm) {
  constexpr int kWaveQueries = NQ * kTile;
  __shared__ u32x4 s_t[2][KS * kThreads];  // 64 rows x KS x 64 bytes
  __shared__ int s_grp[2][FOLDS ? kChunk : 4];
  const int wave = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int half = lane / kTile, col = lane % kTile;
  const int q_block = prm.query_begin + static_cast<int>(blockIdx.x) * (4 * kWaveQueries);
  const StreamRange g = stream_range(prm, q_block);
  if (q_block >= g.q_end) return;
  const int q_wave = q_block + wave * kWaveQueries;
  f16x8 bq[NQ][2 * KS];
  load_queries<KS, NQ>(prm, q_wave, g.q_end, lane, bq);
  int fold[NQ];
  float top[NQ][16];  // class 8 sub + r / 2
#pragma unroll
  for (int t = 0; t < NQ; ++t) {
    const int q = q_wave + t * kTile + col;
    fold[t] = FOLDS && q < g.q_end ? prm.folds[q + g.delta] : -1;
#pragma unroll
    for (int i = 0; i < 16; ++i) top[t][i] = -INFINITY;
  }
  // Sampled chunks, evenly spread and distinct (a row counted in two classes
  // would spoil the threshold): chunk i of `picked` is floor(i chunks / picked).
  const int chunks = (g.t_end - g.t_begin + kChunk - 1) / kChunk;
  const int picked = min(chunks, prm.sample_chunks);
  const int step = chunks / picked, rest = chunks - step * picked;
  const int i0 = picked * static_cast<int>(blockIdx.y) / prm.max_slices;
  const int i1 = picked * static_cast<int>(blockIdx.y + 1) / prm.max_slices;
  auto chunk_row = [&](int i) {
    return g.t_begin + (i * step + (rest != 0 ? i * rest / picked : 0)) * kChunk;
  };
  u32x4 pre[KS];
  int pre_grp = -2;
  if (i0 < i1) {
    fetch_chunk<KS, FOLDS>(prm, g, chunk_row(i0), pre, pre_grp);
    store_chunk<KS, FOLDS>(prm, pre, pre_grp, s_t[0], s_grp[0]);
  }
  __builtin_amdgcn_s_waitcnt(0);  // the operands too: no wait for them (and the prefetch) in the loop
  __syncthreads();
  int buf = 0;
  for (int i = i0; i < i1; ++i, buf ^= 1) {
    if (i + 1 < i1) fetch_chunk<KS, FOLDS>(prm, g, chunk_row(i + 1), pre, pre_grp);
    const int c0 = chunk_row(i);
    // `cut`: rows past the end (the last chunk only) must not count.
    auto score = [&](auto cut) {
#pragma unroll
      for (int sub = 0; sub < kChunk / kTile; ++sub) {
        f32x16 acc[NQ];
        score_tile<KS, NQ>(&s_t[buf][sub * 2 * KS * 64], lane, bq, acc);
        if constexpr (decltype(cut)::value) {
          const int j0 = c0 + sub * kTile + 4 * half;
#pragma unroll
          for (int t = 0; t < NQ; ++t) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[t][r] = j0 + tile_row(r) < g.t_end ? acc[t][r] : -INFINITY;
          }
        }
        if constexpr (FOLDS) {
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            const int4 f = *reinterpret_cast<const int4*>(&s_grp[buf][sub * kTile + 8 * b + 4 * half]);
#pragma unroll
            for (int t = 0; t < NQ; ++t) {
              acc[t][4 * b] = f.x != fold[t] ? acc[t][4 * b] : -INFINITY;
              acc[t][4 * b + 1] = f.y != fold[t] ? acc[t][4 * b + 1] : -INFINITY;
              acc[t][4 * b + 2] = f.z != fold[t] ? acc[t][4 * b + 2] : -INFINITY;
              acc[t][4 * b + 3] = f.w != fold[t] ? acc[t][4 * b + 3] : -INFINITY;
            }
          }
        }
#pragma unroll
        for (int t = 0; t < NQ; ++t) {
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            float& c = top[t][8 * sub + i];
            c = fmaxf(fmaxf(c, acc[t][2 * i]), acc[t][2 * i + 1]);
          }
        }
      }
    };
    if (c0 + kChunk > g.t_end) score(std::true_type{});
    else score(std::false_type{});
    if (i + 1 < i1) store_chunk<KS, FOLDS>(prm, pre, pre_grp, s_t[buf ^ 1], s_grp[buf ^ 1]);
    __syncthreads();
  }
#pragma unroll
  for (int t = 0; t < NQ; ++t) {
    const int q = q_wave + t * kTile + col;
    if (q < g.q_end) {
      float4* dst = reinterpret_cast<float4*>(
        prm.maxima + (static_cast<size_t>(q - prm.query_begin) * prm.max_slices + blockIdx.y) * 32 + half * 16);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        dst[i] = make_float4(top[t][4 * i], top[t][4 * i + 1], top[t][4 * i + 2], top[t][4 * i + 3]);
      }
    }
  }
}

// One wave per operand row; REGS x 64 class maxima (empty ones -inf).
template <int REGS>
__global__ void __launch_bounds__(256) knn_threshold_kernel(KnnStreamParams prm, int per_query) {
  // Row of the buffers, and operand row.
  const int local = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x) * 4 + static_cast<int>(threadIdx.x / kWave));
  const int q = prm.query_begin + local;
  const int lane = threadIdx.x & (kWave - 1);
  if (local >= prm.query_rows) return;
  int delta = 0;
  if (prm.block_run != nullptr) {
    const StreamRange g = stream_range(prm, q);
    if (q >= g.q_end) return;
    delta = g.delta;
  }
  const float* src = prm.maxima + static_cast<size_t>(local) * per_query;
  uint32_t key[REGS];
  int valid = 0;
#pragma unroll
  for (int i = 0; i < REGS; ++i) {
    const float v = i * kWave + lane < per_query ? src[i * kWave + lane] : -INFINITY;
    key[i] = v > -INFINITY ? order_key(v) : 0u;
    valid += __popcll(__ballot(key[i] != 0u));
  }
  // One more than k where a query may exclude a train row (tables mask the
  // query's own fold before the maxima).
  const int want = prm.k + (prm.exclude != nullptr ? 1 : 0);
  float bound = norms_usable(prm.norm2_max) ? -INFINITY : INFINITY;
  if (valid >= want && bound < 0.0f) {
    bound = drop_bound(key_value(kth_largest<REGS>(key, REGS, want)), drop_error(prm, prm.query_norm2[q + delta]));
  }
  if (lane == 0) prm.threshold[local] = bound;
}

// R: capacity / 64. blockIdx.x: query block, blockIdx.y: slice of the train rows.
template <int KS, int NQ, int R, bool FOLDS>
__global__ void __launch_bounds__(256, KS <= 2 ? 4 : 2) knn_candidates_kernel(KnnStreamParams prm) {
  constexpr int kCap = 64 * R;
  constexpr int kFull = kCap - kTile;      // a tile of train rows may add 32 to a query
  constexpr int kCompact = kFull - 8;
  constexpr int kWaveQueries = NQ * kTile;
  __shared__ u32x4 s_t[2][KS * kThreads];  // 64 rows x KS x 64 bytes
  __shared__ int s_grp[2][FOLDS ? kChunk : 4];
  __shared__ int s_cnt[4][kWaveQueries];
  __shared__ float s_th[4][kWaveQueries];
  __shared__ int s_ex[4][kWaveQueries];
  const int wave = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int half = lane / kTile, col = lane % kTile;
  const int q_block = prm.query_begin + static_cast<int>(blockIdx.x) * (4 * kWaveQueries);
  StreamRange g = stream_range(prm, q_block);
  if (q_block >= g.q_end) return;
  // This slice's rows (a multiple of 64 except at the end; may be empty).
  if (prm.slices > 1) {
    const int rows = g.t_end - g.t_begin;
    const int per = ((rows + prm.slices - 1) / prm.slices + kChunk - 1) / kChunk * kChunk;
    g.t_begin += per * static_cast<int>(blockIdx.y);
    g.t_end = min(g.t_end, g.t_begin + per);
  }
  const int q_wave = q_block + wave * kWaveQueries;
  const size_t slot0 = static_cast<size_t>(q_wave - prm.query_begin) * prm.slices + blockIdx.y;  // query i: + i * slices
  const bool usable = norms_usable(prm.norm2_max);

  f16x8 bq[NQ][2 * KS];
  load_queries<KS, NQ>(prm, q_wave, g.q_end, lane, bq);
  float th[NQ];
#pragma unroll
  for (int t = 0; t < NQ; ++t) {
    const int q = q_wave + t * kTile + col;
    const bool live = q < g.q_end;
    th[t] = live ? prm.threshold[q - prm.query_begin] : INFINITY;
    if (half == 0) {
      int ex = -1;  // the query's own fold or row
      if (live) {
        if (FOLDS) ex = prm.folds[q + g.delta];
        else if (prm.exclude != nullptr) ex = prm.exclude[q];
      }
      s_ex[wave][t * kTile + col] = ex;
      s_cnt[wave][t * kTile + col] = usable ? 0 : -1;
      s_th[wave][t * kTile + col] = th[t];
    }
  }

  // Compaction of every query of the wave with more than `limit` candidates.
  auto compact = [&](int limit) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");  // the appended entries and the counts
    __builtin_amdgcn_wave_barrier();
    const int mine = lane < kWaveQueries ? s_cnt[wave][lane] : 0;
    uint64_t todo = __ballot(mine > limit);
    while (todo != 0ull) {
      const int q = __builtin_ctzll(todo);
      todo &= todo - 1ull;
      const int n = __builtin_amdgcn_readlane(mine, q);
      uint2* base = prm.cand + (slot0 + static_cast<size_t>(q) * prm.slices) * kCap;
      uint2 ent[R];
      uint32_t key[R];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int e = i * kWave + lane;
        ent[i] = e < n ? base[e] : make_uint2(0xFF800000u, 0u);  // -inf
        key[i] = e < n ? order_key(__uint_as_float(ent[i].x)) : 0u;
      }
      const float bound = drop_bound(key_value(kth_largest<R>(key, R, prm.k)),
                                     drop_error(prm, prm.query_norm2[q_wave + q + g.delta]));
      int kept = 0;
      const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const bool keep = key[i] != 0u && __uint_as_float(ent[i].x) >= bound;
        const uint64_t m = __ballot(keep);
        if (keep) base[kept + __popcll(m & below)] = ent[i];
        kept += __popcll(m);
      }
      const bool over = kept > kCompact;
      if (lane == 0) {
        s_cnt[wave][q] = over ? -1 : kept;
        s_th[wave][q] = over ? INFINITY : fmaxf(bound, s_th[wave][q]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < NQ; ++t) th[t] = s_th[wave][t * kTile + col];
  };

  u32x4 pre[KS];
  int pre_grp = -2;
  if (g.t_begin < g.t_end) {
    fetch_chunk<KS, FOLDS>(prm, g, g.t_begin, pre, pre_grp);
    store_chunk<KS, FOLDS>(prm, pre, pre_grp, s_t[0], s_grp[0]);
  }
  __builtin_amdgcn_s_waitcnt(0);  // the operands too: no wait for them (and the prefetch) in the loop
  __syncthreads();
  int buf = 0;
  for (int c0 = g.t_begin; c0 < g.t_end; c0 += kChunk, buf ^= 1) {
    const bool more = c0 + kChunk < g.t_end;
    if (more) fetch_chunk<KS, FOLDS>(prm, g, c0 + kChunk, pre, pre_grp);  // in flight during the scoring
    const int limit = more ? c0 + kChunk : g.t_end;
#pragma unroll 1
    for (int sub = 0; sub < kChunk / kTile; ++sub) {
      f32x16 acc[NQ];
      score_tile<KS, NQ>(&s_t[buf][sub * 2 * KS * 64], lane, bq, acc);
      uint64_t hit[NQ], any = 0ull;
#pragma unroll
      for (int t = 0; t < NQ; ++t) {
        // Strictly above (the bound has slack): eight three-way maxima and a compare.
        float top = th[t];
#pragma unroll
        for (int i = 0; i < 8; ++i) top = fmaxf(fmaxf(top, acc[t][2 * i]), acc[t][2 * i + 1]);
        hit[t] = __ballot(top > th[t]);
        any |= hit[t];
      }
      if (any != 0ull) {
        const int in_chunk = sub * kTile + 4 * half;
        int c_of = col;  // opaque: no buffer addresses kept in registers over the loop
        asm volatile("" : "+v"(c_of));
        bool full = false;
#pragma unroll
        for (int t = 0; t < NQ; ++t) {
          if (hit[t] == 0ull) continue;
          const int qi = t * kTile + c_of;
          const int ex = s_ex[wave][qi];
          uint2* dst = prm.cand + (slot0 + static_cast<size_t>(qi) * prm.slices) * kCap;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const bool above = acc[t][r] > th[t];
            if (__ballot(above) == 0ull) continue;
            const int j = c0 + in_chunk + tile_row(r);
            const int group = FOLDS ? s_grp[buf][in_chunk + tile_row(r)] : j;
            if (above && group != ex && j < limit) {
              const int slot = atomicAdd(&s_cnt[wave][qi], 1);
              dst[slot] = make_uint2(__float_as_uint(acc[t][r]), static_cast<uint32_t>(j + g.delta));
              full = full || slot >= kFull;
            }
          }
        }
        if (__ballot(full) != 0ull) compact(kCompact);
      }
    }
    if (more) store_chunk<KS, FOLDS>(prm, pre, pre_grp, s_t[buf ^ 1], s_grp[buf ^ 1]);
    __syncthreads();
  }
  // Several slices: keep each list short enough for the rerank to hold all.
  if (prm.slices > 1) compact(max(prm.k + 8, 24));
#pragma unroll
  for (int t = 0; t < NQ; ++t) {
    const int q = q_wave + t * kTile + col;
    if (half == 0 && q < g.q_end) {
      const size_t o = slot0 + static_cast<size_t>(t * kTile + col) * prm.slices;
      prm.cand_count[o] = s_cnt[wave][t * kTile + col];
      prm.cand_bound[o] = th[t];
    }
  }
}

// Reference-order FP32 distance (native_knn.cpp:41-95), one lane per train
// row, the query row uniform over the wave (scalar loads). The train row's
// stride is a multiple of four floats: each lane reads its own row, so every
// load costs the L1 one line per lane, and 16-byte loads take a quarter of
// what single columns do.
template <bool EUCLID>
__device__ __forceinline__ float stream_exact_distance(const float* __restrict__ q, const f32x4* __restrict__ c, int p) {
  float acc[32];
#pragma unroll
  for (int s = 0; s < 32; ++s) acc[s] = 0.0f;
  const int full = p & ~31;
  for (int b = 0; b < full; b += 32) {
    f32x4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = c[b / 4 + i];
#pragma unroll
    for (int s = 0; s < 32; ++s) {
      const float cv = v[s / 4][s % 4];
      if (EUCLID) {
        const float t = __fsub_rn(q[b + s], cv);
        acc[s] = __fmaf_rn(t, t, acc[s]);
      } else {
        acc[s] = __fmaf_rn(q[b + s], cv, acc[s]);
      }
    }
  }
  // The tail of up to 31 columns, in flight while the lane tree is summed.
  f32x4 tail[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) tail[i] = full + 4 * i < p ? c[full / 4 + i] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float v4[4];
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    const float lo = __fadd_rn(__fadd_rn(acc[l], acc[8 + l]), __fadd_rn(acc[16 + l], acc[24 + l]));
    const float hi = __fadd_rn(__fadd_rn(acc[4 + l], acc[12 + l]), __fadd_rn(acc[20 + l], acc[28 + l]));
    v4[l] = __fadd_rn(lo, hi);
  }
  float r = __fadd_rn(__fadd_rn(v4[0], v4[1]), __fadd_rn(v4[2], v4[3]));
#pragma unroll
  for (int s = 0; s < 31; ++s) {
    if (full + s < p) {
      const float cv = tail[s / 4][s % 4];
      if (EUCLID) {
        const float t = __fsub_rn(q[full + s], cv);
        r = __fmaf_rn(t, t, r);
      } else {
        r = __fmaf_rn(q[full + s], cv, r);
      }
    }
  }
  return EUCLID ? r : -r;
}

// The k-th largest of n scores in LDS entries, in R registers per lane.
template <int R>
__device__ __forceinline__ uint32_t kth_of_entries(const uint2* ent, int n, int k, int lane) {
  uint32_t key[R];
#pragma unroll
  for (int i = 0; i < R; ++i) key[i] = i * kWave + lane < n ? order_key(__uint_as_float(ent[i * kWave + lane].x)) : 0u;
  return kth_largest<R>(key, (n + kWave - 1) / kWave, k);
}

template <bool EUCLID>
__global__ void __launch_bounds__(256, 4) knn_stream_rerank_kernel(KnnStreamParams prm) {
  // Two entries past the end: the ranking reads pairs.
  __shared__ __align__(16) uint2 s_ent[4][kStreamMerge + 2];
  __shared__ float s_dist[4][kStreamMerge];
  const int wave = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int local = __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x) * 4 + wave);  // row of the buffers
  const int op_row = prm.query_begin + local;
  const int k = prm.k, p = prm.dims, cap = 16 * prm.list;
  const bool tables = prm.block_run != nullptr;
  if (local >= prm.query_rows) return;  // whole waves; no block barrier below
  const StreamRange g = stream_range(prm, op_row);
  if (op_row >= g.q_end) return;
  const int q = op_row + g.delta;
  uint2* ent = s_ent[wave];
  const uint64_t below = (1ull << lane) - 1ull;
  // Merge: what scores at or above the tightest slice's bound.
  bool bad = false;
  float bound = -INFINITY;
  for (int sl = 0; sl < prm.slices; ++sl) {
    const size_t o = static_cast<size_t>(local) * prm.slices + sl;
    bad = bad || prm.cand_count[o] < 0;
    bound = fmaxf(bound, prm.cand_bound[o]);
  }
  int n = 0;
  for (int sl = 0; sl < prm.slices && !bad; ++sl) {
    const size_t o = static_cast<size_t>(local) * prm.slices + sl;
    const int c = prm.cand_count[o];
    for (int e0 = 0; e0 < c; e0 += kWave) {
      const int e = e0 + lane;
      const uint2 v = e < c ? prm.cand[o * cap + e] : make_uint2(0xFF800000u, 0u);
      const bool keep = e < c && __uint_as_float(v.x) >= bound;
      const uint64_t m = __ballot(keep);
      const int add = __popcll(m);
      if (n + add > kStreamMerge) {
        bad = true;
        break;
      }
      if (keep) ent[n + __popcll(m & below)] = v;
      n += add;
    }
  }
  if (bad) {
    if (lane == 0) prm.flags[q] = 1;
    return;
  }
  if (lane == 0) prm.flags[q] = 0;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  // A tighter bound only where it can save a round of 64 exact distances.
  if ((n + kWave - 1) / kWave > (k + kWave - 1) / kWave) {
    const uint32_t kth = n <= 2 * kWave   ? kth_of_entries<2>(ent, n, k, lane)
                         : n <= 4 * kWave ? kth_of_entries<4>(ent, n, k, lane)
                                          : kth_of_entries<kStreamMerge / kWave>(ent, n, k, lane);
    bound = drop_bound(key_value(kth), drop_error(prm, prm.query_norm2[q]));
    // In-place compaction: a register's entries go to slots at or before
    // their own, and each is read before a later register's is written.
    int kept = 0;
    for (int e0 = 0; e0 < n; e0 += kWave) {
      const int e = e0 + lane;
      const uint2 v = e < n ? ent[e] : make_uint2(0xFF800000u, 0u);
      const bool keep = e < n && __uint_as_float(v.x) >= bound;
      const uint64_t m = __ballot(keep);
      __builtin_amdgcn_wave_barrier();
      if (keep) ent[kept + __popcll(m & below)] = v;
      __builtin_amdgcn_wave_barrier();
      kept += __popcll(m);
    }
    n = kept;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  // Exact distances, as (distance order, row) keys: .y above .x.
  const float* qrow = prm.query + static_cast<size_t>(q) * prm.query_stride;
  for (int e = lane; e < n; e += kWave) {
    const uint32_t row = ent[e].y;
    const float d = stream_exact_distance<EUCLID>(
        qrow, reinterpret_cast<const f32x4*>(prm.train + static_cast<size_t>(row) * prm.train_stride), p);
    // -0 sorts with +0, as the float comparison has it.
    ent[e] = make_uint2(row, order_key(d + 0.0f));
    s_dist[wave][e] = d;
  }
  if (lane < 2) ent[n + lane] = make_uint2(0xFFFFFFFFu, 0xFFFFFFFFu);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  // [query x k] rows and distances; for tables the transposed vote layout
  // [k x pad_rows]: padded rows and scores (minus the distance).
  const size_t step = tables ? static_cast<size_t>(prm.pad_rows) : 1;
  int* out_i = prm.out_index + (tables ? static_cast<size_t>(op_row) : static_cast<size_t>(q) * k);
  float* out_d = prm.out_dist + (tables ? static_cast<size_t>(op_row) : static_cast<size_t>(q) * k);
  const ulonglong2* keys = reinterpret_cast<const ulonglong2*>(ent);
  for (int e = lane; e < n; e += kWave) {
    const unsigned long long mine = reinterpret_cast<const unsigned long long*>(ent)[e];
    int rank = 0;
#pragma unroll 4
    for (int t = 0; t < (n + 1) / 2; ++t) {
      const ulonglong2 o = keys[t];
      rank += (o.x < mine ? 1 : 0) + (o.y < mine ? 1 : 0);
    }
    if (rank < k) {
      const float d = s_dist[wave][e];
      out_i[rank * step] = static_cast<int>(static_cast<uint32_t>(mine)) - (tables ? g.delta : 0);
      out_d[rank * step] = tables ? -d : d;
    }
  }
  for (int t = n + lane; t < k; t += kWave) {
    out_i[t * step] = -1;
    out_d[t * step] = tables ? -INFINITY : INFINITY;
  }
}

hipError_t launch_stream_center(const float* x, int rows, int p, int stride, float* center, hipStream_t s) {
  if (rows < 1 || p < 1 || stride < p) return hipErrorInvalidValue;
  hipLaunchKernelGGL(stream_center_kernel, dim3(static_cast<unsigned>((p + 15) / 16)), dim3(1024), 0, s, x, rows,
                     p, stride, center);
  return hipGetLastError();
}

hipError_t launch_stream_norms(const StreamNormsJob& job, hipStream_t s) {
  if (job.rows == 0) return hipSuccess;
  if (job.p < 1 || job.stride < job.p || job.norm2_max == nullptr) return hipErrorInvalidValue;
  const int blocks = (job.rows + 15) / 16;
  hipLaunchKernelGGL(stream_norms_kernel, dim3(static_cast<unsigned>(blocks < 4096 ? blocks : 4096)), dim3(256), 0, s,
                     job);
  return hipGetLastError();
}

hipError_t launch_stream_operands(const StreamOperandJob& job, hipStream_t s) {
  if (job.pad_rows == 0) return hipSuccess;
  const int steps = stream_steps(job.p, job.parts, job.euclid != 0);
  if ((job.tile != 16 && job.tile != 32) || job.pad_rows % job.tile != 0 || job.p < 1 || steps > kStreamMaxSteps ||
      (job.parts != 1 && job.parts != 3)) {
    return hipErrorInvalidValue;
  }
  const size_t total = static_cast<size_t>(job.pad_rows) / 16 * steps * 64;
  hipLaunchKernelGGL(stream_operands_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, s, job,
                     steps);
  return hipGetLastError();
}

template <int KS>
static void launch_steps(const KnnStreamParams& prm, hipStream_t s) {
  const int rows = prm.query_rows;
  constexpr int NQ = KS <= 4 ? 2 : 1;
  const int qpb = 4 * NQ * kTile;
  const unsigned qblocks = static_cast<unsigned>((rows + qpb - 1) / qpb);
  const dim3 mgrid(qblocks, static_cast<unsigned>(prm.max_slices));
  if (prm.folds != nullptr) hipLaunchKernelGGL((knn_maxima_kernel<KS, NQ, true>), mgrid, dim3(256), 0, s, prm);
  else hipLaunchKernelGGL((knn_maxima_kernel<KS, NQ, false>), mgrid, dim3(256), 0, s, prm);
  const int per_query = prm.max_slices * 32;
  const dim3 tgrid(static_cast<unsigned>((rows + 3) / 4));
  if (per_query <= 64) hipLaunchKernelGGL((knn_threshold_kernel<1>), tgrid, dim3(256), 0, s, prm, per_query);
  else if (per_query <= 128) hipLaunchKernelGGL((knn_threshold_kernel<2>), tgrid, dim3(256), 0, s, prm, per_query);
  else if (per_query <= 256) hipLaunchKernelGGL((knn_threshold_kernel<4>), tgrid, dim3(256), 0, s, prm, per_query);
  else hipLaunchKernelGGL((knn_threshold_kernel<8>), tgrid, dim3(256), 0, s, prm, per_query);
  const dim3 grid(qblocks, static_cast<unsigned>(prm.slices));
  if (prm.folds != nullptr) {
    if (prm.list == 8) hipLaunchKernelGGL((knn_candidates_kernel<KS, NQ, 2, true>), grid, dim3(256), 0, s, prm);
    else hipLaunchKernelGGL((knn_candidates_kernel<KS, NQ, 4, true>), grid, dim3(256), 0, s, prm);
  } else {
    if (prm.list == 8) hipLaunchKernelGGL((knn_candidates_kernel<KS, NQ, 2, false>), grid, dim3(256), 0, s, prm);
    else hipLaunchKernelGGL((knn_candidates_kernel<KS, NQ, 4, false>), grid, dim3(256), 0, s, prm);
  }
}

hipError_t launch_knn_stream(const KnnStreamParams& prm, hipStream_t s) {
  if (prm.query_rows == 0) return hipSuccess;
  const int steps = stream_steps(prm.dims, prm.parts, prm.euclid != 0);
  if (prm.dims < 1 || steps > kStreamMaxSteps || prm.k < 1 || prm.k > kStreamMaxK || prm.train_rows < 1 ||
      prm.train_stride % 4 != 0 || prm.train_stride < prm.dims || prm.query_stride < prm.dims) {
    return hipErrorInvalidValue;
  }
  if (prm.slices < 1 || prm.slices > kStreamMaxSlices || prm.max_slices < 1 || prm.max_slices > kStreamMaxSlices ||
      prm.sample_chunks < 1 || (prm.list != 8 && prm.list != 16) || (prm.list == 8 && prm.k > 32)) {
    return hipErrorInvalidValue;
  }
  const bool tables = prm.block_run != nullptr;
  if (tables != (prm.folds != nullptr) || prm.query_begin % kStreamBlockRows != 0 ||
      (tables ? prm.pad_rows % kStreamBlockRows != 0 || prm.query_rows > prm.pad_rows - prm.query_begin
              : prm.query_begin != 0)) {
    return hipErrorInvalidValue;
  }
  switch (steps) {
    case 1: launch_steps<1>(prm, s); break;
    case 2: launch_steps<2>(prm, s); break;
    case 3: launch_steps<3>(prm, s); break;
    case 4: launch_steps<4>(prm, s); break;
    case 5: launch_steps<5>(prm, s); break;
    case 6: launch_steps<6>(prm, s); break;
    case 7: launch_steps<7>(prm, s); break;
    case 8: launch_steps<8>(prm, s); break;
    default: launch_steps<9>(prm, s); break;
  }
  const unsigned rblocks = static_cast<unsigned>((prm.query_rows + 3) / 4);
  if (prm.euclid) hipLaunchKernelGGL((knn_stream_rerank_kernel<true>), dim3(rblocks), dim3(256), 0, s, prm);
  else hipLaunchKernelGGL((knn_stream_rerank_kernel<false>), dim3(rblocks), dim3(256), 0, s, prm);
  return hipGetLastError();
}

}  // namespace kodama_hip
