// mrl_rerank.hip -- gfx950 post-scan rerank: every candidate row of a shortlist is
// scored against the full f32 query, then the list is stably sorted by score,
// descending.  This is QueryPipeline::rerank_exact_rows (src/pipeline.rs:157-169)
// and the precision loop of the retrieval bench (src/retrieval_bench.rs:739-745)
// over rerank_dot (src/lowprec.rs:103-121).
//
// Numerics match the reference bit for bit:
//  - 768 dims: dot_768 / dot_f16_768 / dot_i8_768 (src/embed.rs:130-206) run eight
//    accumulators, accumulator j summing the products of the elements i = j mod 8
//    in index order from +0.0; the result is acc0 + acc1 + ... + acc7, left to
//    right (times the f16 scale for int8).  Here lane j of an 8-lane group runs
//    accumulator j of one candidate, so the 96 dependent adds of a chain stay
//    sequential and the eight chains run side by side.
//  - other dims (fp32 only): the sequential sum of a[i]*b[i] from -0.0
//    (src/embed.rs:123), one lane per candidate.
//  - the sort is stable: ties (including +0.0 against -0.0, which partial_cmp
//    calls equal) keep the candidates' input order.
//
// Store layout (768 dims).  A row's elements are kept "accumulator-major":
// element i = 8t + j sits at position 96j + t, so accumulator j reads one
// contiguous run of 96 elements with 16-byte loads (24 for f32, 12 for f16, 6
// for int8) instead of 96 strided scalar loads.  The stores for f16 and int8 are
// built here from f32 rows with the reference's conversions
// (Fp16Vec768::from_f32, Int8Vec768::from_f32, src/lowprec.rs:49-94).
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "mrl_half.h"
#include "mrl_internal.h"

namespace mrl {

namespace {

constexpr int kStoreThreads = 256;  // four rows per workgroup, one per wave
constexpr int kScoreThreads = 256;  // 768 dims: 32 candidates per workgroup (8 lanes each)
constexpr int kSortThreads = 256;
constexpr int kSortCap = MRL_MAX_SHORTLIST;
constexpr int kRankMax = 512;
constexpr int kQStride = 100;       // LDS row of one accumulator's 96 query values (bank spread)

__device__ __forceinline__ float zero_acc() {
  float z = 0.0f;
  asm volatile("" : "+v"(z));
  return z;
}

__device__ __forceinline__ uint32_t store_pos(uint32_t i) { return (i & 7u) * 96u + (i >> 3); }

// Order-preserving map f32 -> u32 (larger score -> larger key); -0 == +0.
__device__ __forceinline__ uint32_t score_key(float s) {
  uint32_t u = __float_as_uint(s);
  if ((u << 1) == 0u) u = 0u;
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Int8Vec768::from_f32 code of one element (src/lowprec.rs:83-86):
// round half away from zero, clamp (NaN passes), `as i32` (NaN -> 0).
__device__ __forceinline__ uint32_t int8_code(float v, float inv) {
  float q = roundf(v * inv);
  if (q < -127.0f) q = -127.0f;
  if (q > 127.0f) q = 127.0f;
  const int32_t i = (q == q) ? (int32_t)q : 0;
  return (uint32_t)i & 0xffu;
}

// ---------------------------------------------------------------------------
// store build: f32 rows (row-major, 768 dims) -> accumulator-major rows
// ---------------------------------------------------------------------------
template <int P>
__global__ __launch_bounds__(kStoreThreads) void k_store768(const float* __restrict__ x, uint8_t* __restrict__ data,
                                                            uint16_t* __restrict__ scales, uint64_t n_rows) {
  constexpr uint32_t kRowBytes = P == MRL_RERANK_FP32 ? 3072u : P == MRL_RERANK_FP16 ? 1536u : 768u;
  __shared__ __align__(16) uint8_t s_row[kStoreThreads / 64][3072];
  const uint32_t w = threadIdx.x >> 6, lane = threadIdx.x & 63u;
  uint8_t* sb = s_row[w];
  for (uint64_t r0 = (uint64_t)blockIdx.x * 4u; r0 < n_rows; r0 += (uint64_t)gridDim.x * 4u) {
    const uint64_t r = r0 + w;
    const bool live = r < n_rows;
    float v[12];
    if (live) {
      const float4* src = reinterpret_cast<const float4*>(x + r * 768u);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const float4 f = src[lane + 64u * k];
        v[4 * k] = f.x;
        v[4 * k + 1] = f.y;
        v[4 * k + 2] = f.z;
        v[4 * k + 3] = f.w;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 12; ++e) v[e] = 0.0f;
    }
    float inv = 0.0f;
    if (P == MRL_RERANK_INT8) {
      // max_abs = fold of f32::max over |x| from 0.0 (NaN ignored); max is exact,
      // so the wave reduction order does not matter.
      float m = 0.0f;
#pragma unroll
      for (int e = 0; e < 12; ++e) m = fmaxf(m, fabsf(v[e]));
#pragma unroll
      for (int h = 1; h < 64; h <<= 1) m = fmaxf(m, __shfl_xor(m, h));
      const float scale = m < 1e-12f ? 0.0f : m / 127.0f;
      inv = scale > 0.0f ? 1.0f / scale : 0.0f;
      if (live && lane == 0) scales[r] = (uint16_t)f32_to_f16(scale);
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t i = 4u * lane + 256u * k + e;
        const uint32_t p = store_pos(i);
        const float f = v[4 * k + e];
        if (P == MRL_RERANK_FP32) reinterpret_cast<float*>(sb)[p] = f;
        else if (P == MRL_RERANK_FP16) reinterpret_cast<uint16_t*>(sb)[p] = (uint16_t)f32_to_f16(f);
        else sb[p] = (uint8_t)int8_code(f, inv);
      }
    }
    __syncthreads();
    if (live) {
      uint4* dst = reinterpret_cast<uint4*>(data + r * kRowBytes);
      const uint4* s4 = reinterpret_cast<const uint4*>(sb);
      for (uint32_t c = lane; c < kRowBytes / 16u; c += 64u) dst[c] = s4[c];
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// scoring
// ---------------------------------------------------------------------------
// Row markers in the scratch row array: a row outside the store, and a ring
// hit that scored_hits_to_row_ids drops.
constexpr uint64_t kRowBad = ~0ull;
constexpr uint64_t kRowSkip = ~0ull - 1u;

__device__ __forceinline__ uint32_t count_of(const RerankArgs& a, uint32_t q) {
  return a.counts ? a.counts[q] : a.stride;
}

// Makes this wave's LDS writes visible to its own later reads.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Candidate c of query q -> store row.  *ok false: no row to score (*row says why).
__device__ __forceinline__ void resolve_row(const RerankArgs& a, uint32_t q, uint32_t c, uint64_t* row, bool* ok) {
  if (!a.cand) {
    *row = c;
    *ok = c < a.n_rows;
    if (!*ok) *row = kRowBad;
    return;
  }
  const uint64_t id = a.cand[(uint64_t)q * a.stride + c];
  if (a.cand_ids && (id >> 16) == 0xffffffffull) {  // ring sentinel (block == u32::MAX): skipped
    *row = kRowSkip;
    *ok = false;
    return;
  }
  // scored_hits_to_row_ids (src/pipeline.rs:175-180): block * 64 + slot
  const uint64_t r = a.cand_ids ? (id >> 16) * 64u + (id & 0xffffu) : id;
  *ok = r < a.n_rows;
  *row = *ok ? r : kRowBad;
}

// Accumulator j of one candidate over its 96 stored elements.
template <int P>
__device__ __forceinline__ float chain768(const RerankArgs& a, uint64_t row, uint32_t j, const float* qj) {
  float acc = zero_acc();
  if (P == MRL_RERANK_FP32) {
    const float4* r4 = reinterpret_cast<const float4*>(static_cast<const float*>(a.data) + row * 768u + j * 96u);
    float4 b[24];
#pragma unroll
    for (int u = 0; u < 24; ++u) b[u] = r4[u];
#pragma unroll
    for (int u = 0; u < 24; ++u) {
      const float4 qv = reinterpret_cast<const float4*>(qj)[u];
      acc = acc + qv.x * b[u].x;
      acc = acc + qv.y * b[u].y;
      acc = acc + qv.z * b[u].z;
      acc = acc + qv.w * b[u].w;
    }
  } else if (P == MRL_RERANK_FP16) {
    const uint4* r4 = reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.data) + row * 768u + j * 96u);
    uint4 b[12];
#pragma unroll
    for (int u = 0; u < 12; ++u) b[u] = r4[u];
#pragma unroll
    for (int u = 0; u < 12; ++u) {
      const uint32_t wd[4] = {b[u].x, b[u].y, b[u].z, b[u].w};
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const float lo = h2f((uint16_t)(wd[h] & 0xffffu));
        const float hi = h2f((uint16_t)(wd[h] >> 16));
        acc = acc + qj[8 * u + 2 * h] * lo;
        acc = acc + qj[8 * u + 2 * h + 1] * hi;
      }
    }
  } else {
    const uint4* r4 = reinterpret_cast<const uint4*>(static_cast<const int8_t*>(a.data) + row * 768u + j * 96u);
    uint4 b[6];
#pragma unroll
    for (int u = 0; u < 6; ++u) b[u] = r4[u];
#pragma unroll
    for (int u = 0; u < 6; ++u) {
      const uint32_t wd[4] = {b[u].x, b[u].y, b[u].z, b[u].w};
#pragma unroll
      for (int h = 0; h < 4; ++h) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float c = (float)(int8_t)((wd[h] >> (8 * e)) & 0xffu);
          acc = acc + qj[16 * u + 4 * h + e] * c;
        }
      }
    }
  }
  return acc;
}

template <int P>
__global__ __launch_bounds__(kScoreThreads) void k_score768(RerankArgs a, uint32_t n_chunks) {
  __shared__ __align__(16) float s_q[8 * kQStride];
  const uint32_t q = blockIdx.x / n_chunks;
  const uint32_t base = (blockIdx.x % n_chunks) * (kScoreThreads / 8);
  const uint32_t cnt = count_of(a, q);
  if (base >= cnt) return;  // uniform over the workgroup
  // query element i = 8t + j at s_q[kQStride*j + t]
  const float* qv = a.queries + (uint64_t)q * 768u;
  for (uint32_t i = threadIdx.x; i < 768u; i += kScoreThreads) s_q[kQStride * (i & 7u) + (i >> 3)] = qv[i];
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63u, j = lane & 7u;
  const uint32_t c = base + threadIdx.x / 8u;
  uint64_t row = ~0ull;
  bool ok = false;
  if (c < cnt) resolve_row(a, q, c, &row, &ok);
  float acc = 0.0f;
  if (ok) acc = chain768<P>(a, row, j, s_q + kQStride * j);
  // acc0 + acc1 + ... + acc7, left to right, in lane j == 0 of the group
  const uint32_t g0 = lane & ~7u;
  float part[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) part[k] = __shfl(acc, (int)(g0 + k));
  if (j == 0 && c < cnt) {
    float s = part[0] + part[1];
#pragma unroll
    for (int k = 2; k < 8; ++k) s = s + part[k];
    if (P == MRL_RERANK_INT8 && ok) s = s * h2f(a.scales[row]);
    const uint64_t o = (uint64_t)q * a.stride + c;
    a.score[o] = ok ? s : 0.0f;
    a.row[o] = row;
  }
}

// fp32 at dims != 768: sequential sums from -0.0, one lane per candidate.  A
// wave takes kSeqCand candidates; pieces of kSeqDims dims come in with
// coalesced loads, one piece ahead of their use, and their products go through
// the wave's LDS to the lanes that add.  What bounds it: HBM for batches (a
// lane that reads its own row touches a cache line per 4 bytes loaded), for
// few candidates the memory latency of a piece, so 16 per wave: more loads in
// flight per candidate and four times the waves of 64.  WIDE: 16-byte loads,
// where rows start at 16-byte multiples.  us per mrl_rerank_rows call, one
// lane reading its own row -> this: 16 queries of 256 rows x 1024 dims
// 57-64 -> 40, 64 of 256 x 512 60 -> 46.5, 256 of 256 x 1024 167 -> 150 (the
// rest is the transfer of the lists), one of 64 x 1024 38.4 -> 31.5, 64 of
// 256 x 1001 (4-byte loads) 103 -> 61.5.
constexpr uint32_t kSeqCand = 16;
constexpr uint32_t kSeqDims = 128;
constexpr uint32_t kSeqStride = kSeqDims + 4;  // LDS row (16 rows' 16-byte reads cover every bank)
constexpr uint32_t kSeqGroup = kScoreThreads / 64 * kSeqCand;
template <bool WIDE>
__global__ __launch_bounds__(kScoreThreads) void k_score_seq(RerankArgs a, uint32_t n_chunks) {
  __shared__ __align__(16) float s_prod[kScoreThreads / 64][kSeqCand * kSeqStride];
  const uint32_t q = blockIdx.x / n_chunks;
  const uint32_t w = threadIdx.x >> 6, lane = threadIdx.x & 63u;
  const uint32_t base = (blockIdx.x % n_chunks) * kSeqGroup + w * kSeqCand;
  const uint32_t cnt = count_of(a, q);
  if (base >= cnt) return;  // (the wave's; no workgroup barrier follows)
  const uint32_t dims = a.dims;
  const float* qv = a.queries + (uint64_t)q * dims;
  const uint32_t c = base + (lane & (kSeqCand - 1u));
  uint64_t row = kRowBad;
  bool ok = false;
  if (c < cnt) resolve_row(a, q, c, &row, &ok);
  const float* data = static_cast<const float*>(a.data);
  const unsigned long long off = ok ? row * dims : ~0ull;
  // element u of a lane: candidate kStep u + lane / kLanes, kPer dims from lane % kLanes
  constexpr uint32_t kPer = WIDE ? 4u : 2u;
  constexpr uint32_t kLanes = kSeqDims / kPer, kStep = 64u / kLanes, kLoads = kSeqCand / kStep;
  const uint32_t d = WIDE ? 4u * (lane & (kLanes - 1u)) : lane;  // not WIDE: dims d and d + 64
  float* sp = s_prod[w];
  float v[kLoads][kPer], qd[kPer];
  unsigned long long wide_off[WIDE ? kLoads : 1];
  if constexpr (WIDE) {
#pragma unroll
    for (uint32_t u = 0; u < kLoads; ++u) wide_off[u] = __shfl(off, (int)(kStep * u + lane / kLanes));
  }
  auto load = [&](uint32_t at) {
#pragma unroll
    for (uint32_t e = 0; e < kPer; ++e) {
      const uint32_t i = at + d + (WIDE ? e : 64u * e);
      qd[e] = i < dims ? qv[i] : 0.0f;
    }
#pragma unroll
    for (uint32_t u = 0; u < kLoads; ++u) {
      unsigned long long o;
      if constexpr (WIDE)
        o = wide_off[u];
      else  // one candidate for the whole wave
        o = (unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(off >> 32), (int)u) << 32 |
            (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)off, (int)u);
      const float* r = data + o + at + d;
      const uint32_t left = o != ~0ull && at + d < dims ? dims - at - d : 0u;  // of the row, from r on
      if (WIDE) {
        float4 f = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (left) f = *reinterpret_cast<const float4*>(r);
        v[u][0] = f.x;
        v[u][1] = f.y;
        v[u][kPer - 2] = f.z;
        v[u][kPer - 1] = f.w;
      } else {
#pragma unroll
        for (uint32_t e = 0; e < kPer; ++e) v[u][e] = 64u * e < left ? r[64u * e] : 0.0f;
      }
    }
  };
  float s = -0.0f;
  load(0);
  for (uint32_t at = 0; at < dims; at += kSeqDims) {
#pragma unroll
    for (uint32_t u = 0; u < kLoads; ++u) {
      float* o = sp + (kStep * u + lane / kLanes) * kSeqStride + d;
      if (WIDE)
        *reinterpret_cast<float4*>(o) = make_float4(qd[0] * v[u][0], qd[1] * v[u][1], qd[kPer - 2] * v[u][kPer - 2],
                                                    qd[kPer - 1] * v[u][kPer - 1]);
      else
#pragma unroll
        for (uint32_t e = 0; e < kPer; ++e) o[64u * e] = qd[e] * v[u][e];
    }
    wave_lds_sync();
    if (at + kSeqDims < dims) load(at + kSeqDims);
    if (lane < kSeqCand) {
      const float* p = sp + lane * kSeqStride;
      const uint32_t nd = dims - at < kSeqDims ? dims - at : kSeqDims;
      uint32_t t = 0;
      for (; t + 16u <= nd; t += 16u) {
        float4 f[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) f[u] = *reinterpret_cast<const float4*>(p + t + 4 * u);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          s = s + f[u].x;
          s = s + f[u].y;
          s = s + f[u].z;
          s = s + f[u].w;
        }
      }
      for (; t < nd; ++t) s = s + p[t];
    }
    wave_lds_sync();  // the sums are done before the next products
  }
  if (lane < kSeqCand && c < cnt) {
    const uint64_t o = (uint64_t)q * a.stride + c;
    a.score[o] = ok ? s : 0.0f;
    a.row[o] = row;
  }
}

// ---------------------------------------------------------------------------
// stable descending sort of one query's scored candidates
// ---------------------------------------------------------------------------
__device__ void bitonic_desc(uint64_t* s, int n2) {
  for (int size = 2; size <= n2; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = threadIdx.x; i < n2 / 2; i += blockDim.x) {
        const int lo = 2 * i - (i & (stride - 1));
        const int hi = lo + stride;
        const bool desc = (lo & size) == 0;
        const uint64_t x = s[lo], y = s[hi];
        if (desc ? (x < y) : (x > y)) {
          s[lo] = y;
          s[hi] = x;
        }
      }
      __syncthreads();
    }
  }
}

// Key = (score key, ~position): descending keys give score descending, then
// input position ascending -- the order of a stable sort.  Keys are distinct;
// skipped ring hits get a zero score key, below every scored entry (the
// smallest score key, that of -inf, is 0x007fffff), and are not emitted.
__global__ __launch_bounds__(kSortThreads) void k_rerank_sort(RerankArgs a) {
  __shared__ uint64_t s_key[kSortCap];
  __shared__ uint16_t s_order[kRankMax];
  __shared__ uint32_t s_bad, s_skip;
  const uint32_t q = blockIdx.x, tid = threadIdx.x;
  const uint32_t m = count_of(a, q);
  const uint64_t base = (uint64_t)q * a.stride;
  if (tid == 0) {
    s_bad = 0u;
    s_skip = 0u;
  }
  __syncthreads();
  uint32_t bad = 0u, skip = 0u;
  for (uint32_t i = tid; i < m; i += kSortThreads) {
    const float s = a.score[base + i];
    const uint64_t r = a.row[base + i];
    uint32_t key = score_key(s);
    if (r == kRowSkip) {
      key = 0u;
      ++skip;
    } else {
      if (!(s == s)) bad |= 1u;     // partial_cmp(..).unwrap() panics
      if (r == kRowBad) bad |= 2u;  // row index out of range
    }
    s_key[i] = ((uint64_t)key << 32) | (uint64_t)(~i);
  }
  if (bad) atomicOr(&s_bad, bad);
  if (skip) atomicAdd(&s_skip, skip);
  __syncthreads();
  // The order first, then rows and scores in order with whole-wave stores (the
  // outputs may lie in host memory, behind PCIe); zeros past the list.  Writing
  // 256 x 256 rows and scores there instead of to HBM and copying them:
  // 168.5 -> 142.9 us per mrl_rerank_rows call (fp32, 768 dims).
  const bool small = m <= (uint32_t)kRankMax;
  if (small) {
    for (uint32_t i = tid; i < m; i += kSortThreads) {
      const uint64_t key = s_key[i];
      uint32_t r = 0;
      for (uint32_t k = 0; k < m; ++k) r += s_key[k] > key ? 1u : 0u;
      s_order[r] = (uint16_t)i;
    }
    __syncthreads();
  } else {
    int n2 = 1;
    while ((uint32_t)n2 < m) n2 <<= 1;
    for (uint32_t i = m + tid; i < (uint32_t)n2; i += kSortThreads) s_key[i] = 0ull;
    __syncthreads();
    bitonic_desc(s_key, n2);
  }
  for (uint32_t r = tid; r < a.stride; r += kSortThreads) {
    const bool in = r < m;
    const uint32_t i = !in ? 0u : small ? (uint32_t)s_order[r] : ~(uint32_t)s_key[r];
    a.out_rows[base + r] = in ? a.row[base + i] : 0ull;
    a.out_scores[base + r] = in ? a.score[base + i] : 0.0f;
  }
  if (a.signal) signal_barrier();  // every thread's outputs before the status
  if (tid == 0) {
    const uint32_t status = s_bad | (a.scan_status ? (a.scan_status[q] & 7u) << 8 : 0u);
    if (a.out_counts) a.out_counts[q] = m - s_skip;
    if (a.signal) signal_status(a.status + q, status);
    else a.status[q] = status;
  }
}

// IndexEngine::query_filtered's ring merge (src/engine.rs:584-594): the ring
// hits, sorted descending, are pushed one by one into the query's Shortlist
// holding the scan hits (Shortlist::push, src/scan.rs:351-369), then
// into_sorted.  Pushing a descending sequence keeps the K largest of both
// lists where a ring hit never displaces an entry of equal score (push
// replaces the minimum only if strictly greater; below capacity it appends).
// So the result is the merge of the two sorted lists with the scan entry first
// on equal scores, cut at K.  Entry positions come from binary searches:
// scan entry i lands at i + #(ring > s_i), ring entry j at j + #(scan >= r_j).
__device__ __forceinline__ uint32_t count_greater(const float* v, uint32_t n, float x, bool or_equal) {
  uint32_t lo = 0, hi = n;  // v descending: first index whose value fails the test
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    const bool pass = or_equal ? (v[mid] >= x) : (v[mid] > x);
    if (pass) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

__global__ __launch_bounds__(kSortThreads) void k_ring_merge(RingMergeArgs a) {
  const uint32_t q = blockIdx.x;
  const uint64_t sb = (uint64_t)q * a.k, rb = (uint64_t)q * a.n_ring;
  const uint32_t c = a.counts[q];
  const bool ok = a.ring_status[q] == 0u;
  const uint32_t r = ok ? (a.n_ring < a.k ? a.n_ring : a.k) : 0u;  // search_exact truncates to top_k
  const float* ss = a.scores + sb;
  const float* rs = a.ring_scores + rb;
  for (uint32_t i = threadIdx.x; i < c; i += kSortThreads) {
    const uint32_t pos = i + count_greater(rs, r, ss[i], false);
    if (pos < a.k) {
      a.out_ids[sb + pos] = a.ids[sb + i];
      a.out_scores[sb + pos] = ss[i];
    }
  }
  for (uint32_t j = threadIdx.x; j < r; j += kSortThreads) {
    const uint32_t pos = j + count_greater(ss, c, rs[j], true);
    if (pos < a.k) {
      // VectorId::new(u32::MAX, local_i as u16)
      a.out_ids[sb + pos] = (0xffffffffull << 16) | (a.ring_rows[rb + j] & 0xffffull);
      a.out_scores[sb + pos] = rs[j];
    }
  }
  if (threadIdx.x == 0) a.out_counts[q] = (c + r < a.k) ? c + r : a.k;
}

// Up to kRingFused pending rows against one query per workgroup: dot, sort,
// and the merge of k_ring_merge or the first `keep` hits.  The products of 64
// rows x 256 dims at a time go to LDS (coalesced loads, the next piece in
// flight during the sums); the additions run in the reference's order, at 768
// dims eight accumulators per row in threads of their own, else one lane per
// row.  What bounds it: latency (63 rows x 512 dims: 126 KB from L2 per query,
// and a chain of 512 additions).  The whole merge call (16 queries, 63 pending
// rows of 512 dims, behind a scan of 250,000 vectors): 243 -> 184 us, in place
// of score, sort and merge launches, four allocations and six copies.
constexpr int kRingThreads = 1024;
constexpr int kRingTileDims = 256;
constexpr uint32_t kRingRowStep = kRingThreads / kRingTileDims;  // rows loaded at a time
constexpr int kRingStride = kRingTileDims + 4;  // LDS row (16 rows' 16-byte reads cover every bank)
template <bool D768>
__global__ __launch_bounds__(kRingThreads) void k_ring(RingArgs a) {
  // products of a piece, then the shortlist's ids
  __shared__ __align__(16) float s_prod[64 * kRingStride];
  static_assert(sizeof(float) * 64 * kRingStride >= 8 * MRL_MAX_SHORTLIST, "the ids fit");
  __shared__ float s_list[MRL_MAX_SHORTLIST];
  __shared__ float s_part[D768 ? 64 * 8 : 1];
  __shared__ uint64_t s_key[kRingFused];
  __shared__ float s_ring[kRingFused];  // sorted scores
  __shared__ uint32_t s_row[kRingFused];
  __shared__ uint32_t s_bad;
  const uint32_t q = blockIdx.x, tid = threadIdx.x, n = a.n_ring;
  const bool merge = a.ids != nullptr;
  const uint32_t gate = a.gate ? a.gate[q] : 0u;
  bool stop = false;
  if (a.gate) {
    uint32_t any = 0u;
    for (uint32_t i = tid; i < a.n_q; i += kRingThreads) any |= a.gate[i];
    stop = __syncthreads_or((int)any) != 0;
  }
  if (tid == 0) s_bad = 0u;
  if (stop) {  // (uniform) the host resolves the scan first
    if (tid == 0) a.out_status[q] = gate;
    return;
  }
  const uint32_t k = merge ? a.k : 0u;
  const uint32_t c = merge ? a.counts[q] : 0u;
  for (uint32_t i = tid; i < c; i += kRingThreads) s_list[i] = a.scores[(uint64_t)q * k + i];

  const float* qv = a.queries + (uint64_t)q * a.dims;
  const uint32_t d = tid & (kRingTileDims - 1u);
  for (uint32_t g = 0; g < n; g += 64u) {  // groups of 64 rows
    const uint32_t rows = n - g < 64u ? n - g : 64u;
    float acc0 = D768 ? zero_acc() : -0.0f;
    float v[64 / kRingRowStep], qd = 0.0f;
    auto load = [&](uint32_t base) {  // element u of a thread: row kRingRowStep u + tid / kRingTileDims, dim base + d
      const bool in = base + d < a.dims;
      qd = in ? qv[base + d] : 0.0f;
#pragma unroll
      for (uint32_t u = 0; u < 64u / kRingRowStep; ++u) {
        const uint32_t r = kRingRowStep * u + tid / kRingTileDims;
        v[u] = in && r < rows ? a.rows[(uint64_t)(g + r) * a.dims + base + d] : 0.0f;
      }
    };
    load(0);
    for (uint32_t base = 0; base < a.dims; base += kRingTileDims) {
      __syncthreads();  // the previous piece's sums are done
#pragma unroll
      for (uint32_t u = 0; u < 64u / kRingRowStep; ++u)
        s_prod[(kRingRowStep * u + tid / kRingTileDims) * kRingStride + d] = qd * v[u];
      __syncthreads();
      if (base + kRingTileDims < a.dims) load(base + kRingTileDims);
      if (D768) {  // accumulator tid % 8 of row tid / 8
        if (tid < 512u) {
          const float* p0 = s_prod + (tid >> 3) * kRingStride + (tid & 7u);
#pragma unroll
          for (int t = 0; t < kRingTileDims / 8; ++t) acc0 = acc0 + p0[8 * t];
        }
      } else if (tid < 64u) {
        const uint32_t nd = a.dims - base < (uint32_t)kRingTileDims ? a.dims - base : (uint32_t)kRingTileDims;
        const float* p = s_prod + tid * kRingStride;
        uint32_t t = 0;
        for (; t + 16u <= nd; t += 16u) {
          float4 f[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) f[u] = *reinterpret_cast<const float4*>(p + t + 4 * u);
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            acc0 = acc0 + f[u].x;
            acc0 = acc0 + f[u].y;
            acc0 = acc0 + f[u].z;
            acc0 = acc0 + f[u].w;
          }
        }
        for (; t < nd; ++t) acc0 = acc0 + p[t];
      }
    }
    if (D768) {  // acc0 + acc1 + ... + acc7, left to right
      if (tid < 512u) s_part[tid] = acc0;
      __syncthreads();
      if (tid < 64u) {
        acc0 = s_part[8 * tid] + s_part[8 * tid + 1];
#pragma unroll
        for (int j = 2; j < 8; ++j) acc0 = acc0 + s_part[8 * tid + j];
      }
    }
    if (tid < rows) {
      // ties (and -0 against +0) keep the rows' order, as a stable sort does
      s_key[g + tid] = ((uint64_t)score_key(acc0) << 32) | (uint64_t)(~(g + tid));
      if (!(acc0 == acc0)) s_bad = 1u;  // partial_cmp(..).unwrap() panics
      s_ring[g + tid] = acc0;
    }
  }
  __syncthreads();
  // rank sort: the keys are distinct
  float rs = 0.0f;
  uint32_t rank = 0u;
  if (tid < n) {
    const uint64_t key = s_key[tid];
    for (uint32_t j = 0; j < n; ++j) rank += s_key[j] > key ? 1u : 0u;
    rs = s_ring[tid];
  }
  __syncthreads();
  if (tid < n) {
    s_ring[rank] = rs;
    s_row[rank] = tid;
  }
  uint64_t* s_ids = reinterpret_cast<uint64_t*>(s_prod);
  for (uint32_t i = tid; i < c; i += kRingThreads) s_ids[i] = a.ids[(uint64_t)q * k + i];
  __syncthreads();
  if (merge) {
    // positions as in k_ring_merge; a query whose ring search failed is left as is
    const uint32_t r = s_bad ? 0u : (n < k ? n : k);
    for (uint32_t i = tid; i < c; i += kRingThreads) {
      const uint32_t pos = i + count_greater(s_ring, r, s_list[i], false);
      if (pos < k) {
        a.ids[(uint64_t)q * k + pos] = s_ids[i];
        a.scores[(uint64_t)q * k + pos] = s_list[i];
      }
    }
    for (uint32_t j = tid; j < r; j += kRingThreads) {
      const uint32_t pos = j + count_greater(s_list, c, s_ring[j], true);
      if (pos < k) {
        a.ids[(uint64_t)q * k + pos] = (0xffffffffull << 16) | (uint64_t)(s_row[j] & 0xffffu);
        a.scores[(uint64_t)q * k + pos] = s_ring[j];
      }
    }
    if (tid == 0) a.counts[q] = c + r < k ? c + r : k;
  } else {
    for (uint32_t j = tid; j < a.keep; j += kRingThreads) {
      a.out_local[(uint64_t)q * a.keep + j] = s_row[j];
      a.out_scores[(uint64_t)q * a.keep + j] = s_ring[j];
    }
  }
  if (tid == 0) a.out_status[q] = gate | (s_bad ? 0x100u : 0u);
}

template <typename K, typename... Args>
void launch(K kernel, dim3 grid, dim3 block, hipStream_t s, const LaunchEvents& ev, Args... args) {
  if (ev.start) hipExtLaunchKernelGGL(kernel, grid, block, 0, s, ev.start, ev.stop, 0u, args...);
  else hipLaunchKernelGGL(kernel, grid, block, 0, s, args...);
}

}  // namespace

hipError_t launch_rerank_store(const float* rows, uint64_t n_rows, int precision, void* data, uint16_t* scales,
                               hipStream_t s) {
  if (n_rows == 0) return hipSuccess;
  const uint64_t wgs = (n_rows + 3) / 4;
  const dim3 grid((uint32_t)(wgs < 65536 ? wgs : 65536));
  uint8_t* d = static_cast<uint8_t*>(data);
  if (precision == MRL_RERANK_FP32)
    hipLaunchKernelGGL(k_store768<MRL_RERANK_FP32>, grid, dim3(kStoreThreads), 0, s, rows, d, scales, n_rows);
  else if (precision == MRL_RERANK_FP16)
    hipLaunchKernelGGL(k_store768<MRL_RERANK_FP16>, grid, dim3(kStoreThreads), 0, s, rows, d, scales, n_rows);
  else
    hipLaunchKernelGGL(k_store768<MRL_RERANK_INT8>, grid, dim3(kStoreThreads), 0, s, rows, d, scales, n_rows);
  return hipGetLastError();
}

hipError_t launch_ring(const RingArgs& a, hipStream_t s, const LaunchEvents& ev) {
  if (a.n_q == 0) return hipSuccess;
  if (a.n_ring == 0 || a.n_ring > kRingFused || (a.ids && a.k > MRL_MAX_SHORTLIST) || (!a.ids && a.keep > a.n_ring))
    return hipErrorInvalidValue;
  if (a.dims == 768) launch(k_ring<true>, dim3(a.n_q), dim3(kRingThreads), s, ev, a);
  else launch(k_ring<false>, dim3(a.n_q), dim3(kRingThreads), s, ev, a);
  return hipGetLastError();
}

hipError_t launch_ring_merge(const RingMergeArgs& a, hipStream_t s, const LaunchEvents& ev) {
  if (a.n_q == 0) return hipSuccess;
  launch(k_ring_merge, dim3(a.n_q), dim3(kSortThreads), s, ev, a);
  return hipGetLastError();
}

hipError_t launch_rerank(const RerankArgs& a, hipStream_t s, const LaunchEvents& ev_score,
                         const LaunchEvents& ev_sort) {
  if (a.n_q == 0 || a.stride == 0) return hipSuccess;
  if (a.dims == 768) {
    const uint32_t per = kScoreThreads / 8;
    const uint32_t n_chunks = (a.stride + per - 1) / per;
    const dim3 grid(n_chunks * a.n_q);
    if (a.precision == MRL_RERANK_FP32)
      launch(k_score768<MRL_RERANK_FP32>, grid, dim3(kScoreThreads), s, ev_score, a, n_chunks);
    else if (a.precision == MRL_RERANK_FP16)
      launch(k_score768<MRL_RERANK_FP16>, grid, dim3(kScoreThreads), s, ev_score, a, n_chunks);
    else
      launch(k_score768<MRL_RERANK_INT8>, grid, dim3(kScoreThreads), s, ev_score, a, n_chunks);
  } else {
    const uint32_t n_chunks = (a.stride + kSeqGroup - 1) / kSeqGroup;
    const dim3 grid(n_chunks * a.n_q);
    if (a.dims % 4u == 0 && (reinterpret_cast<uintptr_t>(a.data) & 15u) == 0)
      launch(k_score_seq<true>, grid, dim3(kScoreThreads), s, ev_score, a, n_chunks);
    else
      launch(k_score_seq<false>, grid, dim3(kScoreThreads), s, ev_score, a, n_chunks);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  launch(k_rerank_sort, dim3(a.n_q), dim3(kSortThreads), s, ev_sort, a);
  return hipGetLastError();
}

}  // namespace mrl
