// mrl_encode.hip -- gfx950 encoder: f32 rows -> PaxBlock64 records, byte-identical to
// encode_block_with_fits (src/quantize.rs:36-96) as driven by encode_f32_corpus_par
// (src/encoder.rs:195-219): timestamp = row index, one source id for every row.
//
// One wave per block.  The f32 arithmetic keeps the reference's operations and order
// (-ffp-contract=off, correctly rounded division/sqrt, IEEE denormals):
//  - lane = vector: running sums (norms, EDEN inner products) add a vector's terms in
//    index order, and the FWHT stages combine registers of one lane, element j with
//    j + h, as the reference's in-place loops do;
//  - the bitplanes are wave ballots (bit v of plane word d = slot v);
//  - CRC-32 of the 4096 bytes: lane k folds bytes 64k..64k+63 into a register from
//    zero (four at a time, slicing tables), the registers are moved to the end of the block with precomputed
//    zero-extension maps and xor-ed (CRC is linear over GF(2)), then the
//    all-ones initial register and final xor are applied.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "mrl_half.h"
#include "mrl_internal.h"

namespace mrl {

namespace {

// tail_rademacher / rademacher_diag sign (rotate.rs:53-67, eden.rs:75-88)
__host__ __device__ constexpr bool mix_negative(uint64_t a, uint64_t i) {
  uint64_t x = (a * 0x9E3779B97F4A7C15ull + i) * 0xBF58476D1CE4E5B9ull;
  x ^= x >> 30;
  x = x * 0x94D049BB133111EBull;
  x ^= x >> 27;
  return (x & 1ull) != 0;
}
// bit i set: sign i of row a is -1
__host__ __device__ constexpr uint64_t mix_mask(uint64_t a, uint64_t first) {
  uint64_t m = 0;
  for (uint64_t i = 0; i < 64; ++i) m |= (uint64_t)mix_negative(a, first + i) << i;
  return m;
}
static_assert(kTailFoldBlocks == 9, "kFoldSigns lists nine blocks");
__device__ constexpr uint64_t kFoldSigns[kTailFoldBlocks] = {
    mix_mask(0, 0), mix_mask(1, 0), mix_mask(2, 0), mix_mask(3, 0), mix_mask(4, 0),
    mix_mask(5, 0), mix_mask(6, 0), mix_mask(7, 0), mix_mask(8, 0)};

__device__ __forceinline__ float sign_of(uint64_t mask, int i) { return (mask >> i) & 1ull ? -1.0f : 1.0f; }

__device__ __forceinline__ float rclamp(float x, float lo, float hi) {
  if (x < lo) x = lo;
  if (x > hi) x = hi;
  return x;
}

// Rust `f32 as u8`: saturating, NaN -> 0
__device__ __forceinline__ uint32_t as_u8(float x) {
  if (!(x == x) || x <= 0.0f) return 0u;
  if (x >= 255.0f) return 255u;
  return (uint32_t)x;
}

// Both values are at hand: a select, never a branch.
__device__ __forceinline__ float sel(bool c, float yes, float no) { return c ? yes : no; }

// In-place FWHT stages over 64 elements of one lane (the reference's in-place
// loops, rotate.rs / eden.rs: low + high, low - high per stage).
__device__ __forceinline__ void fwht64(float (&y)[64]) {
#pragma unroll
  for (int h = 1; h < 64; h <<= 1) {
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      if (i & h) continue;
      const float lo = y[i], hi = y[i + h];
      y[i] = lo + hi;
      y[i + h] = lo - hi;
    }
  }
}

// v_writelane_b32: lane `lane` of old becomes v (a wave-uniform value).
extern "C" __device__ __attribute__((const)) uint32_t mrl_writelane(uint32_t v, uint32_t lane, uint32_t old) __asm(
    "llvm.amdgcn.writelane.i32");

// One bitplane of a block: lane d collects plane word d (bit v = slot v).
struct Plane {
  uint32_t lo = 0, hi = 0;
  __device__ __forceinline__ void set(int d, bool bit) {
    const uint64_t b = __ballot(bit);
    lo = mrl_writelane((uint32_t)b, (uint32_t)d, lo);
    hi = mrl_writelane((uint32_t)(b >> 32), (uint32_t)d, hi);
  }
  __device__ __forceinline__ void store(uint8_t* at, uint32_t lane, uint64_t valid) const {
    reinterpret_cast<uint2*>(at)[lane] = make_uint2(lo & (uint32_t)valid, hi & (uint32_t)(valid >> 32));
  }
};

// Makes this wave's LDS writes visible to its own later reads.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Keeps the scheduler from interleaving unrolled groups of elements past this
// point (their masks and scalars would spill).
__device__ __forceinline__ void group_end(int i, int n) {
  if (i % n == n - 1) __builtin_amdgcn_sched_barrier(0);
}

constexpr int kEncWaves = 4;          // waves per workgroup, one block each
constexpr int kEncTile = 64 * 64 * 4;  // LDS bytes per wave: 64 rows x 64 dims
constexpr uint32_t kEncVecDims = 1u << 22;  // the 16-byte loads index a block's rows with 31 bits

// The lane number, opaque to the optimiser: what is computed from it is
// recomputed where it is used, instead of kept in registers over the loops.
__device__ __forceinline__ uint32_t fresh(uint32_t lane) {
  asm volatile("" : "+v"(lane));
  return lane;
}

__device__ __forceinline__ uint64_t fresh(uint64_t mask) {  // wave-uniform
  asm volatile("" : "+s"(mask));
  return mask;
}

// The 64 x 64 piece of a block's rows starting at dim 64 ch, as one wave holds
// it on the way into LDS.  VEC: float4 k of a lane is row 4k + lane / 16,
// dims 4 (lane % 16) .., read through a buffer descriptor that ends with the
// block's last row, so rows past it (and dims past the end, sent there) read
// as zero.  Otherwise element j is row j (the last one again past the end),
// dim `lane`.  What rows past the last one hold is masked out of the record.
template <bool VEC>
__device__ __forceinline__ void load_piece(const EncodeArgs& a, uint64_t b, uint32_t ch, uint32_t lane0, float (&p)[64]) {
  const uint64_t row0 = b * 64;
  const uint32_t rows = (uint32_t)((a.n - row0) < 64 ? (a.n - row0) : 64);
  const uint32_t lane = fresh(lane0);
  const float* base = a.x + row0 * a.dims;
  if (VEC) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(base), (short)0, (int)(rows * a.dims * 4u), 0x00020000);
    const uint32_t c = 64u * ch + 4u * (lane & 15u);
    const uint32_t at = c < a.dims ? ((lane >> 4) * a.dims + c) * 4u : 0xc0000000u;  // rows * dims * 4 < 2^31
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const auto f = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(at + (uint32_t)k * 16u * a.dims), 0, 0);
      p[4 * k] = __uint_as_float(f[0]);
      p[4 * k + 1] = __uint_as_float(f[1]);
      p[4 * k + 2] = __uint_as_float(f[2]);
      p[4 * k + 3] = __uint_as_float(f[3]);
    }
  } else {
    const uint32_t c = 64u * ch + lane;
    const bool in = c < a.dims;
#pragma unroll
    for (int j = 0; j < 64; ++j) {
      const uint32_t row = (uint32_t)j < rows ? (uint32_t)j : rows - 1u;
      p[j] = in ? base[(uint64_t)row * a.dims + c] : 0.0f;
    }
  }
}

// The piece through LDS into x: lane v gets row v.  16-byte column c of row r
// sits at column c ^ (r % 16) of the tile, so both the writes (16 lanes per
// row) and the reads (one column of 16 consecutive rows) cover every bank.
template <bool VEC>
__device__ __forceinline__ void transpose(uint8_t* tile, uint32_t lane0, const float (&p)[64], float (&x)[64]) {
  const uint32_t lane = fresh(lane0);
  __builtin_amdgcn_sched_barrier(0);
  wave_lds_sync();  // the tile's previous readers are done
  if (VEC) {
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const uint32_t r = 4u * k + (lane >> 4);
      *reinterpret_cast<float4*>(tile + r * 256u + (((lane & 15u) ^ (r & 15u)) << 4)) =
          make_float4(p[4 * k], p[4 * k + 1], p[4 * k + 2], p[4 * k + 3]);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 64; ++j)
      *reinterpret_cast<float*>(tile + j * 256 + (((lane >> 2) ^ (j & 15)) << 4) + ((lane & 3u) << 2)) = p[j];
  }
  wave_lds_sync();
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    const float4 f = *reinterpret_cast<const float4*>(tile + lane * 256u + ((c ^ (lane & 15u)) << 4));
    x[4 * c] = f.x;
    x[4 * c + 1] = f.y;
    x[4 * c + 2] = f.z;
    x[4 * c + 3] = f.w;
  }
  __builtin_amdgcn_sched_barrier(0);
}

}  // namespace

// What bounds it: HBM (4 dims + 64 bytes per row).  Every f32 chain of a row
// (norms, inner products, the FWHT stages in registers) runs in one lane, in
// the reference's order, so no step crosses lanes; the rows' 64-dim pieces
// come in with coalesced 16-byte loads one piece ahead of their use and are
// transposed through 16 KB of LDS per wave.  One wave per SIMD: a wave then
// has 512 registers for the piece in flight (64), the piece at work (64), the
// first half of the mid band or the folded tail (64) and their temporaries.
// Measured: 1M x 768 EDEN 12,990 -> 615 us (5.1 TB/s; a device copy reaches
// 4.8 there), 130,999 x 1024 MinMax4 1,624 -> 140 us, against one wave per
// block with lane = vector sums and lane = dim transforms over LDS.  Two
// waves per SIMD (256 registers) spill: 1,083 and 177 us.
template <bool EDEN, bool B1, bool VEC>
__global__ __launch_bounds__(64 * kEncWaves, kEncWaves / 4) void k_encode(EncodeArgs a) {
  __shared__ __align__(16) uint8_t s_tile[kEncWaves][kEncTile];
  __shared__ uint32_t s_crc[1024];  // slicing tables: [k][i] = byte i followed by k zero bytes
  __shared__ float s_cw[16];        // eden_codebook[l] * inv_sqrt64
  __shared__ __align__(16) float s_mean[192];
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (uint32_t i = threadIdx.x; i < 1024u; i += 64u * kEncWaves) s_crc[i] = a.crc_tab[i];
  const float inv64 = a.c.inv_sqrt64, inv128 = a.c.inv_sqrt128;
  if (EDEN && threadIdx.x < 192u) s_mean[threadIdx.x] = a.means[threadIdx.x];
  if (threadIdx.x < 16u) s_cw[threadIdx.x] = a.c.eden_codebook[threadIdx.x] * inv64;
  __syncthreads();

  uint8_t* tile = s_tile[wave];
  const uint32_t dims = a.dims;
  const uint32_t n_pieces = (dims + 63u) / 64u;
  const uint32_t tail_blocks = (dims - (uint32_t)kTailStart) / 64u;
  const uint32_t fold_end =
      3u + (tail_blocks < (uint32_t)kTailFoldBlocks ? tail_blocks : (uint32_t)kTailFoldBlocks);  // first piece not folded
  // level thresholds in registers (an instruction reads one scalar operand)
  float thr[15];
  if (EDEN) {
#pragma unroll
    for (int i = 0; i < 15; ++i) {
      thr[i] = a.level_max[i];
      asm volatile("" : "+v"(thr[i]));
    }
  }

  // consecutive blocks go to consecutive workgroups, so that a short input spreads over the CUs
  const uint64_t step = (uint64_t)gridDim.x * kEncWaves;
  uint64_t b = (uint64_t)wave * gridDim.x + blockIdx.x;
  float p[64], x[64];
  if (b < a.n_blocks) load_piece<VEC>(a, b, 0, lane, p);
  for (; b < a.n_blocks; b += step) {
    const uint64_t row0 = b * 64;
    const uint32_t rows = (uint32_t)((a.n - row0) < 64 ? (a.n - row0) : 64);
    const uint64_t valid = rows < 64u ? (1ull << rows) - 1ull : ~0ull;

    float scale, offset;
    Plane l3, l2, l1, l0, s1a, s1b, s4;
    // ---- prefix: EDEN-prod (quantize.rs:265-295, eden.rs:225-269) or MinMax4 (220-246)
    transpose<VEC>(tile, lane, p, x);
    load_piece<VEC>(a, b, 1, lane, p);
    if (EDEN) {
      float nsq = 0.0f;
#pragma unroll
      for (int i = 0; i < 64; ++i) {
        x[i] = x[i] - s_mean[i];
        nsq += x[i] * x[i];
        group_end(i, 16);
      }
      const float cn = fmaxf(sqrtf(nsq), 1e-12f);
      const float inv = 1.0f / cn;
      const uint64_t sg = fresh(a.eden_signs);
#pragma unroll
      for (int i = 0; i < 64; ++i) {
        x[i] = (x[i] * inv) * sign_of(sg, i);
        group_end(i, 16);
      }
      fwht64(x);
      float ip = 0.0f;
#pragma unroll
      for (int i = 0; i < 64; ++i) {
        // the level is the number of thresholds below t (EncodeArgs::level_max): four steps of a binary search
        const float z = x[i] * inv64;
        const float t = z * a.sqrt64;
        const bool b3 = t > thr[7];
        const bool b2 = t > sel(b3, thr[11], thr[3]);
        const bool b1 = t > sel(b2, sel(b3, thr[13], thr[5]), sel(b3, thr[9], thr[1]));
        const bool b0 = t > sel(b1, sel(b2, sel(b3, thr[14], thr[6]), sel(b3, thr[10], thr[2])),
                                sel(b2, sel(b3, thr[12], thr[4]), sel(b3, thr[8], thr[0])));
        l3.set(i, b3);
        l2.set(i, b2);
        l1.set(i, b1);
        l0.set(i, b0);
        ip += z * s_cw[(b3 ? 8u : 0u) | (b2 ? 4u : 0u) | (b1 ? 2u : 0u) | (b0 ? 1u : 0u)];
        group_end(i, 4);
      }
      const float s = fabsf(ip) > 1e-12f ? 1.0f / ip : 0.0f;
      scale = cn * s;
      offset = 0.0f;
    } else {
      float mn = INFINITY, mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 64; ++i) mn = fminf(mn, x[i]);
#pragma unroll
      for (int i = 0; i < 64; ++i) mx = fmaxf(mx, x[i]);
      const float range = fmaxf(mx - mn, 1e-8f);
      scale = range / 15.0f;
      offset = mn;
#pragma unroll
      for (int i = 0; i < 64; ++i) {
        // levels 0..15 as floats; a NaN has no bit set (`as u8` gives 0)
        const float l = rclamp(roundf((x[i] - offset) / scale), 0.0f, 15.0f);
        const bool b3 = l >= 8.0f;
        const float r3 = b3 ? l - 8.0f : l;
        const bool b2 = r3 >= 4.0f;
        const float r2 = b2 ? r3 - 4.0f : r3;
        const bool b1 = r2 >= 2.0f;
        const float r1 = b1 ? r2 - 2.0f : r2;
        l3.set(i, b3);
        l2.set(i, b2);
        l1.set(i, b1);
        l0.set(i, r1 >= 1.0f);
        group_end(i, 4);
      }
    }

    // ---- mid band: EdenB1 (eden.rs:225-269 with d = 128, b = 1) or RaBitQ signs (quantize.rs:199-206)
    float msq = 0.0f, nsq = 0.0f;
    {
      float y[64];
      transpose<VEC>(tile, lane, p, y);
      load_piece<VEC>(a, b, 2, lane, p);
#pragma unroll
      for (int i = 0; i < 64; ++i) {
        msq += y[i] * y[i];
        group_end(i, 16);
      }
      if (B1) {
#pragma unroll
        for (int i = 0; i < 64; ++i) {
          y[i] = y[i] - s_mean[64 + i];
          nsq += y[i] * y[i];
          group_end(i, 16);
        }
      } else {
        fwht64(y);
      }
      transpose<VEC>(tile, lane, p, x);
      if (n_pieces > 3u) load_piece<VEC>(a, b, 3, lane, p);
      else if (b + step < a.n_blocks) load_piece<VEC>(a, b + step, 0, lane, p);
#pragma unroll
      for (int i = 0; i < 64; ++i) {
        msq += x[i] * x[i];
        group_end(i, 16);
      }
      float cn = 0.0f;
      if (B1) {
#pragma unroll
        for (int i = 0; i < 64; ++i) {
          x[i] = x[i] - s_mean[128 + i];
          nsq += x[i] * x[i];
          group_end(i, 16);
        }
        cn = fmaxf(sqrtf(nsq), 1e-12f);
        const float inv = 1.0f / cn;
        const uint64_t sg0 = fresh(a.mid_signs[0]), sg1 = fresh(a.mid_signs[1]);
#pragma unroll
        for (int i = 0; i < 64; ++i) {
          y[i] = (y[i] * inv) * sign_of(sg0, i);
          group_end(i, 16);
        }
#pragma unroll
        for (int i = 0; i < 64; ++i) {
          x[i] = (x[i] * inv) * sign_of(sg1, i);
          group_end(i, 16);
        }
        fwht64(y);
      }
      fwht64(x);
#pragma unroll
      for (int i = 0; i < 64; ++i) {  // the 128-point transform's last stage
        const float lo = y[i], hi = x[i];
        y[i] = (lo + hi) * inv128;
        x[i] = (lo - hi) * inv128;
      }
      if (B1) {
        const float cw0 = a.c.eden_mid_codebook[0] * inv128, cw1 = a.c.eden_mid_codebook[1] * inv128;
        float ip = 0.0f;
#pragma unroll
        for (int i = 0; i < 64; ++i) {
          const bool up = y[i] * a.sqrt128 > a.mid_level_max;
          s1a.set(i, up);
          ip += y[i] * (up ? cw1 : cw0);
          group_end(i, 8);
        }
#pragma unroll
        for (int i = 0; i < 64; ++i) {
          const bool up = x[i] * a.sqrt128 > a.mid_level_max;
          s1b.set(i, up);
          ip += x[i] * (up ? cw1 : cw0);
          group_end(i, 8);
        }
        const float s = fabsf(ip) > 1e-12f ? 1.0f / ip : 0.0f;
        offset = cn * s;
      } else {
#pragma unroll
        for (int i = 0; i < 64; ++i) {
          s1a.set(i, y[i] >= 0.0f);
          group_end(i, 16);
        }
#pragma unroll
        for (int i = 0; i < 64; ++i) {
          s1b.set(i, x[i] >= 0.0f);
          group_end(i, 16);
        }
      }
    }

    // ---- folded tail (rotate.rs:73-100, quantize.rs:207-213) and the tail norm
    float hsq = 0.0f;
    {
      float t[64];
#pragma unroll
      for (int i = 0; i < 64; ++i) t[i] = 0.0f;
      for (uint32_t ch = 3; ch < n_pieces; ++ch) {
        transpose<VEC>(tile, lane, p, x);
        if (ch + 1u < n_pieces) load_piece<VEC>(a, b, ch + 1u, lane, p);
        else if (b + step < a.n_blocks) load_piece<VEC>(a, b + step, 0, lane, p);
#pragma unroll
        for (int i = 0; i < 64; ++i) {
          hsq += x[i] * x[i];
          group_end(i, 16);
        }
        if (ch < fold_end) {
          // t + sign * x: the product with +-1 is exact, so one fused operation rounds as the two do
          const uint64_t m = kFoldSigns[ch - 3u];
#pragma unroll
          for (int i = 0; i < 64; ++i) {
            t[i] = __builtin_fmaf(x[i], sign_of(m, i), t[i]);
            group_end(i, 16);
          }
        }
      }
      fwht64(t);
#pragma unroll
      for (int i = 0; i < 64; ++i) {
        s4.set(i, t[i] * inv64 >= 0.0f);
        group_end(i, 16);
      }
    }

    // ---- the record, in the wave's tile
    const float rest = sqrtf(msq + hsq);
    const float high = sqrtf(hsq);
    uint32_t flags = 0;
    if (!(rest <= 1e-12f)) flags = as_u8(rclamp(roundf(rclamp(high / rest, 0.0f, 1.0f) * 255.0f), 0.0f, 255.0f));
    wave_lds_sync();
    uint8_t* img = tile;
    if (lane < 16u) reinterpret_cast<uint32_t*>(img)[lane] = 0u;
    wave_lds_sync();
    {
      uint8_t* mt = img + kOrigMeta + 7 * lane;
      const bool live = lane < rows;
      const uint32_t hs = live ? f32_to_f16(scale) : 0u, ho = live ? f32_to_f16(offset) : 0u,
                     hr = live ? f32_to_f16(rest) : 0u;
      mt[0] = (uint8_t)hs;
      mt[1] = (uint8_t)(hs >> 8);
      mt[2] = (uint8_t)ho;
      mt[3] = (uint8_t)(ho >> 8);
      mt[4] = (uint8_t)hr;
      mt[5] = (uint8_t)(hr >> 8);
      mt[6] = (uint8_t)(live ? flags : 0u);
    }
    l3.store(img + kOrigS0, lane, valid);
    s1a.store(img + kOrigS1, lane, valid);
    s1b.store(img + kOrigS1 + 512, lane, valid);
    l2.store(img + kOrigS2, lane, valid);
    l1.store(img + kOrigS3, lane, valid);
    s4.store(img + kOrigS4, lane, valid);
    l0.store(img + kOrigS5, lane, valid);
    if (lane == 0) {
      uint32_t* h = reinterpret_cast<uint32_t*>(img);
      h[0] = (uint32_t)row0;               // min_timestamp
      h[1] = (uint32_t)(row0 + rows - 1);  // max_timestamp
      h[2] = a.source;                     // source_mask
      h[4] = (uint32_t)~valid;             // tombstones: the slots past the last row
      h[5] = (uint32_t)(~valid >> 32);
    }
    if (a.cluster) {
      // cluster-grouped convention: coarse_cluster_id and block_flags (block.rs:38-39) when every row of the
      // block is in one cluster below 65536
      const uint32_t c = lane < rows ? a.cluster[row0 + lane] : 0u;
      const uint32_t c0 = __shfl(c, 0);
      const bool one = __ballot(lane < rows && c != c0) == 0 && c0 < 65536u;
      if (lane == 0 && one) reinterpret_cast<uint32_t*>(img)[3] = c0 | (kBlockFlagOneCluster << 16);
    }
    wave_lds_sync();

    // ---- CRC-32 (recompute_crc, block.rs:186-190) over the block with crc = 0: lane k folds bytes 64k..64k+63,
    // four at a time
    uint32_t c = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint4 w4 = reinterpret_cast<const uint4*>(img)[4 * lane + j];
      const uint32_t w[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        c ^= w[k];
        c = s_crc[768 + (c & 0xffu)] ^ s_crc[512 + ((c >> 8) & 0xffu)] ^ s_crc[256 + ((c >> 16) & 0xffu)] ^
            s_crc[c >> 24];
      }
    }
    uint32_t z = 0;
    const uint4* zt = reinterpret_cast<const uint4*>(a.crc_zt + 32 * lane);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint4 t = zt[i];
      z ^= (0u - ((c >> (4 * i)) & 1u)) & t.x;
      z ^= (0u - ((c >> (4 * i + 1)) & 1u)) & t.y;
      z ^= (0u - ((c >> (4 * i + 2)) & 1u)) & t.z;
      z ^= (0u - ((c >> (4 * i + 3)) & 1u)) & t.w;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) z ^= (uint32_t)__shfl_xor((int)z, off);
    if (lane == 0) reinterpret_cast<uint32_t*>(img)[kOrigCrc / 4] = z ^ a.crc_const;
    wave_lds_sync();
    const uint4* src = reinterpret_cast<const uint4*>(img);
    uint4* dst = reinterpret_cast<uint4*>(a.out + b * kBlockBytes);
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[64 * i + lane] = src[64 * i + lane];
  }
}

// The 16-byte loads need rows that start 16-byte aligned; other row lengths or addresses take 4-byte loads.
template <bool EDEN, bool B1>
static void launch_codec(const EncodeArgs& a, uint32_t grid, hipStream_t s) {
  if ((reinterpret_cast<uintptr_t>(a.x) & 15u) == 0 && a.dims % 4u == 0 && a.dims <= kEncVecDims)
    hipLaunchKernelGGL((k_encode<EDEN, B1, true>), dim3(grid), dim3(64 * kEncWaves), 0, s, a);
  else
    hipLaunchKernelGGL((k_encode<EDEN, B1, false>), dim3(grid), dim3(64 * kEncWaves), 0, s, a);
}

hipError_t launch_encode(const EncodeArgs& args, hipStream_t s) {
  if (args.n_blocks == 0) return hipSuccess;
  static const uint32_t n_cu = [] {
    int dev = 0, n = 0;
    return hipGetDevice(&dev) == hipSuccess &&
                   hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0
               ? (uint32_t)n
               : 256u;
  }();
  EncodeArgs a = args;
  a.eden_signs = mix_mask(a.eden_seed, 0);
  a.mid_signs[0] = mix_mask(a.mid_seed, 0);
  a.mid_signs[1] = mix_mask(a.mid_seed, 64);
  // one workgroup per CU (the tiles take 128 KB of its 160 KB of LDS)
  const uint32_t grid = (uint32_t)(a.n_blocks < n_cu ? a.n_blocks : n_cu);
  if (a.eden && a.mid) launch_codec<true, true>(a, grid, s);
  else if (a.eden) launch_codec<true, false>(a, grid, s);
  else launch_codec<false, false>(a, grid, s);
  return hipGetLastError();
}

}  // namespace mrl
