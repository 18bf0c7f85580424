// Weight-format kernels: int4 and int8 block quantization (src/quant.rs:74-82
// closed form), fp8 e4m3fn repack (reference/fp8_reference.py:83-91), and the
// dequantize kernels that expose the f32 values (src/quant.rs:232,
// src/fp8.rs:306-318) and the bf16 matrix-core operands.
//
// All of these are HBM-bound byte/integer work: 16-byte loads and stores, one
// thread per run of values; the blocked layout's transpose goes through LDS.
#include "lrq_common.h"
#include "lrq_kernels.h"

// ------------------------------------------------------------------ int4 / int8 quantize
// QMAX 7: Q4S, packed nibbles q + 8; QMAX 127: Q8S, int8 bytes (src/quant.rs:156-162).
// One thread per (row, 32-value half-block); a block of `group` values is
// covered by group/32 consecutive threads that reduce absmax with lane
// shuffles (group/32 <= 64 lanes, a power of two or not: a plain loop over
// the partner lanes keeps it exact).
// FP8: the input is e4m3fn bytes [n, k] with a scalar or per-row f32 scale,
// and each value is LUT[byte] * scale in f32 first (src/fp8.rs:306-318), the
// reference's f32 snapshot of an fp8 checkpoint tensor, which its load pass
// then quantizes (src/diffusion_trainer.rs:1143-1169); no f32 copy is kept.
template <bool FP8, int QMAX>
__global__ void __launch_bounds__(256) k_quantize(const void* __restrict__ wv, const float* __restrict__ fsc,
                                                       int per_channel, int64_t n, int64_t k, int g,
                                                       uint8_t* __restrict__ packed, float* __restrict__ scales) {
  const int64_t runs_per_row = k / 32;
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (tid >= n * runs_per_row) return;
  const int64_t row = tid / runs_per_row;
  const int64_t run = tid % runs_per_row;
  float v[32];
  float amax = 0.0f;
  if constexpr (FP8) {
    const uint8_t* src = static_cast<const uint8_t*>(wv) + row * k + run * 32;
    const float sc = fsc[per_channel ? row : 0];
#pragma unroll
    for (int i = 0; i < 32; i += 16) {
      const u32x4 b = ld16(src + i);
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        float f[4];
        fp8x4_to_f32(b[d], f);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[i + 4 * d + e] = f[e] * sc;
      }
    }
  } else {
    const float* src = static_cast<const float*>(wv) + row * k + run * 32;
#pragma unroll
    for (int i = 0; i < 32; i += 4) {
      f32x4 t = *reinterpret_cast<const f32x4*>(src + i);
      v[i] = t[0]; v[i + 1] = t[1]; v[i + 2] = t[2]; v[i + 3] = t[3];
    }
  }
#pragma unroll
  for (int i = 0; i < 32; ++i) amax = fmaxf(amax, fabsf(v[i]));
  // absmax over the whole block: the block's runs are consecutive tids,
  // hence consecutive lanes of one wavefront (g/32 divides... g is a multiple
  // of 32 and rows start at run 0, but a block may straddle two wavefronts
  // when g/32 does not divide 64; the host restricts g/32 to a divisor of 64).
  const int rpb = g / 32;
  if (rpb > 1) {
    const int lane = threadIdx.x & 63;
    const int first = lane - (int)(run % rpb);
    float m = 0.0f;
    for (int j = 0; j < rpb; ++j) m = fmaxf(m, __shfl(amax, first + j, 64));
    amax = m;
  }
  const float s = amax / (float)QMAX;  // correctly rounded f32 division
  if (run % rpb == 0) scales[row * (k / g) + run / rpb] = s;
  // q = clamp(round_half_away(RN(v / s))). The quotient RN(v / s) is formed
  // without a division per value: with y = RN(1 / s), q0 = RN(v y) and the
  // exact remainder r = v - q0 s (one fma), RN(q0 + r y) == RN(v / s)
  // (Markstein: y within half an ulp of 1/s and q0 within one ulp of v/s,
  // no underflow). r stays normal for s >= 2^-80; smaller scales divide.
  int q[32];
  auto to_int = [](float t) {
    const float r = fminf(fmaxf(roundf(t), -(float)QMAX), (float)QMAX);  // half away from zero
    return (int)r;
  };
  if (s >= 0x1p-80f) {
    const float y = 1.0f / s;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const float q0 = v[i] * y;
      const float rem = __builtin_fmaf(-q0, s, v[i]);
      q[i] = to_int(__builtin_fmaf(rem, y, q0));
    }
  } else if (s != 0.0f) {
#pragma unroll
    for (int i = 0; i < 32; ++i) q[i] = to_int(v[i] / s);
  } else {
#pragma unroll
    for (int i = 0; i < 32; ++i) q[i] = 0;
  }
  if constexpr (QMAX == 7) {
    u32x4 o = zero4();
#pragma unroll
    for (int i = 0; i < 32; ++i) o[i >> 3] |= (uint32_t)(q[i] + 8) << (4 * (i & 7));
    st16(packed + row * (k / 2) + run * 16, o);
  } else {
    u32x4 o[2] = {zero4(), zero4()};
#pragma unroll
    for (int i = 0; i < 32; ++i) o[i >> 4][(i >> 2) & 3] |= ((uint32_t)q[i] & 0xffu) << (8 * (i & 3));
    st16(packed + row * k + run * 32, o[0]);
    st16(packed + row * k + run * 32 + 16, o[1]);
  }
}

// ------------------------------------------------------------------ fp8 quantize
// Exact RNE e4m3fn encode of an f32 that is already divided by the scale.
__device__ __forceinline__ uint32_t fp8_encode_rne(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const uint32_t sign = (u >> 24) & 0x80u;
  const uint32_t a = u & 0x7fffffffu;
  if (a > 0x7f800000u) return sign | 0x7fu;     // NaN
  if (a >= 0x43e00000u) return sign | 0x7eu;    // |x| >= 448: saturate
  if (a < 0x3c800000u) {                        // |x| < 2^-6: subnormal grid 2^-9
    const float ax = __builtin_bit_cast(float, a) * 512.0f;  // exact
    const float r = __builtin_rintf(ax);                      // RNE
    return sign | (uint32_t)r;                                // 8 rolls into 0x08
  }
  // normal: keep 3 mantissa bits with RNE on the f32 bit pattern
  const uint32_t lsb = (a >> 20) & 1u;
  const uint32_t rounded = a + 0x7ffffu + lsb;
  const uint32_t e = (rounded >> 23) - 120u;  // fp8 exponent field
  const uint32_t m = (rounded >> 20) & 7u;
  uint32_t code = (e << 3) | m;
  if (code > 0x7eu) code = 0x7eu;
  return sign | code;
}

// The largest |v| over a 256-thread workgroup, in every thread (NaN is passed
// over, as fmaxf does).
LRQ_DEV float wg_max(float m) {
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  __shared__ float red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

LRQ_DEV float fp8_scale(float amax) {
  const float s = amax / 448.0f;
  return s < 1e-12f ? 1e-12f : s;
}

// Four f32 over their scale -> four e4m3fn bytes. The quotient is RN(v / s)
// without a division (as in k_quantize: y = RN(1/s), q0 = RN(v y), exact
// remainder, one fma; s >= 1e-12 and |v/s| <= 448, so no remainder that
// matters underflows; an infinite scale divides), and |v/s| < 464 always, so
// the hardware's round-to-nearest-even conversion never overflows. A NaN
// quotient keeps its sign bit and encodes as 0x7f, like fp8_encode_rne.
LRQ_DEV uint32_t fp8x4_encode(const f32x4& v, float s, float y, bool fast) {
  float q[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (fast) {
      const float q0 = v[j] * y;
      // (the sign of a zero or a NaN would be lost on the way)
      q[j] = __builtin_copysignf(__builtin_fmaf(__builtin_fmaf(-q0, s, v[j]), y, q0), v[j]);
    } else {
      q[j] = v[j] / s;
    }
  }
  uint32_t w = 0;
  if (fast) {
    int r = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
    r = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], r, true);
    w = (uint32_t)r;
    if (q[0] + q[1] + q[2] + q[3] == q[0] + q[1] + q[2] + q[3]) return w;  // no NaN (finite: |q| <= 448)
    w = 0;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) w |= fp8_encode_rne(q[j]) << (8 * j);
  return w;
}

// Per-row amax (the first pass of a scalar scale, and of rows longer than
// k_fp8_rows holds). One workgroup per row, 16-byte loads.
__global__ void __launch_bounds__(256) k_rowabsmax(const float* __restrict__ w, int64_t k,
                                                   float* __restrict__ out) {
  const f32x4* src = reinterpret_cast<const f32x4*>(w + (int64_t)blockIdx.x * k);
  float m = 0.0f;
  for (int64_t i = threadIdx.x; i < k / 4; i += 1024) {
    f32x4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = i + 256 * u < k / 4 ? src[i + 256 * u] : (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) m = fmaxf(m, fabsf(v[u][e]));
  }
  m = wg_max(m);
  if (threadIdx.x == 0) out[blockIdx.x] = m;
}

// Per-row scale and bytes in one pass: a workgroup holds its row (k <= 1024
// NV values) in registers between the absmax and the encoding, so the weight
// is read once. HBM-bound: 5 bytes per value; 9216 x 3072 in 33 us against 75
// us for absmax, scale and encode launches (0.23 GB moved instead of 0.14).
template <int NV>
__global__ void __launch_bounds__(256) k_fp8_rows(const float* __restrict__ w, int64_t k, float* __restrict__ scales,
                                                  uint8_t* __restrict__ out) {
  const int64_t row = blockIdx.x;
  const f32x4* src = reinterpret_cast<const f32x4*>(w + row * k);
  const int n4 = (int)(k / 4);
  f32x4 v[NV];
  float m = 0.0f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (int)threadIdx.x + 256 * i;
    v[i] = c < n4 ? src[c] : (f32x4){0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) m = fmaxf(m, fabsf(v[i][e]));
  const float s = fp8_scale(wg_max(m));
  if (threadIdx.x == 0) scales[row] = s;
  const bool fast = s < 3.0e38f;
  const float y = 1.0f / s;
  uint32_t* dst = reinterpret_cast<uint32_t*>(out + row * k);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (int)threadIdx.x + 256 * i;
    if (c < n4) dst[c] = fp8x4_encode(v[i], s, y, fast);
  }
}

__global__ void __launch_bounds__(256) k_fp8_scales(float* __restrict__ amax, int64_t n,
                                                    int per_channel, float* __restrict__ scales) {
  if (per_channel) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
      scales[i] = fp8_scale(amax[i]);
    }
  } else if (blockIdx.x == 0) {
    float m = 0.0f;
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) m = fmaxf(m, amax[i]);
    m = wg_max(m);
    if (threadIdx.x == 0) scales[0] = fp8_scale(m);
  }
}

__global__ void __launch_bounds__(256) k_fp8_encode(const float* __restrict__ w, int64_t n, int64_t k,
                                                    int per_channel, const float* __restrict__ scales,
                                                    uint8_t* __restrict__ out) {
  // one thread per 4 consecutive values (k % 32 == 0 so rows hold whole runs)
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t total = n * k / 4;
  if (tid >= total) return;
  const int64_t row = (tid * 4) / k;
  const float s = per_channel ? scales[row] : scales[0];
  reinterpret_cast<uint32_t*>(out)[tid] =
      fp8x4_encode(*reinterpret_cast<const f32x4*>(w + tid * 4), s, 1.0f / s, s < 3.0e38f);
}

// ------------------------------------------------------------------ blocked layout
// The fused GEMMs read the frozen weight in 64 (n) x 64 (k) blocks that are
// contiguous in memory (int4: 64 rows x 32 bytes; fp8, int8: 64 rows x 64
// bytes), block (nb, kb) at (nb * KB + kb) * block bytes, KB = ceil(k / 64);
// int4 and int8 scales as [NB][Gp][64] (Gp = 64*KB / group). Rows past n and
// columns past k are padding: int4 nibbles 8 (q = 0) with scale 0, int8 and
// fp8 bytes 0 (int8 with scale 0). A second,
// transposed section of the same size follows (k_block_data_t).
LRQ_DEV int64_t blk_data_off(int fmt, int64_t n, int64_t k, int64_t KB) {
  const int64_t rb = (fmt == LRQ_FMT_INT4) ? 32 : 64;  // bytes per block row
  const int64_t kb = k >> 6, kin = k & 63;
  return (((n >> 6) * KB + kb) * 64 + (n & 63)) * rb + ((fmt == LRQ_FMT_INT4) ? (kin >> 1) : kin);
}

// Both sections and both scale tables in one pass. The second, transposed
// section is read by the input-gradient GEMM (its reduction runs along n):
// the blocked layout of W^T [k, n], i.e. 64 (k) x 64 (n) blocks, block (kb,
// nb) at (kb * NB + nb) * block bytes, block row r = k. int4: 32 bytes per
// row, byte c holding n = 2c in its low nibble and 2c+1 in its high nibble,
// each nibble q in two's complement (the kernel sign-extends it); fp8 and
// int8: 64 bytes per row, bytes as in the row layout. Padding is q = 0
// (int4) or byte 0 (fp8, int8). Scales: [NB][Gp][64] and ST [Gp][NB*64],
// ST[kg][n] = scale of row n, group kg (zero for padding rows and groups).
//
// A workgroup takes 64 rows x 128 bytes of the row layout (int4: 256 columns,
// four blocks; 8-bit: 128 columns, two) through LDS: 16-byte coalesced loads,
// 16-byte stores of whole blocks in both sections. The transpose works in
// registers on 8 x 8 nibbles (8 dwords, three rounds of exchanges, 4
// instructions a value) or 4 x 4 bytes. HBM-bound: the packed bytes read once
// and written twice. 12288 x 3072 int4 13 us; one thread per 16 output bytes
// gathering 32 single bytes from as many rows, and three more launches, took
// 58 us.
constexpr int BLK_ST = 33;  // LDS row stride in dwords (an odd number: no bank conflicts down a column)

LRQ_DEV void transpose8_nibbles(uint32_t (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {  // 16-bit halves
    const uint32_t a = v[i], b = v[i + 4];
    v[i] = __builtin_amdgcn_perm(b, a, 0x05040100u);
    v[i + 4] = __builtin_amdgcn_perm(b, a, 0x07060302u);
  }
#pragma unroll
  for (int h = 0; h < 8; h += 4)
#pragma unroll
    for (int i = h; i < h + 2; ++i) {  // bytes
      const uint32_t a = v[i], b = v[i + 2];
      v[i] = __builtin_amdgcn_perm(b, a, 0x06020400u);
      v[i + 2] = __builtin_amdgcn_perm(b, a, 0x07030501u);
    }
#pragma unroll
  for (int i = 0; i < 8; i += 2) {  // nibbles
    const uint32_t a = v[i], b = v[i + 1];
    v[i] = (a & 0x0f0f0f0fu) | ((b << 4) & 0xf0f0f0f0u);
    v[i + 1] = ((a >> 4) & 0x0f0f0f0fu) | (b & 0xf0f0f0f0u);
  }
}

LRQ_DEV void transpose4_bytes(uint32_t (&v)[4]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t a = v[i], b = v[i + 2];
    v[i] = __builtin_amdgcn_perm(b, a, 0x05040100u);
    v[i + 2] = __builtin_amdgcn_perm(b, a, 0x07060302u);
  }
#pragma unroll
  for (int i = 0; i < 4; i += 2) {
    const uint32_t a = v[i], b = v[i + 1];
    v[i] = __builtin_amdgcn_perm(b, a, 0x06020400u);
    v[i + 1] = __builtin_amdgcn_perm(b, a, 0x07030501u);
  }
}

template <bool I4>
__global__ void __launch_bounds__(256) k_block(const uint8_t* __restrict__ src, const float* __restrict__ ssrc, int64_t n,
                                               int64_t k, int g, int64_t NB, int64_t KB, int64_t KBX, uint8_t* __restrict__ dst,
                                               uint8_t* __restrict__ dstt, float* __restrict__ sdst,
                                               float* __restrict__ sdstt) {
  constexpr int NBK = I4 ? 4 : 2;          // blocks per workgroup
  constexpr int RB = I4 ? 32 : 64;         // bytes per block row
  constexpr uint32_t fill = I4 ? 0x88888888u : 0u;
  __shared__ uint32_t sr[64 * BLK_ST];                                      // rows [64][128 bytes]
  __shared__ __attribute__((aligned(16))) uint32_t st_[64 * NBK * RB / 4];  // transposed [64 NBK][RB bytes]
  const int tid = threadIdx.x;
  const int64_t nb = blockIdx.x / KBX, kb0 = blockIdx.x % KBX * NBK;
  const int64_t rowb = I4 ? k / 2 : k, b0 = kb0 * RB;  // the row layout's row bytes; this workgroup's first
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int id = tid + 256 * q, r = id >> 3, c = (id & 7) * 16;
    u32x4 v = {fill, fill, fill, fill};
    // (k is a multiple of 32, so 16 bytes are in or out together)
    if (nb * 64 + r < n && b0 + c < rowb) v = ld16(src + (nb * 64 + r) * rowb + b0 + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) sr[r * BLK_ST + (c >> 2) + e] = v[e];
  }
  __syncthreads();
  // row section: 16-byte chunk id of the workgroup's blocks
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int id = tid + 256 * q, blk = id / (4 * RB), in = id % (4 * RB), r = in / (RB / 16), c = in % (RB / 16);
    u32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = sr[r * BLK_ST + blk * (RB / 4) + c * 4 + e];
    if (kb0 + blk < KB) st16(dst + ((nb * KB + kb0 + blk) * 64 + r) * RB + c * 16, v);
  }
  if (I4) {
    // columns 8 i .. +8 of rows 8 j .. +8
    const int i = tid >> 3, j = tid & 7;
    uint32_t v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = sr[(8 * j + e) * BLK_ST + i];
    transpose8_nibbles(v);
#pragma unroll
    for (int e = 0; e < 8; ++e) st_[(8 * i + e) * (RB / 4) + j] = v[e] ^ 0x88888888u;  // q + 8 -> two's complement
  } else {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int id = tid + 256 * q, i = id >> 4, j = id & 15;
      uint32_t v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = sr[(4 * j + e) * BLK_ST + i];
      transpose4_bytes(v);
#pragma unroll
      for (int e = 0; e < 4; ++e) st_[(4 * i + e) * (RB / 4) + j] = v[e];
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int id = tid + 256 * q, blk = id / (4 * RB), in = id % (4 * RB);
    if (kb0 + blk < KB) st16(dstt + ((kb0 + blk) * NB + nb) * 64 * RB + in * 16, *reinterpret_cast<const u32x4*>(st_ + id * 4));
  }
  if (!sdst) return;
  // group scales of the workgroup's columns (a group wider than them: its
  // first workgroup), one row per thread
  const int64_t G = k / g, Gp = KB * 64 / g;
  const int64_t j0 = (kb0 * 64 + g - 1) / g, j1 = min(Gp, ((kb0 + NBK) * 64 + g - 1) / g);
  const int64_t row = nb * 64 + (tid & 63);
  for (int64_t j = j0 + (tid >> 6); j < j1; j += 4) {
    const float v = (row < n && j < G) ? ssrc[row * G + j] : 0.0f;
    sdst[(nb * Gp + j) * 64 + (tid & 63)] = v;
    sdstt[j * NB * 64 + row] = v;
  }
}

// ------------------------------------------------------------------ dequantize
// int4 -> f32 (bit-exact q*s) or bf16 operand; one thread per 8-value run.
template <bool BF16>
__global__ void __launch_bounds__(256) k_dequant_int4(const uint8_t* __restrict__ packed,
                                                      const float* __restrict__ scales, int64_t n,
                                                      int64_t k, int g, int blocked, void* __restrict__ out) {
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t runs = n * (k / 8);
  if (tid >= runs) return;
  const int64_t row = tid / (k / 8);
  const int64_t kk = (tid % (k / 8)) * 8;
  const int64_t KB = (k + 63) / 64;
  const int64_t Gp = KB * 64 / g;
  const int64_t doff = blocked ? blk_data_off(LRQ_FMT_INT4, row, kk, KB) : row * (k / 2) + kk / 2;
  const int64_t soff = blocked ? (((row >> 6) * Gp + kk / g) * 64 + (row & 63)) : row * (k / g) + kk / g;
  const uint32_t word = *reinterpret_cast<const uint32_t*>(packed + doff);
  const float s = scales[soff];
  if (BF16) {
    st16(reinterpret_cast<uint16_t*>(out) + row * k + kk, dequant8_int4_bf16(word, s));
  } else {
    float f[8];
    dequant8_int4_f32(word, s, f);
    float* o = reinterpret_cast<float*>(out) + row * k + kk;
    f32x4 a = {f[0], f[1], f[2], f[3]};
    f32x4 b = {f[4], f[5], f[6], f[7]};
    *reinterpret_cast<f32x4*>(o) = a;
    *reinterpret_cast<f32x4*>(o + 4) = b;
  }
}

// int8 -> f32 (bit-exact q*s) or bf16 operand; one thread per 8-value run.
template <bool BF16>
__global__ void __launch_bounds__(256) k_dequant_int8(const uint8_t* __restrict__ data,
                                                      const float* __restrict__ scales, int64_t n,
                                                      int64_t k, int g, int blocked, void* __restrict__ out) {
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t runs = n * (k / 8);
  if (tid >= runs) return;
  const int64_t row = tid / (k / 8);
  const int64_t kk = (tid % (k / 8)) * 8;
  const int64_t KB = (k + 63) / 64;
  const int64_t Gp = KB * 64 / g;
  const int64_t doff = blocked ? blk_data_off(LRQ_FMT_INT8, row, kk, KB) : row * k + kk;
  const int64_t soff = blocked ? (((row >> 6) * Gp + kk / g) * 64 + (row & 63)) : row * (k / g) + kk / g;
  const u32x2 word = *reinterpret_cast<const u32x2*>(data + doff);
  const float s = scales[soff];
  if (BF16) {
    st16(reinterpret_cast<uint16_t*>(out) + row * k + kk, dequant8_int8_bf16(word, s));
  } else {
    float f[8];
    dequant8_int8_f32(word, s, f);
    float* o = reinterpret_cast<float*>(out) + row * k + kk;
    *reinterpret_cast<f32x4*>(o) = (f32x4){f[0], f[1], f[2], f[3]};
    *reinterpret_cast<f32x4*>(o + 4) = (f32x4){f[4], f[5], f[6], f[7]};
  }
}

// fp8 -> f32 (LUT value * scale, one f32 rounding) or the unscaled bf16 operand.
template <bool BF16>
__global__ void __launch_bounds__(256) k_dequant_fp8(const uint8_t* __restrict__ bytes,
                                                     const float* __restrict__ scales, int64_t n,
                                                     int64_t k, int per_channel, int blocked,
                                                     void* __restrict__ out) {
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t quads = n * k / 4;
  if (tid >= quads) return;
  const int64_t row = (tid * 4) / k, kk = (tid * 4) % k;
  const int64_t doff = blocked ? blk_data_off(LRQ_FMT_FP8, row, kk, (k + 63) / 64) : tid * 4;
  const uint32_t word = *reinterpret_cast<const uint32_t*>(bytes + doff);
  if (BF16) {
    reinterpret_cast<u32x2*>(out)[tid] = fp8x4_to_bf16(word);
  } else {
    const float s = per_channel ? scales[row] : scales[0];
    f32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = fp8_e4m3fn_to_f32((word >> (8 * j)) & 0xffu) * s;
    reinterpret_cast<f32x4*>(out)[tid] = o;
  }
}

// ------------------------------------------------------------------ launchers
static inline unsigned blocks_for(int64_t items, int per_block) {
  return (unsigned)((items + per_block - 1) / per_block);
}

hipError_t launch_quantize_int4(hipStream_t st, const float* w, int64_t n, int64_t k, int g,
                                uint8_t* packed, float* scales) {
  const int64_t items = n * (k / 32);
  if (items == 0) return hipSuccess;
  hipLaunchKernelGGL((k_quantize<false, 7>), dim3(blocks_for(items, 256)), dim3(256), 0, st, w, nullptr, 0, n, k,
                     g, packed, scales);
  return hipGetLastError();
}

hipError_t launch_quantize_int8(hipStream_t st, const float* w, int64_t n, int64_t k, int g, int8_t* q,
                                float* scales) {
  const int64_t items = n * (k / 32);
  if (items == 0) return hipSuccess;
  hipLaunchKernelGGL((k_quantize<false, 127>), dim3(blocks_for(items, 256)), dim3(256), 0, st, w, nullptr, 0, n, k,
                     g, reinterpret_cast<uint8_t*>(q), scales);
  return hipGetLastError();
}

hipError_t launch_requantize_fp8_int4(hipStream_t st, const uint8_t* bytes, const float* scale, int per_channel,
                                      int64_t n, int64_t k, int g, uint8_t* packed, float* scales) {
  const int64_t items = n * (k / 32);
  if (items == 0) return hipSuccess;
  hipLaunchKernelGGL((k_quantize<true, 7>), dim3(blocks_for(items, 256)), dim3(256), 0, st, bytes, scale,
                     per_channel, n, k, g, packed, scales);
  return hipGetLastError();
}

hipError_t launch_quantize_fp8(hipStream_t st, const float* w, int64_t n, int64_t k,
                               int per_channel, uint8_t* bytes, float* scales, float* amax_ws) {
  if (n == 0 || k == 0) return hipSuccess;
  if (per_channel && k <= 16 * 1024) {
    const dim3 grid((unsigned)n);
    if (k <= 2 * 1024)
      hipLaunchKernelGGL(k_fp8_rows<2>, grid, dim3(256), 0, st, w, k, scales, bytes);
    else if (k <= 4 * 1024)
      hipLaunchKernelGGL(k_fp8_rows<4>, grid, dim3(256), 0, st, w, k, scales, bytes);
    else if (k <= 8 * 1024)
      hipLaunchKernelGGL(k_fp8_rows<8>, grid, dim3(256), 0, st, w, k, scales, bytes);
    else
      hipLaunchKernelGGL(k_fp8_rows<16>, grid, dim3(256), 0, st, w, k, scales, bytes);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_rowabsmax, dim3((unsigned)n), dim3(256), 0, st, w, k, amax_ws);
  hipLaunchKernelGGL(k_fp8_scales, dim3(per_channel ? blocks_for(n, 256) : 1), dim3(256), 0, st,
                     amax_ws, n, per_channel, scales);
  hipLaunchKernelGGL(k_fp8_encode, dim3(blocks_for(n * k / 4, 256)), dim3(256), 0, st, w, n, k,
                     per_channel, scales, bytes);
  return hipGetLastError();
}

hipError_t launch_dequant(hipStream_t st, const lrq_weight* w, void* out, bool bf16) {
  const int64_t n = w->n, k = w->k;
  if (n == 0 || k == 0) return hipSuccess;
  const uint8_t* d = reinterpret_cast<const uint8_t*>(w->data);
  const int blocked = w->layout == LRQ_LAYOUT_BLOCKED;
  if (w->format == LRQ_FMT_INT4) {
    const int64_t runs = n * (k / 8);
    if (bf16)
      hipLaunchKernelGGL(k_dequant_int4<true>, dim3(blocks_for(runs, 256)), dim3(256), 0, st, d,
                         w->scales, n, k, w->group, blocked, out);
    else
      hipLaunchKernelGGL(k_dequant_int4<false>, dim3(blocks_for(runs, 256)), dim3(256), 0, st, d,
                         w->scales, n, k, w->group, blocked, out);
  } else if (w->format == LRQ_FMT_INT8) {
    const int64_t runs = n * (k / 8);
    if (bf16)
      hipLaunchKernelGGL(k_dequant_int8<true>, dim3(blocks_for(runs, 256)), dim3(256), 0, st, d,
                         w->scales, n, k, w->group, blocked, out);
    else
      hipLaunchKernelGGL(k_dequant_int8<false>, dim3(blocks_for(runs, 256)), dim3(256), 0, st, d,
                         w->scales, n, k, w->group, blocked, out);
  } else {
    const int64_t quads = n * k / 4;
    if (bf16)
      hipLaunchKernelGGL(k_dequant_fp8<true>, dim3(blocks_for(quads, 256)), dim3(256), 0, st, d,
                         w->scales, n, k, w->per_channel, blocked, out);
    else
      hipLaunchKernelGGL(k_dequant_fp8<false>, dim3(blocks_for(quads, 256)), dim3(256), 0, st, d,
                         w->scales, n, k, w->per_channel, blocked, out);
  }
  return hipGetLastError();
}

void blocked_sections(int fmt, int64_t n, int64_t k, int64_t group, int64_t* data_bytes, int64_t* scale_count) {
  const int64_t NB = (n + 63) / 64, KB = (k + 63) / 64;
  *data_bytes = NB * KB * 64 * (fmt == LRQ_FMT_INT4 ? 32 : 64);
  *scale_count = (fmt != LRQ_FMT_FP8) ? NB * (KB * 64 / group) * 64 : 0;
}

int64_t blocked_t_scale_count(int fmt, int64_t n, int64_t k, int64_t group) {
  if (fmt == LRQ_FMT_FP8) return 0;
  const int64_t NB = (n + 63) / 64, KB = (k + 63) / 64;
  return (KB * 64 + group - 1) / group * NB * 64;
}

void blocked_sizes(int fmt, int64_t n, int64_t k, int64_t group, int64_t* data_bytes, int64_t* scale_count) {
  int64_t db = 0, sc = 0;
  blocked_sections(fmt, n, k, group, &db, &sc);
  *data_bytes = 2 * db;
  *scale_count = sc + blocked_t_scale_count(fmt, n, k, group);
}

hipError_t launch_block(hipStream_t st, const lrq_weight* w, uint8_t* data, float* scales) {
  const int64_t n = w->n, k = w->k;
  const int64_t NB = (n + 63) / 64, KB = (k + 63) / 64;
  int64_t db = 0, sc = 0;
  blocked_sections(w->format, n, k, w->group, &db, &sc);
  if (db == 0) return hipSuccess;
  const uint8_t* src = reinterpret_cast<const uint8_t*>(w->data);
  const bool gs = w->format != LRQ_FMT_FP8 && sc > 0;
  const int nbk = w->format == LRQ_FMT_INT4 ? 4 : 2;
  const int64_t kbx = (KB + nbk - 1) / nbk;
  const dim3 grid((unsigned)(kbx * NB));
  float* const s0 = gs ? scales : nullptr;
  float* const s1 = gs ? scales + sc : nullptr;
  if (w->format == LRQ_FMT_INT4)
    hipLaunchKernelGGL(k_block<true>, grid, dim3(256), 0, st, src, w->scales, n, k, w->group, NB, KB, kbx, data,
                       data + db, s0, s1);
  else
    hipLaunchKernelGGL(k_block<false>, grid, dim3(256), 0, st, src, w->scales, n, k, w->group, NB, KB, kbx, data,
                       data + db, s0, s1);
  return hipGetLastError();
}
