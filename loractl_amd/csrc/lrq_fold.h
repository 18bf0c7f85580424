// The mid-size passes' in-launch side products, shared by the kernels that
// run them (lrq_gemm_mid.hip, lrq_gemm_w8.hip): the token-side LoRA factor
// (t forward, u backward) formed by workgroups ahead of the tiles, and the
// weight gradients (dB, dA) by workgroups after them. Each body is the work
// of 256 threads; a 512-thread workgroup runs two side by side, one per half
// (threads 0..255 and 256..511), each with its own LDS. A half whose body
// ends early simply ends its wavefronts: a barrier counts the wavefronts
// that are still running.
#pragma once

#include "lrq_common.h"
#include "lrq_kernels.h"
#include "lrq_tn.h"

namespace {

// device-scope accesses of the fold's cross-workgroup data (written through
// and read past the per-XCD L2s), as in lrq_skinny.hip
constexpr int MXSCOPE = __HIP_MEMORY_SCOPE_AGENT;
LRQ_DEV uint32_t madd_dev(uint32_t* c) { return __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, MXSCOPE); }
LRQ_DEV void mzero_dev(uint32_t* c) { __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, MXSCOPE); }
LRQ_DEV uint32_t mload_dev(const uint32_t* c) { return __hip_atomic_load(c, __ATOMIC_RELAXED, MXSCOPE); }
LRQ_DEV u32x4 mbload16_dev(rsrc_t r, uint32_t off) { return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 16); }
LRQ_DEV void mstore16_dev(rsrc_t r, uint32_t off, const u32x4& v) { __builtin_amdgcn_raw_buffer_store_b128(v, r, off, 0, 16); }
LRQ_DEV void mstore8_dev(rsrc_t r, uint32_t off, const u32x2& v) { __builtin_amdgcn_raw_buffer_store_b64(v, r, off, 0, 16); }
LRQ_DEV uint32_t mstamp(uint32_t ep) { return ep + 1 == 0 ? 1u : ep + 1; }
constexpr uint32_t MID_MAX_POLLS = 1u << 22;  // about 0.2 s of s_sleep 2
// the fold's counters: per 64-token group the slices' arrivals at [0, G)
// and the ready flags at [G, 2 G)

// FOLD: workgroup fw of the factor workgroups: 64-token group fw / fold_slices,
// depth slice fw % fold_slices, RT rank tiles of 16 (rp = 16 RT). Wavefront
// w takes tokens 16 w .. + 16 of the group; each of its lanes loads the
// group's token row 16 w + (l & 15) at depths 32 ss + 8 (l >> 4) .. + 8 of
// the slice (every load of the slice at once) and the factor fragments of
// the same depths for ranks 16 rt + (l & 15): forward A's rows staged
// transposed in LDS (rank tile rt's aT [16][FKT + 8] in lds[rt]), backward
// B's rows read directly. `want` is the launch's stamp.
template <bool BWD, int RT>
LRQ_DEV void mid_fold_slice(const GemmArgs& a, int fw, uint16_t* lds0, uint16_t* lds1, uint32_t want) {
  constexpr int FKT = MID_FOLD_KT, NSS = FKT / 32, AST = FKT + 8, RP = 16 * RT;
  const int tid = threadIdx.x & 255, lane = tid & 63;
  const int half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane & 15, kq = lane >> 4;
  const int fs = a.fold_slices, g = fw / fs, sl = fw % fs;
  const int64_t M = a.m, D = a.l, Mp = (M + 63) / 64 * 64;
  const int r = a.r;
  const int64_t k0 = (int64_t)sl * FKT, k1 = k0 + FKT < D ? k0 + FKT : D;
  const int64_t tok = (int64_t)g * 64 + 16 * w + c16;
  const rsrc_t rx = make_rsrc(a.act, clamp_bytes(M * D * 2));
  const rsrc_t rf = make_rsrc(a.lact, clamp_bytes(D * r * 2));
  uint16_t* const lds[2] = {lds0, lds1};
  u32x4 xf[NSS], bf[RT][NSS];
#pragma unroll
  for (int ss = 0; ss < NSS; ++ss) {
    const int64_t k = k0 + 32 * ss + 8 * kq;
    xf[ss] = bload16(rx, opaque_u32(tok < M && k < k1 ? (uint32_t)((tok * D + k) * 2) : LRQ_OOB));
    if (BWD) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        const int j = 16 * rt + c16;
        bf[rt][ss] = bload16(rf, opaque_u32(j < r && k < k1 ? (uint32_t)(((int64_t)j * D + k) * 2) : LRQ_OOB));
      }
    }
  }
  if (!BWD) {
    // A [D][r] rows of the slice, 8 ranks per 16-byte run: pair i = tid +
    // 256 q is depth i / JB, ranks 8 (i % JB) ..; zeros past the rank or depth
    constexpr int JB = RP / 8, AQ = JB * FKT / 256;
    u32x4 av[AQ];
#pragma unroll
    for (int qq = 0; qq < AQ; ++qq) {
      const int i = tid + 256 * qq, dd = i / JB, j0 = 8 * (i % JB);
      av[qq] = bload16(rf, opaque_u32(k0 + dd < k1 && j0 < r ? (uint32_t)(((k0 + dd) * r + j0) * 2) : LRQ_OOB));
    }
#pragma unroll
    for (int qq = 0; qq < AQ; ++qq) {
      const int i = tid + 256 * qq, dd = i / JB, j0 = 8 * (i % JB);
      uint16_t* t = lds[j0 >> 4];
#pragma unroll
      for (int e = 0; e < 8; ++e) t[((j0 & 15) + e) * AST + dd] = (uint16_t)(av[qq][e >> 1] >> (16 * (e & 1)));
    }
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int ss = 0; ss < NSS; ++ss)
        bf[rt][ss] = *reinterpret_cast<const u32x4*>(lds[rt] + c16 * AST + 32 * ss + 8 * kq);
  }
  // C element v of lane (c16, kq) in rank tile rt: rank 16 rt + 4 kq + v,
  // token 16 w + c16
  f32x4 acc[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    acc[rt] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    // an opaque zero of its own in vector registers, and the last step's
    // result pinned in place (in accumulator registers the compiler wrote it
    // to a tuple that overlapped its SrcC's)
    asm volatile("" : "+v"(acc[rt]));
#pragma unroll
    for (int ss = 0; ss < NSS; ++ss) acc[rt] = mfma16(as_bf16x8(bf[rt][ss]), as_bf16x8(xf[ss]), acc[rt]);
    asm volatile("" : "+v"(acc[rt]));
  }
  const rsrc_t rp = make_rsrc(a.fpart, clamp_bytes((int64_t)fs * Mp * RP * 4));
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
    mstore16_dev(rp, opaque_u32((uint32_t)((((int64_t)sl * Mp + tok) * RP + 16 * rt + 4 * kq) * 4)),
                 __builtin_bit_cast(u32x4, acc[rt]));
  // counted once the partial is acknowledged; the last slice of the group
  // sums the slices in order, stores the factor and publishes the flag
  __builtin_amdgcn_s_waitcnt(0);
  __shared__ int last[2];
  __syncthreads();
  const int64_t G = (M + 63) / 64;
  if (tid == 0) {
    last[half] = madd_dev(a.fcnt + g) + 1 == (uint32_t)fs;
    if (last[half]) mzero_dev(a.fcnt + g);
  }
  __syncthreads();
  if (last[half]) {
    // thread: token g 64 + tid / 4, ranks 16 rt + 4 (tid % 4) ..
    const int64_t tk = (int64_t)g * 64 + (tid >> 2);
    const rsrc_t ro = make_rsrc(a.fout, clamp_bytes(M * a.fout_ld * 2));
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int rq = 16 * rt + 4 * (tid & 3);
      f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
      for (int s0 = 0; s0 < fs; s0 += 8) {
        u32x4 pv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          pv[u] = mbload16_dev(rp, opaque_u32(s0 + u < fs ? (uint32_t)((((int64_t)(s0 + u) * Mp + tk) * RP + rq) * 4) : LRQ_OOB));
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += __builtin_bit_cast(f32x4, pv[u]);
      }
      if (a.fout && tk < M && rq < a.fout_ld) {
        const u32x2 o = {pack_bf16x2(a.fscale * sum[0], a.fscale * sum[1]), pack_bf16x2(a.fscale * sum[2], a.fscale * sum[3])};
        mstore8_dev(ro, opaque_u32((uint32_t)((tk * a.fout_ld + rq) * 2)), o);
      }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) __hip_atomic_store(a.fcnt + G + g, want, __ATOMIC_RELAXED, MXSCOPE);
  }
}

// FOLD: a reader of the ready flags is done with them (a tile after its
// LoRA step, a dA block after its wait). The last of the launch's `readers`
// clears the flags and advances the epoch. Every thread of a reader (NT
// threads) calls it.
template <int NT>
LRQ_DEV void mid_flags_done(const GemmArgs& a, int readers) {
  __shared__ int fin[2];
  const int tid = threadIdx.x % NT, half = __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
  __syncthreads();
  if (tid == 0) fin[half] = madd_dev(a.fcnt + SK_DCNT) + 1 == (uint32_t)readers;
  __syncthreads();
  if (fin[half]) {
    const int64_t G = (a.m + 63) / 64;
    for (int64_t i = tid; i < G; i += NT) mzero_dev(a.fcnt + G + i);
    if (tid == 0) {
      mzero_dev(a.fcnt + SK_DCNT);
      madd_dev(a.fcnt + SK_EPOCH);
    }
  }
}

// FOLD backward: weight-gradient block tb of the launch's tn jobs (after the
// tiles). A dA block first waits (bounded, as the tiles do) for the ready
// flags of the 64-token groups of its token slice, then reads u at device
// scope; a wait that runs out flags the failure and makes its sums NaN.
// The factor slice goes to sq, the combine buffer to sr (LDSB bytes each; one
// buffer may serve as both). VACC: sums in vector registers (the 128-token
// tiles'): in accumulator registers their kernels had 128 vector registers
// left and spilled 33 to 36 of them in a rank-32 block (backward at 384
// tokens, 3072 -> 12288, rank 32: 72 -> 58 us without the spills).
template <int LDSB, bool VACC>
LRQ_DEV void mid_tn(const GemmArgs& a, int tb, uint32_t want, int readers, uint16_t* sq, uint16_t* sr) {
  const bool second = tb >= a.tj[0].blocks;
  const int ji = second ? 1 : 0;
  const TnArgs& j = a.tj[ji];
  const int bid = tb - (second ? a.tj[0].blocks : 0);
  float* const red = reinterpret_cast<float*>(sr);
  if (ji != a.tn_da) {
    if (a.rp == 32)
      tn_block<2, LDSB, LDSB, false, VACC>(j, bid, sq, red, false);
    else
      tn_block<1, LDSB, LDSB, false, VACC>(j, bid, sq, red, false);
    return;
  }
  __shared__ int bad[2];
  const int tid = threadIdx.x & 255, half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  if (tid < 64) {
    const int lane = tid;
    const int64_t G = (a.m + 63) / 64;
    const int64_t m_lo = (int64_t)(bid / j.tiles) * j.m_per;
    const int64_t m_hi = min(j.M, m_lo + j.m_per);
    const int64_t gi = m_lo / 64 + lane;
    const bool mine = gi < (m_hi + 63) / 64 && gi < G;
    uint32_t polls = 0;
    const uint32_t cap = a.fold < 0 ? 16u : MID_MAX_POLLS;  // the test hook: 16 polls
    bool ok = !mine || mload_dev(a.fcnt + G + gi) == want;
    while (!__all(ok) && polls < cap) {
      __builtin_amdgcn_s_sleep(2);
      ++polls;
      ok = !mine || mload_dev(a.fcnt + G + gi) == want;
    }
    if (lane == 0) {
      bad[half] = __all(ok) ? 0 : 1;
      if (!__all(ok)) __hip_atomic_store(a.fcnt + SK_FAIL, 1u, __ATOMIC_RELAXED, MXSCOPE);
    }
  }
  __syncthreads();
  const bool poison = bad[half] != 0;
  mid_flags_done<256>(a, readers);
  if (a.rp == 32)
    tn_block<2, LDSB, LDSB, true, VACC>(j, bid, sq, red, poison);
  else
    tn_block<1, LDSB, LDSB, true, VACC>(j, bid, sq, red, poison);
}

}  // namespace
