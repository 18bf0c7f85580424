// The fused GEMMs of the quantized LoRA linear on 128-row x 128-token tiles,
// for the token counts that leave the 256 x 256 tiles of lrq_gemm.hip too few
// to fill the CUs (the products and operands of lrq_gemm_mid.hip):
//
//   forward   y[m, n]  = x[m, k]  . bf16(dq(w))[n, k]^T (+bias) + t[m, :] . B[:, n]
//   backward  dx[m, k] = dy[m, n] . bf16(dq(w))[n, k]            + u[m, :] . A[k, :]^T
//
// (src/quant.rs:175-176 and :229-233; the LoRA terms of src/lora.rs:199-203.)
//
// "Rows" are the output columns (n forward, k backward), "depth" the
// reduction index. One workgroup of eight wavefronts (two per SIMD) has a CU
// and a tile. The wavefronts split the tile's rows in RW halves of 64 and the
// depth in KG groups: wavefront (rw, kg) forms rows 64 rw .. +64 for all 128
// tokens over the 64-deep blocks kg, kg + KG, .. of the tile's depth:
//   - weight (A role): as the large tiles. A lane loads the packed bytes of
//     its rows l & 31 and 32 + (l & 31), depth 32 (l >> 5) .. +32 of the
//     block, and dequantizes them to the bf16 operand of the matrix cores
//     (sub-step kk takes depth 32 (l >> 5) + 8 kk .. +8). No weight element
//     is dequantized twice in a tile;
//   - activations (B role): each depth group's [128 tokens][64] block goes
//     global -> LDS by buffer loads with an LDS destination, each of the
//     group's wavefronts moving its share; 16-byte chunk c of row r at chunk
//     c ^ ((r >> 1) & 7). Token tile j (32 tokens) of the wavefront is token
//     tile j ^ kg of the tile, so that after the sums below every wavefront
//     owns its local tile 0 and no register index depends on the wavefront;
//   - a stage is KG blocks (256 deep), in two LDS buffers: the next stage's
//     copies and packed weights are issued when the stage begins and have
//     landed when it ends; one barrier per stage;
//   - the depth groups' accumulators meet in LDS: in each of log2(KG) rounds
//     a wavefront hands half of its token tiles to the wavefront kg ^ 1 (then
//     kg ^ 2) of the same rows and adds the half it is handed, in a fixed
//     order; every wavefront ends with 64 rows x 128 / KG tokens;
//   - depth ranges, the fold (t, u, dA and dB in the same launch) and its
//     bounded waits, edges and tile order: as lrq_gemm_mid.hip describes.
//
// Why this split: a wavefront with 64 rows and 128 tokens feeds 8 matrix-core
// steps of 32 x 32 x 16 from 4 LDS fragments and 2 dequantized ones, so per
// 64-deep block of the tile the LDS reads take 256 of the matrix cores' 512
// cycles and the dequantization about 370 (it is spread over all eight
// wavefronts by the depth groups instead of repeated by them).
#include <algorithm>

#include "lrq_common.h"
#include "lrq_fold.h"
#include "lrq_kernels.h"

namespace {

constexpr int WD = 64;         // depth of a block
constexpr int WT = W8_TOKENS;  // tokens per tile
constexpr int WNT = 512;       // threads: eight wavefronts
constexpr int SLICE = WT * WD; // bf16 of one depth group's block in LDS (16 KiB)

LRQ_DEV int wswz(int r) { return (r >> 1) & 7; }

template <bool BWD, int FMT, int RW, bool FOLD>
__global__ void __launch_bounds__(WNT, 2) k_w8(GemmArgs a, int tiles_m, int tiles_e, int group_m) {
  constexpr bool I4 = FMT == LRQ_FMT_INT4;
  constexpr bool I8 = FMT == LRQ_FMT_INT8;
  constexpr bool GS = I4 || I8;          // group scales (int4, int8) or channel scales (fp8)
  constexpr int KG = 8 / RW;             // depth groups
  constexpr int R = 64 * RW;             // rows per tile
  constexpr int WV = I4 ? 1 : 2;         // 16-byte packed loads per row tile and block
  constexpr int NSC = GS ? 2 : 1;        // backward scale registers: per row tile, or shared (fp8)
  constexpr int XL = WT / RW / 8;        // activation copies per wavefront and stage
  constexpr uint32_t blkb = I4 ? 2048u : 4096u;
  constexpr uint32_t rowb = I4 ? 32u : 64u;
  constexpr int FST = 32 + 8;            // LDS row stride of the factor rows
  static_assert(RW == 2 || RW == 4, "the sums below are written for four or two depth groups");
  __shared__ __attribute__((aligned(16))) uint16_t sx0[KG * SLICE];
  __shared__ __attribute__((aligned(16))) uint16_t sx1[KG * SLICE];
  __shared__ __attribute__((aligned(16))) uint16_t sF[FOLD ? R * FST : 8];
  // weight-gradient blocks: W8_TN_LDS per half (the stage buffers hold only half of it with 256 rows)
  __shared__ __attribute__((aligned(16))) uint16_t sT[FOLD && BWD && RW == 4 ? W8_TN_LDS : 8];

  const int ntiles = tiles_m * tiles_e;
  const int S = a.msplit > 1 ? a.msplit : 1;
  const int nunits = ntiles * S;
  uint32_t want = 0;
  if (FOLD) {
    const uint32_t stamp = mstamp(mload_dev(a.fcnt + SK_EPOCH));
    const int half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    if ((int)blockIdx.x < a.fold_wgs) {
      // two factor slices at a time, one per half
      uint16_t* const l0 = sx0 + half * (KG * SLICE / 2);
      uint16_t* const l1 = sx1 + half * (KG * SLICE / 2);
      const int nfs = a.fold_slices * (int)((a.m + 63) / 64);
      for (int fw = 2 * (int)blockIdx.x + half; fw < nfs; fw += 2 * a.fold_wgs) {
        if (a.rp == 32)
          mid_fold_slice<BWD, 2>(a, fw, l0, l1, stamp);
        else
          mid_fold_slice<BWD, 1>(a, fw, l0, l1, stamp);
      }
      return;
    }
    want = stamp + (a.fold < 0 ? 0x40000000u : 0u);
    if constexpr (BWD) {
      if ((int)blockIdx.x >= a.fold_wgs + nunits) {
        static_assert((RW == 4 || W8_TN_LDS <= KG * SLICE * 2) && 16 * (MID_FOLD_KT + 8) <= KG * SLICE / 2, "LDS of a half");
        uint16_t* const lt = RW == 4 ? sT + half * (W8_TN_LDS / 2) : (half ? sx1 : sx0);
        const int nda = a.tn_da >= 0 ? a.tj[a.tn_da].blocks : 0;
        // two blocks of one job per workgroup
        const int wg = (int)blockIdx.x - a.fold_wgs - nunits, w0 = (a.tj[0].blocks + 1) / 2;
        const int tb = wg < w0 ? 2 * wg + half : a.tj[0].blocks + 2 * (wg - w0) + half;
        if (tb < (wg < w0 ? a.tj[0].blocks : a.tn_blocks))
          mid_tn<W8_TN_LDS, true>(a, tb, want, ntiles + nda, lt, lt);
        return;
      }
    }
  }
  const int vb = FOLD ? (int)blockIdx.x - a.fold_wgs : (int)blockIdx.x;
  const int lu = xcd_remap(vb, nunits);
  const int lt = lu / S, sp = lu % S;
  const int per = group_m * tiles_e;
  const int grp = lt / per, within = lt % per;
  const int gm = min(group_m, tiles_m - grp * group_m);
  const int tm = grp * group_m + within % gm, te = within / gm;
  const int64_t M = a.m, D = a.l, E = a.e;
  const int64_t m0 = (int64_t)tm * WT, e0 = (int64_t)te * R;

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rw = w % RW, kg = w / RW;
  const int g = lane >> 5, l32 = lane & 31;
  const int64_t KB = (D + 63) / 64;
  // stages of KG blocks: the whole depth, or range sp's a.mspl stages from
  // stage s0 (the last range to the end); blocks past the depth read zeros
  const int nst = (int)((KB + KG - 1) / KG);
  const int s0 = S > 1 ? sp * a.mspl : 0;
  const int nsp = (S > 1 && sp < S - 1) ? a.mspl : nst - s0;

  // ---- weight: the block row of this wavefront's 64 rows (none past E)
  const int64_t er = e0 + 64 * rw;
  const bool rok = er < E;
  const int64_t rb = rok ? er / 64 : 0;
  const rsrc_t rwd = make_rsrc(a.wdata + rb * KB * blkb, rok ? clamp_bytes(KB * blkb) : 0u);
  const uint32_t woff = (uint32_t)l32 * rowb + (uint32_t)g * (I4 ? 16u : 32u);
  // forward int4 / int8: group scales [NB][Gp][64], this block row's slab.
  // Backward int4 / int8: ST [KGt][64 KB], one table row per 32-row tile,
  // lane l of a 16-lane row holding the scale of depth 32 g + 16 p + l % 16;
  // fp8: the channel scale of each depth, or one scalar
  const uint32_t Gp = (uint32_t)((KB * 64) >> a.gshift);
  const bool pc = !GS && a.per_channel;
  const int64_t NP = KB * 64;
  rsrc_t rs0, rs1;
  if (!BWD) {
    rs0 = make_rsrc(a.wscale + (GS ? rb * Gp * 64 : 0), (GS && rok) ? clamp_bytes((int64_t)Gp * 64 * 4) : 0u);
    rs1 = rs0;
  } else if (GS) {
    rs0 = make_rsrc(a.wscale + (rok ? (er >> a.gshift) * NP : 0), rok ? clamp_bytes(NP * 4) : 0u);
    rs1 = make_rsrc(a.wscale + (rok ? ((er + 32) >> a.gshift) * NP : 0), rok ? clamp_bytes(NP * 4) : 0u);
  } else {
    rs0 = make_rsrc(a.wscale, pc ? clamp_bytes(D * 4) : 0u);
    rs1 = rs0;
  }
  const float s0add = (BWD && !GS && !pc) ? a.wscale[0] : 0.0f;
  const uint32_t soff = BWD ? (uint32_t)(32 * g + (lane & 15)) * 4u : (uint32_t)l32 * 4u;

  u32x4 wp[2][2 * WV];   // packed bytes per register set, row tile
  float wsc[2][2];       // forward group scales
  float bsc[2][NSC][2];  // backward per-depth scales, two halves of a block
  auto load_w = [&](int set, int st) {
    const uint32_t kt = (uint32_t)((st + s0) * KG + kg);
    const uint32_t kb = opaque_u32(woff + kt * blkb);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int h = 0; h < WV; ++h) wp[set][i * WV + h] = bload16(rwd, kb + (uint32_t)i * 32u * rowb + 16u * h);
    if (!BWD && GS) {
      const uint32_t j = (kt * 64u + (uint32_t)g * 32u) >> a.gshift;
      const uint32_t so = opaque_u32(j * 256u + soff);
#pragma unroll
      for (int i = 0; i < 2; ++i) wsc[set][i] = bloadf(rs0, so + (uint32_t)i * 128u);
    }
    if (BWD) {
      const uint32_t sb = opaque_u32(kt * 256u + soff);
      bsc[set][0][0] = bloadf(rs0, sb);
      bsc[set][0][1] = bloadf(rs0, sb + 64u);
      if (GS) {
        bsc[set][NSC - 1][0] = bloadf(rs1, sb);
        bsc[set][NSC - 1][1] = bloadf(rs1, sb + 64u);
      }
    }
  };
  // A-role fragment of row tile i, sub-step kk, from register set `set`
  auto wfrag = [&](int set, int i, int kk) -> bf16x8 {
    if (!BWD) {
      if (I4) return as_bf16x8(dequant8_int4_bf16(wp[set][i][kk], wsc[set][i], a.nib));
      const u32x4 v = wp[set][i * WV + (kk >> 1)];
      if (I8) return as_bf16x8(dequant8_int8_bf16((u32x2){v[2 * (kk & 1)], v[2 * (kk & 1) + 1]}, wsc[set][i]));
      const u32x2 lo = fp8x4_to_bf16(v[2 * (kk & 1)]), hi = fp8x4_to_bf16(v[2 * (kk & 1) + 1]);
      return as_bf16x8((u32x4){lo[0], lo[1], hi[0], hi[1]});
    }
    float f[8];
    float sc = bsc[set][GS ? i : 0][kk >> 1];
    if (I4) {
      int4x8_to_f32_div16(wp[set][i][kk], f);  // q / 16, times 16 x the scale
      sc *= 16.0f;
    } else {
      const u32x4 v = wp[set][i * WV + (kk >> 1)];
      if (I8) {
        int8x4_to_f32(v[2 * (kk & 1)], f);
        int8x4_to_f32(v[2 * (kk & 1) + 1], f + 4);
      } else {
        fp8x4_to_f32(v[2 * (kk & 1)], f);
        fp8x4_to_f32(v[2 * (kk & 1) + 1], f + 4);
        sc += s0add;
      }
    }
    mul_row_bcast8(f, sc, kk & 1);
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = pack_bf16x2(f[2 * q], f[2 * q + 1]);
    return as_bf16x8(o);
  };

  // ---- activations: this wavefront copies LDS rows 64 rw .. +64 of its
  // depth group's block, 8 rows per copy; LDS row r holds token
  // 32 ((r >> 5) ^ kg) + (r & 31). Lane l of copy c lands at row 64 rw + 8c +
  // l/8, chunk l%8, fetching logical chunk (l%8) ^ wswz(row); the row's 8-row
  // group's parity decides the pattern. A chunk at or past the depth reads
  // zeros.
  const rsrc_t rx = make_rsrc(a.act + m0 * D, clamp_bytes(min(M - m0, (int64_t)WT) * D * 2));
  const int lc0 = (lane & 7) ^ ((lane >> 4) & 7), lc1 = (lane & 7) ^ (((lane >> 4) + 4) & 7);
  const uint32_t xo0 = (uint32_t)(((lane >> 3) * D + lc0 * 8) * 2);
  const uint32_t xo1 = (uint32_t)(((lane >> 3) * D + lc1 * 8) * 2);
  const int lim0 = (int)D - 8 * lc0, lim1 = (int)D - 8 * lc1;
  const int pr0 = (WT / RW) * rw;
  auto dma = [&](uint16_t* buf, int st, int clo, int chi) {
    const int k0 = ((st + s0) * KG + kg) * WD;
    const uint32_t o0 = opaque_u32(k0 < lim0 ? xo0 + (uint32_t)(k0 * 2) : LRQ_OOB);
    const uint32_t o1 = opaque_u32(k0 < lim1 ? xo1 + (uint32_t)(k0 * 2) : LRQ_OOB);
    __attribute__((address_space(3))) char* base =
        (__attribute__((address_space(3))) char*)(lds_void*)(buf + kg * SLICE + pr0 * WD);
#pragma unroll
    for (int c = clo; c < chi; ++c) {
      const int pr = pr0 + 8 * c;
      const uint32_t tok = (uint32_t)(32 * ((pr >> 5) ^ kg) + (pr & 31));
      // (past-the-depth offsets stay past the resource: it is under 2^31 bytes here)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void*)(base + c * 8 * WD * 2), 16,
                                               ((c & 1) ? o1 : o0) + tok * (uint32_t)(D * 2), 0, 0, 0);
    }
  };
  // B-role fragment of local token tile j, sub-step kk: row 32 j + l32,
  // logical chunk 4 g + kk
  uint32_t xk[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
    xk[kk] = opaque_u32((uint32_t)(kg * SLICE * 2 + l32 * WD * 2 + (((4 * g + kk) ^ wswz(l32)) * 16)));
  auto xfrag = [&](const uint16_t* buf, int j, int kk) -> bf16x8 {
    return as_bf16x8(ld16(reinterpret_cast<const char*>(buf) + xk[kk] + (uint32_t)(j * 32 * WD * 2)));
  };

  f32x16 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  // FOLD: the weight-side factor rows of the tile to LDS [R][FST], ranks up
  // to a.rp (zero past the rank and past E): forward B [r][E] transposed
  // (divided by an fp8 weight scale, which the epilogue multiplies by),
  // backward A [E][r] as stored. Per pass of 128 rows a thread takes a
  // 16-byte run of B's rank row tid / 16 (8 rows), or 8 ranks of A's row
  // tid / 4. In LDS before the first stage's barrier; read in the epilogue.
  if (FOLD) {
    const int fr = a.r;
#pragma unroll
    for (int q = 0; q < R / 128; ++q) {
      if (!BWD) {
        const int j = tid >> 4, r0 = 128 * q + (tid & 15) * 8;
        const rsrc_t rbf = make_rsrc(a.lw, clamp_bytes((int64_t)fr * E * 2));
        u32x4 v = bload16(rbf, opaque_u32(j < fr && e0 + r0 < E ? (uint32_t)((j * E + e0 + r0) * 2) : LRQ_OOB));
        if (!GS) {
#pragma unroll
          for (int h = 0; h < 4; ++h) {
            const int64_t n = e0 + r0 + 2 * h;
            const float d0 = a.per_channel ? (n < E ? a.wscale[n] : 1.0f) : a.wscale[0];
            const float d1 = a.per_channel ? (n + 1 < E ? a.wscale[n + 1] : 1.0f) : a.wscale[0];
            v[h] = (uint32_t)f32_to_bf16_bits(bf16_lo(v[h]) / d0) | ((uint32_t)f32_to_bf16_bits(bf16_hi(v[h]) / d1) << 16);
          }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) sF[(r0 + e) * FST + j] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
      } else {
        const int row = 128 * q + (tid >> 2), j0 = (tid & 3) * 8;
        const rsrc_t ra = make_rsrc(a.lw, clamp_bytes(E * fr * 2));
        st16(sF + row * FST + j0,
             bload16(ra, opaque_u32(j0 < fr && e0 + row < E ? (uint32_t)(((e0 + row) * fr + j0) * 2) : LRQ_OOB)));
      }
    }
  }

  bf16x8 fa[2][2], fb[2][4];
  // Stage st on buffer and register set b (b = st % 2, static). On entry
  // fa[0] and fb[0] hold sub-step 0's fragments.
  auto stage = [&](const int b, const int st) {
    uint16_t* const cur = b ? sx1 : sx0;
    uint16_t* const nxt = b ? sx0 : sx1;
    // every wavefront is done with the other buffer (the barrier before)
    load_w(b ^ 1, st + 1);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int c = kk & 1;
      if (kk < 2) dma(nxt, st + 1, kk * XL / 2, (kk + 1) * XL / 2);
      if (kk < 3) {
#pragma unroll
        for (int j = 0; j < 4; ++j) fb[c ^ 1][j] = xfrag(cur, j, kk + 1);
#pragma unroll
        for (int i = 0; i < 2; ++i) fa[c ^ 1][i] = wfrag(b, i, kk + 1);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mfma32(fa[c][i], fb[c][j], acc[i][j]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) fa[0][i] = wfrag(b ^ 1, i, 0);
    // the next stage's copies have landed (said here: the compiler does not
    // carry them over the loop's back edge), and this one's reads are done
    __builtin_amdgcn_s_waitcnt(0xf70);  // vmcnt(0)
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) fb[0][j] = xfrag(nxt, j, 0);
  };
  load_w(0, 0);
  dma(sx0, 0, 0, XL);
#pragma unroll
  for (int i = 0; i < 2; ++i) fa[0][i] = wfrag(0, i, 0);
  __builtin_amdgcn_s_waitcnt(0xf70);  // vmcnt(0)
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 4; ++j) fb[0][j] = xfrag(sx0, j, 0);
  int st = 0;
  for (; st + 1 < nsp; st += 2) {
    stage(0, st);
    stage(1, st + 1);
  }
  if (st < nsp) stage(0, st);

  // ---- the depth groups' sums. Every wavefront is past its last fragment
  // reads and copies (the last stage's barrier; the look-ahead stage past
  // the range landed there too); the fragments it prefetched are not used.
  // Round 1, with wavefront kg ^ 1: local token tiles 1 and 3 go out (they
  // are the partner's 0 and 2); round 2 (four groups), with kg ^ 2: local
  // tile 2. A pass moves two tiles of every wavefront, one through each
  // buffer half; slots [wavefront][4][64 lanes] of 16 bytes.
  __syncthreads();
  constexpr int HB = 8 * 4 * 64 * 8;  // bf16 of one tile of every wavefront (32 KiB)
  auto put = [&](uint16_t* buf, const f32x16& c) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const f32x4 q = {c[4 * v], c[4 * v + 1], c[4 * v + 2], c[4 * v + 3]};
      *reinterpret_cast<f32x4*>(buf + ((w * 4 + v) * 64 + lane) * 8) = q;
    }
  };
  auto add = [&](const uint16_t* buf, int from, f32x16& c) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const f32x4 q = *reinterpret_cast<const f32x4*>(buf + ((from * 4 + v) * 64 + lane) * 8);
#pragma unroll
      for (int e = 0; e < 4; ++e) c[4 * v + e] += q[e];
    }
  };
  const int p1 = (kg ^ 1) * RW + rw;
  if constexpr (KG == 4) {
    const int p2 = (kg ^ 2) * RW + rw;
    put(sx0, acc[0][1]);
    put(sx0 + HB, acc[0][3]);
    put(sx1, acc[1][1]);
    put(sx1 + HB, acc[1][3]);
    __syncthreads();
    add(sx0, p1, acc[0][0]);
    add(sx0 + HB, p1, acc[0][2]);
    add(sx1, p1, acc[1][0]);
    add(sx1 + HB, p1, acc[1][2]);
    __syncthreads();
    put(sx0, acc[0][2]);
    put(sx0 + HB, acc[1][2]);
    __syncthreads();
    add(sx0, p2, acc[0][0]);
    add(sx0 + HB, p2, acc[1][0]);
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (i) __syncthreads();
      put(sx0, acc[i][1]);
      put(sx1, acc[i][3]);
      __syncthreads();
      add(sx0, p1, acc[i][0]);
      add(sx1, p1, acc[i][2]);
    }
  }
  // the wavefront's sums: rows er .. +64 of token tiles kg (and, two groups, kg ^ 2)
  constexpr int OT = 4 / KG;
  f32x16 cc[OT][2];
#pragma unroll
  for (int o = 0; o < OT; ++o)
#pragma unroll
    for (int i = 0; i < 2; ++i) cc[o][i] = acc[i][2 * o];
  auto otok = [&](int o) { return m0 + 32 * (kg ^ (2 * o)); };  // first token of tile o

  // ---- depth ranges: every range stores its sums at device scope in their
  // register layout and counts itself at its tile once they are
  // acknowledged; the last to arrive sums the ranges in order and goes on
  // with the epilogue, the others are done
  if (S > 1) {
    const rsrc_t rpp = make_rsrc(a.part + (int64_t)lt * S * R * WT, clamp_bytes((int64_t)S * R * WT * 4));
    auto poff = [&](int r, int v) { return (((uint32_t)r * (8u * OT) + (uint32_t)v) * WNT + (uint32_t)tid) * 16u; };
#pragma unroll
    for (int o = 0; o < OT; ++o)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          mstore16_dev(rpp, opaque_u32(poff(sp, (o * 2 + i) * 4 + v)),
                       (u32x4){__float_as_uint(cc[o][i][4 * v]), __float_as_uint(cc[o][i][4 * v + 1]),
                               __float_as_uint(cc[o][i][4 * v + 2]), __float_as_uint(cc[o][i][4 * v + 3])});
    __builtin_amdgcn_s_waitcnt(0);
    __shared__ int last_range;
    __syncthreads();
    if (tid == 0) {
      last_range = madd_dev(a.mcnt + lt) + 1 == (uint32_t)S;
      if (last_range) mzero_dev(a.mcnt + lt);
    }
    __syncthreads();
    if (!last_range) return;
#pragma unroll
    for (int o = 0; o < OT; ++o)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) cc[o][i][v] = 0.0f;
    // KG ranges at a time (every load of a batch before its sums; ranges past
    // S read zeros): one at a time left a memory round trip per range
    for (int r0 = 0; r0 < S; r0 += KG) {
      u32x4 p[KG][8 * OT];
#pragma unroll
      for (int r = 0; r < KG; ++r)
#pragma unroll
        for (int v = 0; v < 8 * OT; ++v) p[r][v] = mbload16_dev(rpp, opaque_u32(r0 + r < S ? poff(r0 + r, v) : LRQ_OOB));
#pragma unroll
      for (int r = 0; r < KG; ++r)
#pragma unroll
        for (int o = 0; o < OT; ++o)
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
              for (int e = 0; e < 4; ++e) cc[o][i][4 * v + e] += __uint_as_float(p[r][(o * 2 + i) * 4 + v][e]);
    }
  }

  // ---- epilogue
  const int rp = a.rp;
  if (FOLD) {
    // wait for the token-side factor of the tile's 64-token groups (lane
    // i < 2 of wavefront 0 polls group m0 / 64 + i), bounded
    __shared__ int fold_bad;
    const int64_t G = (M + 63) / 64;
    if (w == 0) {
      const int64_t gi = m0 / 64 + lane;
      const bool mine = lane < WT / 64 && gi < G;
      uint32_t polls = 0;
      const uint32_t cap = a.fold < 0 ? 16u : MID_MAX_POLLS;  // the test hook: 16 polls
      bool ok = !mine || mload_dev(a.fcnt + G + gi) == want;
      while (!__all(ok) && polls < cap) {
        __builtin_amdgcn_s_sleep(2);
        ++polls;
        ok = !mine || mload_dev(a.fcnt + G + gi) == want;
      }
      if (lane == 0) {
        fold_bad = __all(ok) ? 0 : 1;
        if (!__all(ok)) __hip_atomic_store(a.fcnt + SK_FAIL, 1u, __ATOMIC_RELAXED, MXSCOPE);
      }
    }
    __syncthreads();
    // the LoRA step: weight-side rows (A role) from LDS, the tile's factor
    // rows (B role) read past the L2s; rank slots 16 kk + 8 g .. +8
    const rsrc_t rfo = make_rsrc(a.fout, clamp_bytes(M * a.fout_ld * 2));
    const bool bad = fold_bad != 0;
    u32x4 lb[OT][2];
#pragma unroll
    for (int o = 0; o < OT; ++o)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const int64_t tok = otok(o) + l32;
        const int j0 = 16 * kk + 8 * g;
        lb[o][kk] = mbload16_dev(rfo, opaque_u32(tok < M && j0 < a.fout_ld ? (uint32_t)((tok * a.fout_ld + j0) * 2) : LRQ_OOB));
        if (bad) lb[o][kk] = (u32x4){0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u};
      }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      if (kk * 16 < rp) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const bf16x8 la = as_bf16x8(ld16(sF + (64 * rw + 32 * i + l32) * FST + 16 * kk + 8 * g));
#pragma unroll
          for (int o = 0; o < OT; ++o) cc[o][i] = mfma32(la, as_bf16x8(lb[o][kk]), cc[o][i]);
        }
      }
    }
  } else if (rp > 0) {
    // weight-side rows [E][rp] and token rows [M][rp] from the workspace
    const rsrc_t rfr = make_rsrc(a.lw + (rok ? er * rp : 0), rok ? clamp_bytes((E - er) * rp * 2) : 0u);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      if (kk * 16 < rp) {
        const uint32_t lo = (uint32_t)((l32 * rp + 16 * kk + 8 * g) * 2);
        const bf16x8 la0 = as_bf16x8(bload16(rfr, opaque_u32(lo)));
        const bf16x8 la1 = as_bf16x8(bload16(rfr, opaque_u32(lo + (uint32_t)(32 * rp * 2))));
#pragma unroll
        for (int o = 0; o < OT; ++o) {
          const int64_t t0 = otok(o);
          const rsrc_t rt = make_rsrc(a.lact + (t0 < M ? t0 * rp : 0), t0 < M ? clamp_bytes((M - t0) * rp * 2) : 0u);
          const bf16x8 lb = as_bf16x8(bload16(rt, opaque_u32(lo)));
          cc[o][0] = mfma32(la0, lb, cc[o][0]);
          cc[o][1] = mfma32(la1, lb, cc[o][1]);
        }
      }
    }
  }
  // output: each [32 tokens][64 rows] bf16 of the wavefront through its own
  // 4 KiB of LDS (16-byte chunk c of token r at c ^ wswz(r)), so that every
  // store writes 128-byte runs. Lane element 4 v + e of row tile i is row
  // 32 i + 8 v + 4 g + e. Two depth groups: the last sums read both buffers,
  // so the staging waits for them.
  if (KG == 2) __syncthreads();
  const float s0v = (!BWD && !GS && !pc) ? a.wscale[0] : 1.0f;
  const rsrc_t rsc = make_rsrc(a.wscale, (!BWD && pc) ? clamp_bytes(E * 4) : 0u);
  const bool has_bias = !BWD && a.bias != nullptr;
  const rsrc_t rbi = make_rsrc(a.bias, has_bias ? clamp_bytes(E * 4) : 0u);
#pragma unroll
  for (int o = 0; o < OT; ++o) {
    uint16_t* const so = (o ? sx0 : sx1) + w * 32 * 64;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const f32x16& c = cc[o][i];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t n = er + 32 * i + 8 * v + 4 * g;
        f32x4 sc = {s0v, s0v, s0v, s0v}, bv = {0.f, 0.f, 0.f, 0.f};
        if (!BWD && pc) sc = __builtin_bit_cast(f32x4, bload16(rsc, opaque_u32(n < E ? (uint32_t)(n * 4) : LRQ_OOB)));
        if (has_bias) bv = __builtin_bit_cast(f32x4, bload16(rbi, opaque_u32(n < E ? (uint32_t)(n * 4) : LRQ_OOB)));
        u32x2 ov;
        ov[0] = pack_bf16x2(__builtin_fmaf(c[4 * v], sc[0], bv[0]), __builtin_fmaf(c[4 * v + 1], sc[1], bv[1]));
        ov[1] = pack_bf16x2(__builtin_fmaf(c[4 * v + 2], sc[2], bv[2]), __builtin_fmaf(c[4 * v + 3], sc[3], bv[3]));
        st8(so + l32 * 64 + (((4 * i + v) ^ wswz(l32)) * 8) + g * 4, ov);
      }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wavefront's rows are in LDS
    const int64_t t0 = otok(o);
    const rsrc_t ry = make_rsrc(a.out + (t0 < M ? t0 * E : 0), t0 < M ? clamp_bytes(min(M - t0, (int64_t)32) * E * 2) : 0u);
    const int64_t ncol = er + (lane & 7) * 8;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int row = 8 * p + (lane >> 3);
      const u32x4 v = ld16(so + row * 64 + ((lane & 7) ^ wswz(row)) * 8);
      __builtin_amdgcn_raw_buffer_store_b128(v, ry, opaque_u32(ncol < E ? (uint32_t)((row * E + ncol) * 2) : LRQ_OOB), 0, 2);
    }
  }
  if (FOLD) mid_flags_done<WNT>(a, ntiles + ((BWD && a.tn_da >= 0) ? a.tj[a.tn_da].blocks : 0));
}

template <bool BWD, int FMT, int RW>
hipError_t run_w8(hipStream_t st, const GemmArgs& a) {
  constexpr int R = 64 * RW;
  const int tiles_m = (int)((a.m + WT - 1) / WT);
  const int tiles_e = (int)((a.e + R - 1) / R);
  const int group_m = tiles_m < 8 ? tiles_m : 8;
  const int S = a.msplit > 1 ? a.msplit : 1;
  const unsigned units = (unsigned)(tiles_m * tiles_e * S);
  if (a.fold) {
    // two factor slices at a time, and two weight-gradient blocks of a job,
    // per workgroup
    GemmArgs b = a;
    const int stages = (int)((a.l + 64 * (8 / RW) - 1) / (64 * (8 / RW)));
    b.fold_wgs = (int)w8_fold_wgs(a.fold_slices * ((a.m + 63) / 64), units, S > 1 ? a.mspl : stages);
    const unsigned tn = BWD ? (unsigned)((a.tj[0].blocks + 1) / 2 + (a.tj[1].blocks + 1) / 2) : 0u;
    hipLaunchKernelGGL((k_w8<BWD, FMT, RW, true>), dim3(units + b.fold_wgs + tn), dim3(WNT), 0, st, b, tiles_m, tiles_e,
                       group_m);
  } else {
    hipLaunchKernelGGL((k_w8<BWD, FMT, RW, false>), dim3(units), dim3(WNT), 0, st, a, tiles_m, tiles_e, group_m);
  }
  return hipGetLastError();
}

template <int RW>
hipError_t run_fmt(hipStream_t st, int fmt, bool bwd, const GemmArgs& a) {
  if (fmt == LRQ_FMT_INT4) return bwd ? run_w8<true, LRQ_FMT_INT4, RW>(st, a) : run_w8<false, LRQ_FMT_INT4, RW>(st, a);
  if (fmt == LRQ_FMT_INT8) return bwd ? run_w8<true, LRQ_FMT_INT8, RW>(st, a) : run_w8<false, LRQ_FMT_INT8, RW>(st, a);
  return bwd ? run_w8<true, LRQ_FMT_FP8, RW>(st, a) : run_w8<false, LRQ_FMT_FP8, RW>(st, a);
}

}  // namespace

// Workgroups for the factor slices (two at a time each, about 4 us). They
// come first, so each one beyond the CUs that the tiles leave free holds up a
// tile by its run time. A tile needs the factor only after its depth: when
// the free CUs can form it in rounds that end by about half of a tile's
// stages (1.5 us each), only they do (512 tokens, 12288 -> 3072, rank 32: 64
// workgroups in two rounds beside 192 tiles, 62 -> 49 us against 128 in one);
// otherwise one round, the least any tile can be held up. A multiple of 8, so
// that the tiles keep their XCDs.
int64_t w8_fold_wgs(int64_t slices, int64_t units, int stages) {
  const int64_t need = (slices + 1) / 2, cus = get_num_cus();
  const int64_t spare = (cus - units % cus) % cus / 8 * 8;
  const int64_t rounds = std::max(1, (int)(stages * 1.5 / 8.0));
  const int64_t wgs = spare * rounds >= need ? std::min(spare, need) : need;
  return (wgs + 7) / 8 * 8;
}

hipError_t launch_w8(hipStream_t st, int fmt, bool bwd, const GemmArgs& a, int rows) {
  return rows == 256 ? run_fmt<4>(st, fmt, bwd, a) : run_fmt<2>(st, fmt, bwd, a);
}
