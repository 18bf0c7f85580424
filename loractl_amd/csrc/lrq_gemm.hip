// The two large GEMMs of the quantized LoRA linear (m > 16 tokens), with the
// weight operand dequantized straight into matrix-core registers:
//
//   forward   y[m, n]  = x[m, k]  . bf16(dq(w))[n, k]^T (+bias) + t[m, :] . B[:, n]
//   backward  dx[m, k] = dy[m, n] . bf16(dq(w))[n, k]            + u[m, :] . A[k, :]^T
//
// (src/quant.rs:175-176 and :229-233 for the base products; the LoRA terms
// are the two small products of src/lora.rs:199-203 and their autodiff, with
// t = bf16(s . x . A), u = bf16(s . dy . B^T) and the weight-side factor
// rows (B^T or A, [rows][rp]) prepared by the LoRA side kernels.)
//
// One kernel template serves both passes. Call the output columns "rows"
// (n forward, k backward) and the reduction index "depth" (k forward, n
// backward). Output tiles are RA rows x 256 tokens; a persistent grid of one
// workgroup per CU walks its tiles, and four wavefronts (one per SIMD) each
// own two 32-row tiles of a tile:
//   - RA = 256: rows 64w .. 64w+63, both row tiles for all 256 tokens;
//   - RA = 192 (when it fills the CUs better, e.g. 3072 output rows): row
//     tile 0 = rows 32w .. +32 for all 256 tokens, row tile 1 = rows
//     128 + 32(w/2) .. +32 for one 128-token half (h = w%2): two wavefronts
//     share that row tile, split by tokens. Those wavefronts see the token
//     tiles rotated by four (local tile j = token tile (j + 4h) % 8), so
//     their half is always local tiles 0..3 and no register index depends on
//     the wavefront.
// Accumulators: v_mfma_f32_32x32x16_bf16, weight rows in the A role, tokens
// in the B role, 2 x 8 tiles of 16 f32 per lane.
//   - weight (A role): each lane loads the packed bytes of its own row from
//     the blocked layout (int4: 16 bytes = 32 depth of one row, fp8: 32
//     bytes), dequantizes them in registers to the exact bf16 operand and
//     feeds the matrix cores. The depth index is permuted inside a 64-wide
//     step: lane group g (lanes 32g .. 32g+31) takes depth 32g + 8kk .. +8 in
//     sub-step kk, so a lane's packed bytes are contiguous. The forward reads
//     the row section (rows n, int4 nibbles q+8, one group scale per lane and
//     step: fma(u, s, -8s) == q*s exactly, then bf16; fp8: the exact e4m3
//     value, its scale applied to the accumulators). The backward reads the
//     transposed section (rows k, depth n): each of a lane's 8 values has its
//     own scale (int4: scale of row n and group k/group; fp8: channel scale of
//     n). Lane l of each 16-lane row holds the scale of depth 32g + 16p + l
//     (p = kk/2, one register per half step) and a DPP row broadcast hands
//     value 8(kk%2) + e to every lane: q (sign-extended nibble, or the e4m3
//     value) times that scale, rounded to bf16 -- the same bf16(q * s) the
//     forward's operand holds;
//   - activations (B role): the 256 x 64 token tile of a step is copied
//     global -> LDS by buffer loads with an LDS destination (each wavefront
//     moves 64 token rows) and read by all four wavefronts;
//   - the pipeline: token tiles in two LDS buffers and packed weights in two
//     register sets, one step ahead, continuing across tiles: the last steps
//     of a tile prefetch the first steps of the workgroup's next tile, so
//     that tile's loads are in flight while this tile's epilogue (LoRA step,
//     bias, stores) runs, and the stores drain under the next tile's
//     matrix-core work. The one barrier of a step sits four matrix-core steps
//     into its fourth sub-step, after the last fragment reads of the current
//     buffer;
//   - the order inside a sub-step: with one wavefront per SIMD nothing else
//     issues while a run of conversions goes by, so what the next sub-step
//     needs (8 activation reads, two weight fragments in 4 or 6 pieces each,
//     and in the fourth sub-step the copies of the refill) is dealt out over
//     the 12 or 16 matrix-core steps. The two passes of the base product at
//     4096 tokens, us (before: reads, conversions and copies in front of the
//     sub-step's matrix-core steps, placed by the compiler):
//                            forward            backward
//       int4  3072->12288    254 -> 252         273 -> 262
//       int4 12288->3072     280 -> 270         268 -> 248
//       int4  4096->4096     116 -> 115         118 -> 112
//       int8  3072->12288    276 -> 257         287 -> 267
//       fp8   3072-> 9216    211 -> 199         223 -> 219
//     which is 1.06 to 1.25 PFLOP/s; a plain bf16 product of these sizes
//     reaches 1.36 to 1.43 here, power-limited;
//   - edges: buffer loads past a resource's size return zeros (partial token
//     and weight tiles, the depth tail and the zero step that rounds a tile's
//     steps up to an even count); padding weight rows and depth columns hold
//     q = 0;
//   - epilogue: the LoRA term is one rank-wide matrix-core step (the tile's
//     token-side and weight-side factor rows, copied into LDS while the
//     tile's main loop runs); then forward fp8 channel scales (they factor
//     out of the depth reduction; B^T arrives divided by them) and the bias;
//     each wavefront then passes its bf16 output rows through LDS so that
//     every store writes whole 128-byte (RA = 256) or 64-byte row segments;
//   - tile order: workgroup b's i-th tile is virtual tile b + i*G, mapped so
//     each XCD (own L2) works on a contiguous range of tiles, grouped four
//     token tiles deep;
//   - split depth: with fewer tiles than CUs (few tokens, or a narrow output)
//     the depth range of every tile is cut into S ranges of whole steps; a
//     work unit is (tile, range), the persistent grid walks units as it walks
//     tiles, each unit writes its f32 accumulators to a partial buffer
//     [S][m][e] (range 0 adds the LoRA term), and k_split_reduce sums the S
//     partials in range order, applies the forward fp8 scales and bias and
//     rounds once to bf16.

#include <atomic>
#include <cmath>
#include <type_traits>

#include "lrq_common.h"
#include "lrq_kernels.h"

namespace {

constexpr int BK = 64;         // reduction step
constexpr int MJ = 8;          // 32-token tiles per wavefront (row tile 0)
constexpr int RB = MJ * 32;    // tokens per tile (256)
constexpr int XBUF = RB * BK;  // bf16 per activation buffer (32 KB)
constexpr int GM = 4;          // token tiles per group of the tile order
constexpr int NBUF = 2;        // pipeline depth (LDS buffers, register sets)

// activation LDS tile [256 rows][64] bf16: 128-byte rows, 16-byte chunk c of
// row r at chunk c ^ swz(r), so the 16 lanes of a read pass (16 rows at one
// logical chunk) cover all 64 banks
LRQ_DEV int swz(int r) { return (r >> 1) & 7; }

// f(0), f(1), .. f(N - 1) with constant arguments
template <int N, int I = 0, class F>
LRQ_DEV void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

// Per-unit load sources: the activation rows of wavefront w's DMA share, the
// weight block row(s) (data; forward int4 scales), backward int4 the byte
// offsets of the two row tiles' group rows in the transposed scale table,
// and the unit's first step and depth range.
struct TileSrc {
  int64_t m0, e0;
  rsrc_t act, wd, ws;
  uint32_t sk0, sk1;
  int k0, sp;
};

template <bool BWD, int FMT, bool R192, bool SPLIT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
k_gemm(GemmArgs a, int tiles_m, int ntiles) {
  constexpr bool I4 = FMT == LRQ_FMT_INT4;
  constexpr bool I8 = FMT == LRQ_FMT_INT8;
  constexpr bool GS = I4 || I8;         // group scales (int4, int8) or channel scales (fp8)
  constexpr int WV = I4 ? 1 : 2;        // 16-byte packed loads per row tile per step
  constexpr int RA = R192 ? 192 : 256;  // rows per tile
  constexpr int MJ1 = R192 ? 4 : MJ;    // token tiles of row tile 1
  constexpr int NSC = GS ? 2 : 1;       // backward scale registers: per row tile (int4, int8) or shared (fp8)
  __shared__ __attribute__((aligned(16))) uint16_t sX0[XBUF];
  __shared__ __attribute__((aligned(16))) uint16_t sX1[XBUF];
  // epilogue region: the tile's LoRA operands (token rows, then weight-side
  // rows, [256][rp] each) copied in during the tile, then each wavefront's
  // output rows
  __shared__ __attribute__((aligned(16))) uint16_t sE[4 * 128 * 64];
  // forward: the tile's bias [256] and fp8 channel scales [256], f32
  __shared__ __attribute__((aligned(16))) float sAux[BWD ? 4 : 2 * 256];

  const int G = gridDim.x;
  const int S = SPLIT ? a.splits : 1;
  const int nunits = ntiles * S;
  int vb = blockIdx.x;
  if (vb >= nunits) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, l32 = lane & 31;
  const int H = R192 ? (w & 1) : 0;  // token-half rotation of this wavefront
  const int64_t M = a.m, K = a.l, E = a.e;
  const int tiles_a = ntiles / tiles_m;
  // rows (within the tile) of the wavefront's two row tiles
  const int ro0 = R192 ? 32 * w : 64 * w;
  const int ro1 = R192 ? 128 + 32 * (w >> 1) : 64 * w + 32;

  const int64_t KB = (K + 63) / 64;
  constexpr uint32_t blkb = I4 ? 2048u : 4096u;  // bytes per 64x64 block
  constexpr uint32_t rowb = I4 ? 32u : 64u;      // bytes per block row
  const uint32_t Gp = (GS && !BWD) ? (uint32_t)((KB * 64) >> a.gshift) : 0u;
  int64_t wbytes, nsc;
  blocked_sizes_dev(FMT, E, K, &wbytes, &nsc, a.gshift);
  const int nk = (int)KB;
  // steps per unit: the whole depth rounded up to whole pipeline rounds, or
  // one split range (a multiple of NBUF; the last range may run past nk)
  const int nkp = SPLIT ? a.spl : (nk + NBUF - 1) / NBUF * NBUF;

  // backward scales: int4 and int8 ST [KGt][64*KB] (row n = depth, group kg
  // of the output row k); fp8 the channel scales [n] or one scalar
  const int64_t NP = KB * 64;
  const int64_t KGt = (BWD && GS) ? (((E + 63) / 64 * 64 + (1 << a.gshift) - 1) >> a.gshift) : 0;
  const bool pc = !GS && a.per_channel;
  const rsrc_t rbs = BWD ? (GS ? make_rsrc(a.wscale, clamp_bytes(KGt * NP * 4))
                               : make_rsrc(a.wscale, pc ? clamp_bytes(K * 4) : 0u))
                         : make_rsrc(a.wscale, 0u);
  // fp8 with one scalar scale: the per-channel loads read zeros, plus this
  const float s0add = (BWD && !GS && !pc) ? a.wscale[0] : 0.0f;

  // sources of virtual unit v (zero-size resources when v is past the grid);
  // the S ranges of a tile are consecutive units
  auto tile_src = [&](int v) -> TileSrc {
    TileSrc t;
    const bool ok = v < nunits;
    const int lu = xcd_remap(ok ? v : 0, nunits);
    const int logical = SPLIT ? lu / S : lu;
    t.sp = SPLIT ? lu % S : 0;
    t.k0 = t.sp * nkp;
    const int grp = logical / (GM * tiles_a), within = logical % (GM * tiles_a);
    const int gm = min(GM, tiles_m - grp * GM);
    const int tm = grp * GM + within % gm, ta = within / gm;
    t.m0 = (int64_t)tm * RB;
    t.e0 = (int64_t)ta * RA;
    const int64_t mw = t.m0 + 64 * w;
    const int64_t mrows = ok ? ((M - mw) < 64 ? (M - mw) : 64) : 0;
    t.act = make_rsrc(a.act + (mw < M ? mw : 0) * K, clamp_bytes(mrows * K * 2));
    // block row of the resource base: the wavefront's own (RA = 256) or the tile's first
    const int64_t nb = t.e0 / 64 + (R192 ? 0 : w);
    t.wd = make_rsrc(a.wdata + nb * KB * blkb, ok ? clamp_bytes(wbytes - nb * KB * blkb) : 0u);
    t.ws = make_rsrc(a.wscale + ((GS && !BWD) ? nb * Gp * 64 : 0),
                     (GS && !BWD && ok) ? clamp_bytes((nsc - nb * Gp * 64) * 4) : 0u);
    t.sk0 = (BWD && GS) ? (uint32_t)(((t.e0 + ro0) >> a.gshift) * NP * 4) : 0u;
    t.sk1 = (BWD && GS) ? (uint32_t)(((t.e0 + ro1) >> a.gshift) * NP * 4) : 0u;
    return t;
  };

  // ---------------- activation DMA: wavefront w moves token rows 64w .. +64
  // 8 buffer loads per step; lane l of load c lands at row 64w + 8c + l/8,
  // physical chunk l%8, and fetches logical chunk (l%8) ^ swz(row), where
  // swz(64w + 8c + l/8) = (4c + l/16) & 7 alternates with the parity of c.
  const int drow = lane >> 3;
  const int dq0 = (lane & 7) ^ ((lane >> 4) & 7), dq1 = (lane & 7) ^ (((lane >> 4) + 4) & 7);
  const uint32_t doff0 = (uint32_t)((drow * K + dq0 * 8) * 2), doff1 = (uint32_t)((drow * K + dq1 * 8) * 2);
  auto dma = [&](uint16_t* buf, const rsrc_t& ract, int kt, int only) {  // copy `only`, or all (-1)
    const int64_t k0 = (int64_t)kt * BK;
    const bool kok0 = k0 + dq0 * 8 < K, kok1 = k0 + dq1 * 8 < K;  // K % 8 == 0
    const uint32_t koff = (uint32_t)(k0 * 2);
    __attribute__((address_space(3))) char* base =
        (__attribute__((address_space(3))) char*)(lds_void*)(buf + 64 * w * BK);
    // the per-load offsets are formed here from opaque bases each step, so
    // the compiler does not keep 16 hoisted copies live across the loop
    const uint32_t o0 = opaque_u32(doff0) + koff, o1 = opaque_u32(doff1) + koff;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if (only >= 0 && c != only) continue;
      const bool kok = (c & 1) ? kok1 : kok0;
      const uint32_t off = opaque_u32(kok ? ((c & 1) ? o1 : o0) + (uint32_t)(c * 8 * K * 2) : LRQ_OOB);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ract, (lds_void*)(base + c * 8 * BK * 2), 16, off, 0, 0, 0);
    }
  };
  // B-role fragment of local token tile j in sub-step kk: token tile
  // j' = (j + 4H) % 8, row 32j' + l32, logical chunk 4g + kk, stored at chunk
  // (4g + kk) ^ swz(l32) (swz(32j' + l32) = swz(l32)). The per-lane chunk
  // bases are fixed (xk: local tiles 0..3, xq: 4..7); tile and buffer offsets
  // are immediates of the LDS read.
  const uint32_t xrow = (uint32_t)(l32 * BK * 2) | (uint32_t)(swz(l32) * 16);
  constexpr uint32_t HALF = 4 * 32 * BK * 2;  // bytes of four token tiles
  uint32_t xk[4], xq[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const uint32_t c = xrow ^ (uint32_t)((4 * g + kk) * 16);
    xk[kk] = opaque_u32(c + (uint32_t)H * HALF);
    xq[kk] = R192 ? opaque_u32(c + (uint32_t)(1 - H) * HALF) : 0u;
  }
  auto xfrag = [&](const uint16_t* buf, int j, int kk) -> bf16x8 {
    const char* b = reinterpret_cast<const char*>(buf);
    if (!R192 || j < 4) return as_bf16x8(ld16(b + xk[kk] + (uint32_t)(j * 32 * BK * 2)));
    return as_bf16x8(ld16(b + xq[kk] + (uint32_t)((j - 4) * 32 * BK * 2)));
  };

  // ---------------- weight: offsets from the resource's block row: the
  // lane's part (row l32 of a row tile, lane group g's 16 (int4) or 32 (fp8,
  // int8) bytes; group scale of row l32) plus a wavefront-uniform part per row tile
  // (a constant for RA = 256, so it folds into the loads' immediates)
  const uint32_t woff = (uint32_t)l32 * rowb + (uint32_t)g * (I4 ? 16u : 32u);
  const uint32_t soff = (uint32_t)l32 * 4u;
  auto wrow = [&](int i) -> uint32_t {  // uniform data offset of row tile i
    if (!R192) return (uint32_t)i * 32u * rowb;
    const int ro = i ? ro1 : ro0;
    return (uint32_t)(ro >> 6) * (uint32_t)KB * blkb + (uint32_t)(ro & 63) * rowb;
  };
  auto srow = [&](int i) -> uint32_t {  // uniform group-scale offset of row tile i
    if (!R192) return (uint32_t)i * 128u;
    const int ro = i ? ro1 : ro0;
    return ((uint32_t)(ro >> 6) * Gp * 64u + (uint32_t)(ro & 63)) * 4u;
  };
  // backward: lane l of a 16-lane row holds the scale of depth 32g + 16p + l%16
  const uint32_t bsoff = (uint32_t)(32 * g + (lane & 15)) * 4u;
  u32x4 wp[NBUF][2 * WV];   // packed weight bytes per register set
  float wsc[NBUF][2];       // forward int4 / int8 group scales per register set
  float bsc[NBUF][NSC][2];  // backward per-depth scales, two halves of a step
  auto load_w = [&](int set, const TileSrc& t, int kt) {
    // steps past the tile's last one read zeros (bytes and scales)
    const uint32_t kb = opaque_u32(kt < nk ? (uint32_t)kt * blkb : LRQ_OOB);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int h = 0; h < WV; ++h) wp[set][i * WV + h] = bload16(t.wd, kb + woff + wrow(i) + 16u * h);
    if (!BWD && GS) {
      const uint32_t j = ((uint32_t)kt * 64u + (uint32_t)g * 32u) >> a.gshift;
      const uint32_t so = opaque_u32(kt < nk ? (j * 64u) * 4u : LRQ_OOB);
#pragma unroll
      for (int i = 0; i < 2; ++i) wsc[set][i] = bloadf(t.ws, so + soff + srow(i));
    }
    if (BWD) {
      const uint32_t sb = opaque_u32(kt < nk ? (uint32_t)kt * 256u + bsoff : LRQ_OOB);
      if (GS) {
        bsc[set][0][0] = bloadf(rbs, sb + t.sk0);
        bsc[set][0][1] = bloadf(rbs, sb + t.sk0 + 64u);
        bsc[set][NSC - 1][0] = bloadf(rbs, sb + t.sk1);
        bsc[set][NSC - 1][1] = bloadf(rbs, sb + t.sk1 + 64u);
      } else {
        bsc[set][0][0] = bloadf(rbs, sb) + s0add;
        bsc[set][0][1] = bloadf(rbs, sb + 64u) + s0add;
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
    const float S = bsc[set][GS ? i : 0][kk >> 1];
    if (I4) {
      const uint32_t d = wp[set][i][kk];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = (float)((int)(d << (28 - 4 * e)) >> 28);
    } else if (I8) {
      const u32x4 v = wp[set][i * WV + (kk >> 1)];
      int8x4_to_f32(v[2 * (kk & 1)], f);
      int8x4_to_f32(v[2 * (kk & 1) + 1], f + 4);
    } else {
      const u32x4 v = wp[set][i * WV + (kk >> 1)];
      fp8x4_to_f32(v[2 * (kk & 1)], f);
      fp8x4_to_f32(v[2 * (kk & 1) + 1], f + 4);
    }
    mul_row_bcast8(f, S, kk & 1);
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] = pack_bf16x2(f[2 * q], f[2 * q + 1]);
    return as_bf16x8(o);
  };

  f32x16 acc[2][MJ];
  auto zero_acc = [&]() {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < MJ; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
  };

  uint16_t* const bufs[2] = {sX0, sX1};
  bf16x8 fa[2][2], fb[2][MJ];

  // The A-role fragment of row tile i, sub-step kk in pieces: piece p
  // (0 .. NPC - 1) forms part of `o` (wfrag's value once all have run). The
  // pieces sit one by one between matrix-core steps: left to itself, the
  // compiler runs 15 to 30 of these instructions in a row with the matrix
  // cores idle (one wavefront per SIMD has nothing else to issue), then eight
  // matrix-core steps with none.
  constexpr int NPC = BWD ? 6 : 4;  // forward: two values each; backward: 2, 2, scale and pack four, again
  auto wpiece = [&](int set, int i, int kk, int p, float (&f)[8], u32x4& o) {
    const u32x4 v = wp[set][i * WV + (I4 ? 0 : (kk >> 1))];
    const uint32_t d4 = v[kk];                                     // int4: eight nibbles
    const uint32_t d8[2] = {v[2 * (kk & 1)], v[2 * (kk & 1) + 1]};  // 8-bit: two dwords of four
    if (!BWD) {
      const int e = 2 * p;  // values e, e + 1
      if (I4) {
        const float sc = wsc[set][i], nb = -8.0f * sc;
        const uint32_t lo = d4 & a.nib, hi = (d4 >> 4) & a.nib;
        o[p] = pack_bf16x2(__builtin_fmaf((float)((lo >> (8 * p)) & 0xffu), sc, nb),
                           __builtin_fmaf((float)((hi >> (8 * p)) & 0xffu), sc, nb));
      } else if (I8) {
        const float sc = wsc[set][i], nb = -128.0f * sc;
        const uint32_t u = d8[e >> 2] ^ 0x80808080u;
        o[p] = pack_bf16x2(__builtin_fmaf((float)((u >> (8 * (e & 3))) & 0xffu), sc, nb),
                           __builtin_fmaf((float)((u >> (8 * (e & 3) + 8)) & 0xffu), sc, nb));
      } else {
        const f32x2 q = (e & 2) ? __builtin_amdgcn_cvt_pk_f32_fp8((int)d8[e >> 2], true)
                                : __builtin_amdgcn_cvt_pk_f32_fp8((int)d8[e >> 2], false);
        o[p] = pack_bf16x2(q[0], q[1]);
      }
      asm volatile("" : "+v"(o[p]));  // formed here, not where it is first used
      return;
    }
    const int h = p / 3, r = p % 3;  // four values 4 h .. 4 h + 3
    if (r < 2) {
      const int e = 4 * h + 2 * r;
      if (I4) {
        f[e] = (float)((int)(d4 << (28 - 4 * e)) >> 28);
        f[e + 1] = (float)((int)(d4 << (24 - 4 * e)) >> 28);
      } else if (I8) {
        f[e] = (float)((int)(d8[h] << (24 - 16 * r)) >> 24);
        f[e + 1] = (float)((int)(d8[h] << (16 - 16 * r)) >> 24);
      } else {
        const f32x2 q = r ? __builtin_amdgcn_cvt_pk_f32_fp8((int)d8[h], true)
                          : __builtin_amdgcn_cvt_pk_f32_fp8((int)d8[h], false);
        f[e] = q[0];
        f[e + 1] = q[1];
      }
      asm volatile("" : "+v"(f[e]), "+v"(f[e + 1]));
      return;
    }
    mul_row_bcast4(f[4 * h], f[4 * h + 1], f[4 * h + 2], f[4 * h + 3], bsc[set][GS ? i : 0][kk >> 1], 8 * (kk & 1) + 4 * h);
    o[2 * h] = pack_bf16x2(f[4 * h], f[4 * h + 1]);
    o[2 * h + 1] = pack_bf16x2(f[4 * h + 2], f[4 * h + 3]);
    asm volatile("" : "+v"(o[2 * h]), "+v"(o[2 * h + 1]));
  };

  // One step on LDS buffer `b` and register set `b` (b = step % 2; the
  // unrolled loop makes both static). On entry fa[0] and fb[0] hold sub-step
  // 0's fragments; on exit they hold the next step's. After the barrier the
  // step refills buffer and set b with step `lkt` of tile `ls`. Each
  // matrix-core step is followed by its share of the next sub-step's
  // fragment reads and dequantization pieces (sub-step 3: and of the refill).
  auto step = [&](auto bc, const TileSrc& ls, const int lkt) {
    constexpr int b = decltype(bc)::value, nb_ = (b + 1) % NBUF;
    uint16_t* const buf = b ? sX1 : sX0;
    uint16_t* const nbuf = b ? sX0 : sX1;
    constexpr int SLOTS = MJ + MJ1;
    constexpr int BAR = 4;  // sub-step 3: slots before the barrier
    // Whether a sched_barrier ends every slot, or the compiler places the
    // pieces. Without / with, us at the sizes above: int4 backward 272 / 262,
    // 256 / 248, 115 / 112, int8 261 / 257 and 279 / 267, fp8 forward 204 /
    // 199; but int4 forward (the fewest conversions) 252 / 259, 270 / 274,
    // 115 / 119 and fp8 backward (the most) 219 / 226.
    constexpr bool SB = !(I4 && !BWD) && !(FMT == LRQ_FMT_FP8 && BWD);
    static_for<4>([&](auto kc) {
      constexpr int kk = decltype(kc)::value, cur = kk & 1;
      float f[2][8];
      u32x4 o[2];
      static_for<SLOTS>([&](auto sc) {
        constexpr int s = decltype(sc)::value;
        // both row tiles of a token tile in turn (row tile 0's others last), but
        // one row tile after the other where the compiler places the pieces
        constexpr int i = SB ? (s < 2 * MJ1 ? s & 1 : 0) : (s < MJ ? 0 : 1);
        constexpr int j = SB ? (s < 2 * MJ1 ? s / 2 : s - MJ1) : (s < MJ ? s : s - MJ);
        acc[i][j] = mfma32(fa[cur][i], fb[cur][j], acc[i][j]);
        if (kk < 3 && s < MJ) fb[cur ^ 1][s < MJ ? s : 0] = xfrag(buf, s, kk + 1);
        if (kk == 3) {
          // every read of buffer b is issued: one barrier, then refill buffer
          // and register set b (its last pieces ran in sub-step 2), and read
          // the next step's first fragments from the other buffer
          if (s == BAR) {
            // the copies into the other buffer have landed: said here, since
            // the compiler does not carry them over the loop's back edge
            __builtin_amdgcn_s_waitcnt(0xf70);  // vmcnt(0)
            __syncthreads();
            load_w(b, ls, lkt);
          }
          if (s >= BAR && s < BAR + MJ) {
            dma(buf, ls.act, lkt, s - BAR);
            fb[cur ^ 1][(s - BAR) & (MJ - 1)] = xfrag(nbuf, s - BAR, 0);
          }
        }
        constexpr int p0 = s * 2 * NPC / SLOTS, p1 = (s + 1) * 2 * NPC / SLOTS;
        static_for<p1 - p0>([&](auto pc) {
          constexpr int p = p0 + decltype(pc)::value;
          wpiece(kk < 3 ? b : nb_, p / NPC, (kk + 1) & 3, p % NPC, f[p / NPC], o[p / NPC]);
        });
        if constexpr (SB) __builtin_amdgcn_sched_barrier(0);
      });
      fa[cur ^ 1][0] = as_bf16x8(o[0]);
      fa[cur ^ 1][1] = as_bf16x8(o[1]);
    });
  };

  const int rp = a.rp;
  // LoRA operands of a tile: token rows [m0, m0+256) and weight-side rows
  // [e0, e0+256) (only RA of them used), 256 * rp bf16 each, contiguous in
  // global memory (rows past M or E read zeros); copied to sE as [256][rp]
  // each, 16 bytes per lane per load
  const rsrc_t rbt = make_rsrc(a.lw, rp > 0 ? clamp_bytes(E * rp * 2) : 0u);
  const rsrc_t rt = make_rsrc(a.lact, rp > 0 ? clamp_bytes(M * rp * 2) : 0u);
  const int lora_loads = rp / 8;  // 16-byte loads per lane per operand: 256*rp*2 / (256*16)
  const bool has_bias = !BWD && a.bias != nullptr;
  const bool fpc = !BWD && pc;  // forward fp8 channel scales in the epilogue
  const rsrc_t rbias = make_rsrc(a.bias, has_bias ? clamp_bytes(E * 4) : 0u);
  const rsrc_t rsc = make_rsrc(a.wscale, fpc ? clamp_bytes(E * 4) : 0u);
  // copies for the tile at (m0, e0), issued at its start: LoRA operands to sE,
  // forward bias and fp8 channel scales of its output columns to sAux
  // (columns past E read zeros)
  auto dma_aux = [&](int64_t m0, int64_t e0) {
    __attribute__((address_space(3))) char* base = (__attribute__((address_space(3))) char*)(lds_void*)sE;
    const uint32_t tb = (uint32_t)(m0 * rp * 2), bb = (uint32_t)(e0 * rp * 2);
    for (int c = 0; c < lora_loads; ++c) {
      const uint32_t o = (uint32_t)((c * 256 + w * 64) * 16);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rt, (lds_void*)(base + o), 16, opaque_u32(tb + o + lane * 16), 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rbt, (lds_void*)(base + 256 * rp * 2 + o), 16,
                                               opaque_u32(bb + o + lane * 16), 0, 0, 0);
    }
    if (!BWD) {
      __attribute__((address_space(3))) char* abase = (__attribute__((address_space(3))) char*)(lds_void*)sAux;
      const uint32_t co = opaque_u32((uint32_t)(e0 * 4 + lane * 16));
      if (w == 0 && has_bias) __builtin_amdgcn_raw_ptr_buffer_load_lds(rbias, (lds_void*)abase, 16, co, 0, 0, 0);
      if (w == 1 && fpc) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsc, (lds_void*)(abase + 256 * 4), 16, co, 0, 0, 0);
    }
  };

  // epilogue of the tile at (m0, e0). Its per-lane values are derived from
  // an opaque copy of the lane id, so the compiler recomputes them per tile
  // instead of hoisting them out of the tile loop (where they would only be
  // spilled: the main loop holds the registers).
  auto epilogue = [&](int64_t m0, int64_t e0) {
    const int lane = (int)opaque_u32((uint32_t)threadIdx.x & 63u);
    const int g = lane >> 5, l32 = lane & 31;
    // LoRA: one rank-wide step from sE; A role = weight-side rows ro_i + l32,
    // B role = token rows 32 ((j + 4H) % 8) + l32, rank columns 16kk + 8g .. +8
    if (rp > 0) {
      const uint16_t* sT = sE;
      const uint16_t* sBt = sE + 256 * rp;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        if (kk * 16 < rp) {
          bf16x8 la[2];
          la[0] = as_bf16x8(ld16(sBt + (ro0 + l32) * rp + kk * 16 + g * 8));
          la[1] = as_bf16x8(ld16(sBt + (ro1 + l32) * rp + kk * 16 + g * 8));
#pragma unroll
          for (int j = 0; j < MJ; ++j) {
            const int tj = R192 ? ((j + 4 * H) & 7) : j;
            const bf16x8 lb = as_bf16x8(ld16(sT + (32 * tj + l32) * rp + kk * 16 + g * 8));
            acc[0][j] = mfma32(la[0], lb, acc[0][j]);
            if (j < MJ1) acc[1][j] = mfma32(la[1], lb, acc[1][j]);
          }
        }
      }
    }
    // keep the accumulators in AGPRs here: the packing below then copies one
    // tile at a time to VGPRs, instead of the whole set before the LoRA step
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < MJ; ++j) asm volatile("" : "+a"(acc[i][j]));
    // every wavefront's LoRA reads are done before sE takes output rows
    __syncthreads();
    // output: per half of the local tokens, the wavefront's [128 tokens][64]
    // bf16 staging rows (columns 0..31 row tile 0, 32..63 row tile 1) go to
    // its sE slice (16-byte chunk c of row r at c ^ swz(r)), then back out in
    // row segments, 8 rows per store
    uint16_t* sO = sE + w * 128 * 64;
    const float s0 = (!BWD && !GS && !pc) ? a.wscale[0] : 1.0f;
    // output rows of this tile: a resource from row m0, so rows past M fall
    // outside it
    const rsrc_t ry = make_rsrc(a.out + m0 * E, clamp_bytes((M - m0) * E * 2));
    const int rr = lane >> 3, cc = lane & 7;
    // staging chunk cc: column 8cc of row tile 0 (cc < 4) or 8(cc-4) of row
    // tile 1; RA = 256 keeps the two row tiles adjacent
    const int64_t ncol = e0 + (R192 ? ((cc < 4) ? ro0 + 8 * cc : ro1 + 8 * (cc - 4)) : ro0 + 8 * cc);
    const uint32_t ybase0 = (uint32_t)(ncol * 2);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const int row = 32 * jj + l32;
        // one 32-token tile at a time, so few accumulators are in flight
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if (R192 && i == 1 && h == 1) continue;  // row tile 1 covers local tokens 0..127
#pragma unroll
          for (int vg = 0; vg < 4; ++vg) {
            const int ro = i ? ro1 : ro0;
            const f32x4 bv = has_bias ? *reinterpret_cast<const f32x4*>(sAux + ro + 8 * vg + 4 * g)
                                      : (f32x4){0.f, 0.f, 0.f, 0.f};
            // forward fp8: the per-output-channel scale factors out of the
            // depth reduction (the LoRA operand bt arrives divided by it);
            // per-channel scales of columns past E are zero (not stored)
            const f32x4 sv = (BWD || GS) ? (f32x4){1.f, 1.f, 1.f, 1.f}
                                         : (pc ? *reinterpret_cast<const f32x4*>(sAux + 256 + ro + 8 * vg + 4 * g)
                                               : (f32x4){s0, s0, s0, s0});
            const f32x16& c = acc[i][4 * h + jj];
            u32x2 o;
            o[0] = pack_bf16x2(__builtin_fmaf(c[4 * vg + 0], sv[0], bv[0]), __builtin_fmaf(c[4 * vg + 1], sv[1], bv[1]));
            o[1] = pack_bf16x2(__builtin_fmaf(c[4 * vg + 2], sv[2], bv[2]), __builtin_fmaf(c[4 * vg + 3], sv[3], bv[3]));
            const int chunk = (4 * i + vg) ^ swz(row);
            st8(sO + row * 64 + chunk * 8 + g * 4, o);
          }
        }
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wavefront's rows are in LDS
      // local half h holds tokens m0 + 128 (h ^ H) ..
      const uint32_t ybase = ybase0 + (uint32_t)(128 * (h ^ H) * E * 2);
      const bool cok = ncol < E && !(R192 && h == 1 && cc >= 4);
#pragma unroll
      for (int p = 0; p < 16; ++p) {
        const int row = 8 * p + rr;
        const u32x4 v = ld16(sO + row * 64 + (cc ^ swz(row)) * 8);
        // columns past E (and the unused half of row tile 1) are skipped
        // (offset past the resource); rows past M are past it already
        const uint32_t off = cok ? ybase + (uint32_t)(row * E * 2) : LRQ_OOB;
        // non-temporal (aux bit 1): the output is not read again in this
        // launch, and streaming it past the caches keeps the activation and
        // weight tiles there (the north-star step 0.9% faster)
        __builtin_amdgcn_raw_buffer_store_b128(v, ry, opaque_u32(off), 0, 2);
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);  // reads done before the next half's writes
    }
  };

  // split-depth epilogue: range 0 adds the LoRA term; every range stores
  // its f32 accumulators to part[range][m][e], four consecutive e per 16-byte
  // store (rows past M fall outside the resource, columns past E are skipped)
  auto epilogue_partial = [&](const TileSrc& u) {
    const int lane = (int)opaque_u32((uint32_t)threadIdx.x & 63u);
    const int g = lane >> 5, l32 = lane & 31;
    if (rp > 0 && u.sp == 0) {
      const uint16_t* sT = sE;
      const uint16_t* sBt = sE + 256 * rp;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        if (kk * 16 < rp) {
          bf16x8 la[2];
          la[0] = as_bf16x8(ld16(sBt + (ro0 + l32) * rp + kk * 16 + g * 8));
          la[1] = as_bf16x8(ld16(sBt + (ro1 + l32) * rp + kk * 16 + g * 8));
#pragma unroll
          for (int j = 0; j < MJ; ++j) {
            const int tj = R192 ? ((j + 4 * H) & 7) : j;
            const bf16x8 lb = as_bf16x8(ld16(sT + (32 * tj + l32) * rp + kk * 16 + g * 8));
            acc[0][j] = mfma32(la[0], lb, acc[0][j]);
            if (j < MJ1) acc[1][j] = mfma32(la[1], lb, acc[1][j]);
          }
        }
      }
    }
    const rsrc_t rp_ = make_rsrc(a.part + ((int64_t)u.sp * M + u.m0) * E, clamp_bytes((M - u.m0) * E * 4));
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < (i == 0 ? MJ : MJ1); ++j) {
        const int tj = R192 ? ((j + 4 * H) & 7) : j;
        const uint32_t rowoff = (uint32_t)((32 * tj + l32) * E * 4);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int vg = 0; vg < 4; ++vg) {
          const int64_t e = u.e0 + (i ? ro1 : ro0) + 8 * vg + 4 * g;
          const f32x16& c = acc[i][j];
          const u32x4 v = {__float_as_uint(c[4 * vg]), __float_as_uint(c[4 * vg + 1]), __float_as_uint(c[4 * vg + 2]),
                           __float_as_uint(c[4 * vg + 3])};
          const uint32_t off = e < E ? rowoff + (uint32_t)(e * 4) : LRQ_OOB;
          __builtin_amdgcn_raw_buffer_store_b128(v, rp_, opaque_u32(off), 0, 0);
        }
      }
  };

  // prologue: the first tile's first two steps in flight
  TileSrc cur = tile_src(vb);
#pragma unroll
  for (int b = 0; b < NBUF; ++b) {
    dma(bufs[b], cur.act, cur.k0 + b, -1);
    load_w(b, cur, cur.k0 + b);
  }
  dma_aux(cur.m0, cur.e0);
  zero_acc();
  __builtin_amdgcn_s_waitcnt(0xf70);  // vmcnt(0)
  __syncthreads();
#pragma unroll
  for (int j = 0; j < MJ; ++j) fb[0][j] = xfrag(bufs[0], j, 0);
#pragma unroll
  for (int i = 0; i < 2; ++i) fa[0][i] = wfrag(0, i, 0);

  for (;;) {
    int kt = 0;
    for (; kt + NBUF < nkp; kt += NBUF) {
      step(std::integral_constant<int, 0>{}, cur, cur.k0 + kt + NBUF);
      step(std::integral_constant<int, 1>{}, cur, cur.k0 + kt + NBUF + 1);
    }
    // last two steps: prefetch the next unit's first steps
    const TileSrc nxt = tile_src(vb + G);
    step(std::integral_constant<int, 0>{}, nxt, nxt.k0);
    step(std::integral_constant<int, 1>{}, nxt, nxt.k0 + 1);
    if (SPLIT)
      epilogue_partial(cur);
    else
      epilogue(cur.m0, cur.e0);
    vb += G;
    if (vb >= nunits) break;
    zero_acc();
    cur = nxt;
    // every wavefront's output reads of sE are done before the next tile's
    // LoRA operands land there
    __syncthreads();
    dma_aux(cur.m0, cur.e0);
  }
  // drain the look-ahead copies before the workgroup ends
  __builtin_amdgcn_s_waitcnt(0);
}

template <bool BWD, int FMT, bool R192, bool SPLIT>
hipError_t run(hipStream_t st, const GemmArgs& a) {
  constexpr int RA = R192 ? 192 : 256;
  const int tiles_m = (int)((a.m + RB - 1) / RB);
  const int tiles_e = (int)((a.e + RA - 1) / RA);
  const int ntiles = tiles_m * tiles_e;
  const int nunits = ntiles * (SPLIT ? a.splits : 1);
  const int grid = nunits < get_num_cus() ? nunits : get_num_cus();
  hipLaunchKernelGGL((k_gemm<BWD, FMT, R192, SPLIT>), dim3(grid), dim3(256), 0, st, a, tiles_m, ntiles);
  return hipGetLastError();
}

// 192-row tiles when they fill the CUs in fewer rounds of work: a tile round
// of RA = 192 costs about 0.8 of a 256-row round (3/4 of the matrix-core
// work, with a larger dequantization share).
bool use_r192(int64_t m, int64_t e) {
  const int64_t tm = (m + RB - 1) / RB, cus = get_num_cus();
  const int64_t r256 = ((e + 255) / 256 * tm + cus - 1) / cus;
  const int64_t r192 = ((e + 191) / 192 * tm + cus - 1) / cus;
  return 0.8 * (double)r192 < (double)r256 - 1e-9;
}

// out[m, e] = bf16(sc(e) * sum over ranges (in order) of part[s][m][e] +
// bias(e)); sc = the forward fp8 channel scale or scalar, else 1. Four
// consecutive e per thread (e % 4 == 0).
__global__ void __launch_bounds__(256) k_split_reduce(const float* __restrict__ part, int S, int64_t M, int64_t E,
                                                      const float* __restrict__ scale, int per_channel,
                                                      const float* __restrict__ bias, uint16_t* __restrict__ out) {
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= M * E / 4) return;
  const int64_t e = (q * 4) % E;
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < S; ++s) {
    const f32x4 v = reinterpret_cast<const f32x4*>(part + (int64_t)s * M * E)[q];
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[i] += v[i];
  }
  f32x4 sc = {1.f, 1.f, 1.f, 1.f}, bv = {0.f, 0.f, 0.f, 0.f};
  if (scale) sc = per_channel ? *reinterpret_cast<const f32x4*>(scale + e) : (f32x4){scale[0], scale[0], scale[0], scale[0]};
  if (bias) bv = *reinterpret_cast<const f32x4*>(bias + e);
  u32x2 o;
  o[0] = pack_bf16x2(__builtin_fmaf(sum[0], sc[0], bv[0]), __builtin_fmaf(sum[1], sc[1], bv[1]));
  o[1] = pack_bf16x2(__builtin_fmaf(sum[2], sc[2], bv[2]), __builtin_fmaf(sum[3], sc[3], bv[3]));
  reinterpret_cast<u32x2*>(out)[q] = o;
}

// Depth ranges: with fewer output tiles than CUs, as many ranges as fill the
// CUs once, of at least four steps each (at most 16 ranges).
struct SplitPlan {
  bool r192;
  int S, spl;
};
SplitPlan plan_split(int64_t m, int64_t e, int64_t depth) {
  SplitPlan p{};
  p.r192 = use_r192(m, e);
  const int64_t RA = p.r192 ? 192 : 256;
  const int64_t tiles = (m + RB - 1) / RB * ((e + RA - 1) / RA), cus = get_num_cus();
  const int64_t nk = (depth + 63) / 64;
  int64_t S = 1;
  if (tiles > 0 && tiles < cus) {
    S = cus / tiles;
    if (S > nk / 4) S = nk / 4;
    if (S > 16) S = 16;
    if (S < 1) S = 1;
  }
  int64_t spl = (nk + S - 1) / S;
  spl = (spl + NBUF - 1) / NBUF * NBUF;
  p.spl = (int)spl;
  p.S = (int)((nk + spl - 1) / spl);  // every range holds at least one step
  return p;
}


template <bool BWD, bool SPLIT>
hipError_t run_fmt(hipStream_t st, int fmt, bool r192, const GemmArgs& a) {
  if (fmt == LRQ_FMT_INT4)
    return r192 ? run<BWD, LRQ_FMT_INT4, true, SPLIT>(st, a) : run<BWD, LRQ_FMT_INT4, false, SPLIT>(st, a);
  if (fmt == LRQ_FMT_INT8)
    return r192 ? run<BWD, LRQ_FMT_INT8, true, SPLIT>(st, a) : run<BWD, LRQ_FMT_INT8, false, SPLIT>(st, a);
  return r192 ? run<BWD, LRQ_FMT_FP8, true, SPLIT>(st, a) : run<BWD, LRQ_FMT_FP8, false, SPLIT>(st, a);
}

// Which GEMM kernel a shape takes: the 256-token tiles above (split in
// depth when they are too few), lrq_gemm_mid.hip's 64-row x 64-token tiles,
// two workgroups per CU, lrq_gemm_w8.hip's 128-token tiles of 128 or 256
// rows, one workgroup per CU, or, for a backward that forms its LoRA factors,
// lrq_gemm_mid.hip's 64-row x 128-token tiles (few outputs at 100 to 640
// tokens: 8192 -> 512 at 128 tokens, rank 16, 13.1 us against 14.2 on the best
// of the others; 3072 -> 3072 at 384 tokens, rank 32, 25.7 against 28.0). The
// choice is the smallest modelled time, in microseconds:
//   - large tiles: LARGE_STEP_US per 256 x 256 x 64 step, LARGE_192 of it for
//     192-row tiles; a split shape's f32 partials (LARGE_SPLIT_MB per MB) and
//     its reduction launch (LARGE_SPLIT_US);
//   - two-per-CU tiles: MID_A per 64-wide depth block when a workgroup has
//     its CU to itself and MID_B each when two share it, the tiles dealt over
//     the CUs two at a time, MID_ROUND_US for each further round;
//   - 128-token tiles: MID_A + MID_B x (the share of the CUs at work: the
//     power limit) per stage, whole rounds of tiles;
//   - MID_FIX per tile: its start and end;
//   - depth ranges: RANGE_US, RANGE_EACH_US per range and RANGE_MB_US per MB
//     of partials written and read. Only where every range's workgroup has a
//     place at once: with more of them the partials cost more than the
//     ranges gave (1024 tokens, 16384 -> 9216: 150 MB in four ranges, 347 us
//     against 316 on the large tiles), and they are bounded by 34 MB;
//   - LoRA factors in the launch (fold_us): FOLD_US, and FOLD_LATE_US when
//     the factor slices' workgroups take places that tiles need. A
//     weight-gradient block takes TN_US + TN_TOKENS_US per 128 tokens
//     (TN_R32 as long at rank 32): as many as the places free beside the
//     tiles can take while these run cost nothing but what they slow the tiles
//     (SHARE_US at ranks to 16 and 32, for full CUs), the others follow the
//     tiles, and dA's blocks wait for u (CHAIN_US);
//   - the large tiles' launches for t, or for u and for dA and dB:
//     LARGE_SIDE_US. (A call that gives up the folded plan takes the kernel
//     that is fastest without the factors, the large tiles or not.)
// The constants are fitted to 153000 timings of every kernel and range count
// over 13400 calls (17 to 16384 tokens, layers 512 to 32768 wide, every
// format, ranks 0 to 64) so that the plan's own time is least: it is 1.3 %
// above the fastest kernel's on average, and 4 of 100 calls take more
// than a tenth longer.
// Decided on whole 64-token groups, so that a workspace reserved for the
// largest of a group's token counts serves them all. A plan keeps the limits
// of the call (its workspace, the counter area) and of the launch (32-bit
// buffer offsets).
//
// By format: int4, int8, fp8; pairs: forward, input gradient.
constexpr double LARGE_STEP_US[3][2] = {{1.434, 1.341}, {1.419, 1.382}, {1.393, 1.6}};
constexpr double LARGE_192 = 0.843, LARGE_US = 11.01;
constexpr double LARGE_SPLIT_US = 8.05, LARGE_SPLIT_MB = 0.525, LARGE_SIDE_US[2] = {11.87, 21.74};
// per MID_64, MID_128, MID_256, MID_64X128: tile tokens and rows, 64-deep
// blocks per pipeline stage, stages a depth range is a multiple of, and the
// most ranges; then the model's
constexpr int MID_T[5] = {0, 64, W8_TOKENS, W8_TOKENS, 128}, MID_R[5] = {0, 64, 128, 256, 64};
constexpr int MID_SD[5] = {0, 2, 4, 2, 1};
constexpr int MID_ROUND[5] = {0, MID_MST, 1, 1, MID_MST};
constexpr int MID_MAXS[5] = {0, MID_MAX_SPLIT, W8_MAX_SPLIT, W8_MAX_SPLIT, MID_MAX_SPLIT};
constexpr double MID_A[3][2][5] =
    {{{0, 0.33, 1.065, 1.099, 0}, {0, 0.319, 1.368, 1.301, 0.453}},
     {{0, 0.322, 1.264, 1.217, 0}, {0, 0.273, 1.456, 1.344, 0.484}},
     {{0, 0.204, 1.272, 1.388, 0}, {0, 0.308, 1.425, 1.322, 0.524}}};
constexpr double MID_B[3][2][5] =
    {{{0, 0.436, 0.548, 0.36, 0}, {0, 0.407, 0.344, 0.215, 0.611}},
     {{0, 0.433, 0.545, 0.285, 0}, {0, 0.408, 0.297, 0.131, 0.858}},
     {{0, 0.29, 0.543, 0.252, 0}, {0, 0.409, 0.434, 0.226, 0.645}}};
constexpr double MID_FIX[2][5] = {{0, 3.56, 6.33, 5.76, 2.23}, {0, 1.19, 5.34, 5.45, 1.92}};
constexpr double MID_ROUND_US[5] = {0, 10.48, 0, 0, 6.66};
constexpr double RANGE_US[5] = {0, 1.09, 2.26, 2.55, 1.24}, RANGE_EACH_US[5] = {0, 0, 0.88, 1.13, 0};
constexpr double RANGE_MB_US[5] = {0, 0.117, 0, 0.112, 0.166};
constexpr double FOLD_US[5] = {0, 1.63, 1.36, 3.35, 0.3}, FOLD_LATE_US[5] = {0, 2.29, 7.21, 5.07, 6.45};
constexpr double TN_US[5] = {0, 3.34, 0.55, 0.19, 2.09}, TN_TOKENS_US[5] = {0, 1.12, 0.76, 0.94, 0.69};
constexpr double TN_R32 = 1.985, CHAIN_US[5] = {0, 1.39, 18.43, 0.55, 9.5};
constexpr double SHARE_US[2][5] = {{0, 2.38, 0.92, 0.15, 4.59}, {0, 4.18, 4.16, 0.4, 12.99}};
bool is_w8(int v) { return v == MID_128 || v == MID_256; }
int model_fmt(int fmt) { return fmt == LRQ_FMT_INT4 ? 0 : fmt == LRQ_FMT_INT8 ? 1 : 2; }
// lrq_debug_gemm_path: 0 planned, 1 large tiles, 2 and 3 MID_64 and MID_128,
// 4 and 5 these with at least two depth ranges where the depth has them; 6
// and 7 the same for MID_256, 8 and 9 for MID_64X128 (where it runs)
int g_gemm_path = 0;

double large_us(int fmt, int64_t m, int64_t e, int64_t depth, bool bwd) {
  const SplitPlan p = plan_split(m, e, depth);
  const int64_t cus = get_num_cus();
  const int64_t RA = p.r192 ? 192 : 256;
  const int64_t tiles = (m + RB - 1) / RB * ((e + RA - 1) / RA);
  const double step = LARGE_STEP_US[model_fmt(fmt)][bwd] * (p.r192 ? LARGE_192 : 1.0);
  if (p.S <= 1) return (double)((tiles + cus - 1) / cus) * (double)((depth + 63) / 64) * step + LARGE_US;
  return (double)p.spl * step + LARGE_SPLIT_MB * 4.0e-6 * (double)p.S * (double)m * (double)e + LARGE_SPLIT_US;
}

// stages per range (whole rounds) for S ranges of a depth, and the ranges
// that gives
int mid_spl(int64_t depth, int v, int S) {
  const int64_t nst = ((depth + 63) / 64 + MID_SD[v] - 1) / MID_SD[v];
  return (int)(((nst + S - 1) / S + MID_ROUND[v] - 1) / MID_ROUND[v] * MID_ROUND[v]);
}
int mid_ranges(int64_t depth, int v, int S) {
  const int64_t nst = ((depth + 63) / 64 + MID_SD[v] - 1) / MID_SD[v];
  const int spl = mid_spl(depth, v, S);
  return (int)((nst + spl - 1) / spl);
}

int64_t mid_tiles(int64_t m, int64_t e, int v) { return (m + MID_T[v] - 1) / MID_T[v] * ((e + MID_R[v] - 1) / MID_R[v]); }

// the product alone in S ranges; *tile: one tile's time
double mid_us(int fmt, int64_t m, int64_t e, int64_t depth, bool bwd, int v, int S, double* tile) {
  const int64_t cus = get_num_cus(), units = mid_tiles(m, e, v) * S;
  const int64_t n = (units + cus - 1) / cus;
  const double A = MID_A[model_fmt(fmt)][bwd][v], B = MID_B[model_fmt(fmt)][bwd][v], fix = MID_FIX[bwd][v];
  const double ranges = S > 1 ? RANGE_US[v] + RANGE_EACH_US[v] * S + RANGE_MB_US[v] * 8.0e-6 * (double)(units * MID_T[v] * MID_R[v]) : 0.0;
  if (is_w8(v)) {
    const int64_t nst = ((depth + 63) / 64 + MID_SD[v] - 1) / MID_SD[v];
    *tile = (double)(S > 1 ? mid_spl(depth, v, S) : nst) * (A + B * std::min(1.0, (double)units / (double)cus)) + fix;
    return (double)n * *tile + ranges;
  }
  const int64_t nb = S > 1 ? std::min<int64_t>((int64_t)mid_spl(depth, v, S) * MID_SD[v], (depth + 63) / 64)
                           : (depth + 63) / 64;
  *tile = (double)nb * (n > 1 ? B : A) + fix;
  return (double)nb * ((double)(n / 2) * B + (double)(n % 2) * A) + fix + MID_ROUND_US[v] * (double)((n + 1) / 2 - 1) +
         ranges;
}

// The LoRA factors formed beside a product, per plan: depth slices of the
// token-side factor, and (backward) the weight gradients' workgroups and
// their token slice, for lrq_gemm_mid.hip [0] and lrq_gemm_w8.hip [1].
struct Side {
  bool on = false;
  int64_t slices = 0;
  int64_t wgs[2] = {0, 0};
  double us[2][5] = {};  // a weight-gradient workgroup, per variant
  bool r32 = false;
};

Side side_work(int64_t m, int64_t e, int64_t depth, bool bwd, int rp) {
  Side s;
  s.on = true;
  s.r32 = rp > 16;
  s.slices = (m + 63) / 64 * ((depth + MID_FOLD_KT - 1) / MID_FOLD_KT);
  for (int w8 = 0; bwd && w8 < 2; ++w8) {
    const int lds = w8 ? W8_TN_LDS : MID_TN_LDS;
    const LoraPlan a = mid_tn_plan(m, depth, e, rp, lds), b = mid_tn_plan(m, e, depth, rp, lds);
    if (a.splits <= 0 || b.splits <= 0) continue;
    const int64_t na = a.tiles * a.splits, nb = b.tiles * b.splits;
    s.wgs[w8] = w8 ? (na + 1) / 2 + (nb + 1) / 2 : na + nb;
    const double per = (double)((m + std::min(a.splits, b.splits) - 1) / std::min(a.splits, b.splits)) / 128.0;
    for (int v = MID_64; v <= MID_64X128; ++v) s.us[w8][v] = (TN_US[v] + TN_TOKENS_US[v] * per) * (s.r32 ? TN_R32 : 1.0);
  }
  return s;
}

// a product's time `us` (tiles of `tile` us, `units` workgroups) with its
// factors in the launch: the factor slices' workgroups first, then the tiles,
// then the weight gradients', on the places (one or two a CU)
double fold_us(const Side& s, int v, int64_t units, int stages, double us, double tile) {
  const bool w8 = is_w8(v);
  const int64_t places = get_num_cus() * (w8 ? 1 : 2), rounds = (units + places - 1) / places * places;
  const int64_t first = w8 ? w8_fold_wgs(s.slices, units, stages) : (s.slices + 7) / 8 * 8;
  const int64_t turns = w8 ? ((s.slices + 1) / 2 + first - 1) / first : 1;
  const double late = (double)(units + first - rounds), lat = FOLD_LATE_US[v];
  us += FOLD_US[v] + (late <= 0 ? 0.0 : w8 ? lat : lat * std::min(1.0, late / (double)first));
  const int64_t wgs = s.wgs[w8];
  if (wgs == 0) return us;
  const double tau = s.us[w8][v];
  const double fit = std::floor(tile / tau);  // one after another beside a tile
  const double beside = units <= places && late <= 0
                            ? (double)(places - first - units) * fit + (double)first * std::floor(std::max(0.0, tile - lat * (double)turns) / tau)
                            : (double)(rounds - units) * fit;
  const double after = std::ceil(std::max(0.0, (double)wgs - beside) / (double)places) * tau;
  const double alone = rounds > units
                           ? std::max(0.0, lat * (double)turns + std::ceil((double)wgs / (double)(rounds - units)) * tau - tile)
                           : after;
  const double share = SHARE_US[s.r32][v] * std::min(1.0, (double)(units + first + wgs) / (double)places);
  return std::max(us + std::min(after, alone) + share, CHAIN_US[v] + tau);
}

struct Pick {
  GemmPlan p;
  double us;
};

// the best number of depth ranges for variant v, its partials and counters
// within the limits (forced: at least two where the depth has them). False
// if the launch cannot take the shape, or none takes less than `below`.
bool mid_best(int fmt, int64_t m, int64_t e, int64_t depth, bool bwd, int v, const Side& side, bool force_split, double below,
              int64_t max_floats, int64_t max_tiles, Pick* out) {
  // 32-bit buffer offsets of a tile's activation rows, outputs and weight rows
  if ((int64_t)128 * depth * 2 >= ((int64_t)1 << 31) || (int64_t)128 * e * 2 >= ((int64_t)1 << 31)) return false;
  if (max_floats < 0) return false;
  const int64_t tiles = mid_tiles(m, e, v), places = get_num_cus() * (is_w8(v) ? 1 : 2);
  bool found = false;
  for (int S = 1; S <= MID_MAXS[v]; ++S) {
    GemmPlan p;
    p.v = v;
    p.S = S;
    if (S > 1) {
      p.spl = mid_spl(depth, v, S);
      p.tiles = tiles;
      p.floats = S * tiles * MID_T[v] * MID_R[v];
      if (tiles > max_tiles || p.floats > max_floats || p.floats * 4 > (int64_t)LRQ_OOB) break;
      if (!force_split && tiles * S > places) break;
      if (mid_ranges(depth, v, S) != S) continue;  // (rounding turns it into fewer ranges, covered by those)
    }
    double tile = 0.0, us = mid_us(fmt, m, e, depth, bwd, v, S, &tile);
    const bool must = force_split && found && out->p.S == 1;
    if (us >= below && !must) continue;
    if (side.on) us = fold_us(side, v, tiles * S, S > 1 ? p.spl : (int)(((depth + 63) / 64 + MID_SD[v] - 1) / MID_SD[v]), us, tile);
    if (us >= below && !must) continue;
    *out = Pick{p, us};
    below = us;
    found = true;
  }
  return found;
}

// the variant that lrq_debug_gemm_path forces (MID_NONE: none), and whether
// with at least two depth ranges
int forced_variant(bool folded_bwd, bool* split) {
  static const int v[10] = {MID_NONE, MID_NONE, MID_64, MID_128, MID_64, MID_128, MID_256, MID_256, MID_64X128, MID_64X128};
  *split = g_gemm_path == 4 || g_gemm_path == 5 || g_gemm_path == 7 || g_gemm_path == 9;
  return g_gemm_path < 8 || folded_bwd ? v[g_gemm_path] : MID_NONE;
}

std::atomic<int64_t> g_plans{0};

template <bool BWD>
hipError_t dispatch(hipStream_t st, int fmt, const GemmPlan& p, const GemmArgs& a) {
  if (a.m == 0 || a.e == 0) return hipSuccess;
  if (p.v != MID_NONE) {
    if (p.S <= 1) return launch_mid(st, fmt, BWD, a, p.v);
    if (!a.part || !a.mcnt) return hipErrorInvalidValue;
    GemmArgs b = a;
    b.msplit = p.S;
    b.mspl = p.spl;
    return launch_mid(st, fmt, BWD, b, p.v);
  }
  if (p.S <= 1) return run_fmt<BWD, false>(st, fmt, p.r192, a);
  if (!a.part) return hipErrorInvalidValue;
  GemmArgs b = a;
  b.splits = p.S;
  b.spl = p.spl;
  hipError_t err = run_fmt<BWD, true>(st, fmt, p.r192, b);
  if (err != hipSuccess) return err;
  // forward fp8: channel scales (or the scalar) and the bias in the reduction
  const bool f8 = !BWD && fmt == LRQ_FMT_FP8;
  const int64_t quads = a.m * a.e / 4;
  hipLaunchKernelGGL(k_split_reduce, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, st, a.part, p.S, a.m, a.e,
                     f8 ? a.wscale : nullptr, a.per_channel, BWD ? nullptr : a.bias, a.out);
  return hipGetLastError();
}

}  // namespace

int g_num_cus_ = 256;  // compute units of the context's device (the persistent grid)
void set_num_cus(int n) { g_num_cus_ = n > 0 ? n : 256; }
int get_num_cus() { return g_num_cus_; }

bool gemm_plan(int fmt, int64_t m, int64_t e, int64_t depth, bool bwd, int64_t max_floats, GemmPlan* p) {
  *p = GemmPlan{};
  if (m <= 0 || e <= 0) return true;
  g_plans.fetch_add(1, std::memory_order_relaxed);
  const int64_t mg = (m + 63) / 64 * 64;
  bool split = false;
  const int fv = forced_variant(false, &split);
  Pick pick{GemmPlan{}, 1e30}, c;
  if (fv != MID_NONE && mid_best(fmt, mg, e, depth, bwd, fv, Side{}, split, 1e30, max_floats, SK_MAX_NB, &c)) {
    *p = c.p;
    return true;
  }
  const SplitPlan sp = plan_split(m, e, depth);
  const int64_t floats = sp.S > 1 ? (int64_t)sp.S * m * e : 0;
  const bool large = floats <= max_floats;
  if (large) {
    pick.p.r192 = sp.r192;
    pick.p.S = sp.S;
    pick.p.spl = sp.spl;
    pick.p.floats = floats;
    pick.us = large_us(fmt, mg, e, depth, bwd);
  }
  bool found = large;
  if (g_gemm_path == 0 || g_gemm_path >= 8)
    for (int v : {MID_64, MID_128, MID_256})
      if (mid_best(fmt, mg, e, depth, bwd, v, Side{}, false, pick.us, max_floats, SK_MAX_NB, &c)) {
        pick = c;
        found = true;
      }
  *p = pick.p;
  return found;
}

bool fold_plan(int fmt, int64_t m, int64_t e, int64_t depth, bool bwd, int rp, int64_t max_floats, bool always,
               GemmPlan* p) {
  *p = GemmPlan{};
  const int64_t G = (m + 63) / 64, mg = G * 64;
  if (m <= 0 || e <= 0 || g_gemm_path == 1) return false;
  // the groups' arrivals and flags have counters; the factor slices address
  // the activations [m][depth], and their partials, as one buffer each, with
  // 32-bit offsets, and a masked access (offset LRQ_OOB) must lie past its end
  if (2 * G > SK_MAX_NB || m * depth * 2 > (int64_t)LRQ_OOB ||
      (depth + MID_FOLD_KT - 1) / MID_FOLD_KT * mg * rp * 4 > (int64_t)LRQ_OOB)
    return false;
  g_plans.fetch_add(1, std::memory_order_relaxed);
  bool split = false;
  const int fv = forced_variant(bwd, &split);
  const Side side = side_work(mg, e, depth, bwd, rp);
  Pick pick{GemmPlan{}, 1e30}, c;
  if (fv == MID_NONE && !always) pick.us = large_us(fmt, mg, e, depth, bwd) + LARGE_SIDE_US[bwd];
  for (int v = MID_64; v <= MID_64X128; ++v) {
    if ((fv != MID_NONE && v != fv) || (v == MID_64X128 && !bwd)) continue;
    if (mid_best(fmt, mg, e, depth, bwd, v, side, split, pick.us, max_floats, SK_MAX_NB - 2 * G, &c)) pick = c;
  }
  *p = pick.p;
  return pick.p.v != MID_NONE;
}

int64_t plans_formed() { return g_plans.load(std::memory_order_relaxed); }

hipError_t launch_fwd(hipStream_t st, int fmt, const GemmPlan& p, const GemmArgs& a) { return dispatch<false>(st, fmt, p, a); }
hipError_t launch_bwd(hipStream_t st, int fmt, const GemmPlan& p, const GemmArgs& a) { return dispatch<true>(st, fmt, p, a); }
void set_gemm_path(int path) { g_gemm_path = path; }
