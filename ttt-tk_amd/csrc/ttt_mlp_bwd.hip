// Remat backward of the non-causal TTT-MLP layer for gfx950 (MI355X).
//
// Behaviour follows the upstream operator `ttt_backward` (kernel kernels/ttt_backward/ttt.cu:179-1443,
// mathematics kernels/ttt_backward/matching.py:57-342, group walk :539-663): for every checkpoint
// group, last to first, the forward is replayed from the checkpoint while the per-mini-batch
// activations are saved, then the group is walked backwards producing the ten output gradients.
//
// Mapping: workgroups of 8 wavefronts (two per SIMD, at most 256 registers each); one per (batch,
// head), or two or three where the device has CUs to spare - then one or two replay the checkpoint groups (taking
// turns) and one walks them backwards, a group or more behind; with fewer to spare than pairs those replay for all of them.  With more room: ttt_mlp_bwd_wide.hip, which takes the
// roles from here (others form grad_L_XK from what the walk hands them).  Wave v owns hidden columns [32v, 32v+32).  All [tokens x hidden] activations live in
// registers in the "Q" orientation (accumulator rows = hidden, lane = token), so per-token scalars
// (eta, dEta partial sums) are per-lane values.  An activation that is also needed with tokens as the
// contraction index is bounced once through a wave-private LDS tile (row store + transposing read).
//
// Waves v and v^4 form a pair.  A wave keeps the two token blocks of a Q tile in the order (r, 1-r),
// r = v / 4: of every product summed over the hidden dimension it keeps token block r and hands token
// block 1-r to its partner through LDS, which adds its own share; the LayerNorm lanes (8 per token,
// 8 tokens per wave) then add the four pair sums.  Every sum has a fixed order.
//
// State in registers:
//   replay : W1s [F x hid], W2s [hid x F] (fp32 accumulator tiles; where W2 is needed with F contracted, the bf16
//            terms of W2s are transposed through a wave-private LDS tile); b1, b2 in LDS
//   reverse: gW1s [F x hid], gW2s [hid x F] (running gradients) only; gb1, gb2 in LDS.  The weights
//            enter the reverse walk as ready-made bf16 MFMA operands: after every mini-batch the replay
//            stores the operand images of W1^T[shard] and W2[shard]^T, and the walk reads the image of
//            the state after and before the step (before the first step of a group: converted straight
//            from the fp32 checkpoint).
// The output branch (Out depends on the state after a step, nothing later depends on it) is taken
// backwards inside the replay, where that state is still in registers: the replay writes dXQ and
// leaves dL/dZ2_bar and the operands X2_bar^T, (dL/dZ1_bar)^T, so that the walk only accumulates their
// products into the running gradients.
// While a group is replayed by the workgroup that also walks, the running gradients are parked in the
// caller's W*_init_group scratch.
// Saved per mini-batch (caller's *_group scratch): Z1 as a bf16 register image (Z1_group); the operand
// images X2_bar^T (X2_bar_group) and (dL/dZ1_bar)^T (Z1_bar_group); the two weight operand images
// (X2_group: W1^T[shard], grad_l_wrt_Z1_group: W2[shard]^T); x_hat / grad_output of the fused LayerNorm
// loss, dl/dZ2 and dL/dZ2_bar (grad_x_hat_fused_group) as bf16 [tok][F] tiles; the fused std in fp32.
#include <type_traits>

#include "ttt_mlp_common.hpp"
#include "ttt_mlp_kernels.hpp"

namespace ttt {

// Zeros standing in for the old contents of an output tile (8 KiB) when the outputs are overwritten rather
// than added to: the load stays where it is in the instruction stream and is served by the L2.
__device__ __attribute__((aligned(256))) const uint4 zero_tile[512] = {};

constexpr int BW_NWAVE = 8;
constexpr int BW_THREADS = 64 * BW_NWAVE;
constexpr int BW_NS = HID / BW_NWAVE;     // hidden columns per wave: 32
constexpr int LDX = 68;                   // row stride (elements) of the shared [64][64] bf16 tiles
constexpr int LDH = 36;                   // row stride of wave-private [64][32 hid] bf16 tiles
constexpr int LDF = 68;                   // row stride of wave-private [32 hid][64 F] bf16 tiles
constexpr int LDR = 68;                   // row stride (floats) of a pair-sum region [32 tok][64 F]: 16-byte accesses of
                                          // 16 consecutive rows fall on 64 distinct banks
constexpr int RGN = 2304;                 // floats per pair-sum region

constexpr int SB_TILE = 64 * LDX * 2;     // 8704
constexpr int SB_XQ = 0;                  // reverse: XQ until the post-update stage is done, then (with SB_E2)
constexpr int SB_E2 = SB_XQ + SB_TILE;    //          the fp32 park of g_y ; replay: XQ and XV
constexpr int SB_XK = SB_E2 + SB_TILE;
constexpr int SB_GZ2 = SB_XK + SB_TILE;   // replay: G2 = -eta*dl/dZ2 ; reverse: raw dl/dZ2
constexpr int SB_A = SB_GZ2 + SB_TILE;    // reverse: gZ2_bar, later dZ2
static_assert(2 * SB_TILE >= CS * FD * 4, "g_y park does not fit");
static_assert(32 * XPAIR * 2 <= SB_TILE, "a tile of row pairs fits a tile slot");
constexpr int SB_P = SB_A + SB_TILE;      // 8 pair-sum regions (one per wave), fp32 [32][LDR]
constexpr int SB_REGION = RGN * 4;        // 9216: also two wave-private bf16 tiles
static_assert(32 * LDR <= RGN, "pair-sum rows do not fit their region");
constexpr int SB_WTILE = 64 * LDH * 2;    // 4608
static_assert(2 * SB_WTILE <= SB_REGION && 32 * LDF * 2 <= SB_WTILE, "private tiles do not fit a region");
constexpr int SB_BNC = SB_P + BW_NWAVE * SB_REGION;   // 8 wave-private bounce tiles [64][LDH]
constexpr int SB_B1 = SB_BNC + BW_NWAVE * SB_WTILE;   // b1 during a replay, 256 floats
constexpr int SB_B2 = SB_B1 + HID * 4;        // b2 during a replay, 64 floats
constexpr int SB_GB1 = SB_B2 + FD * 4;        // running gradient wrt b1
constexpr int SB_GB2 = SB_GB1 + HID * 4;      // running gradient wrt b2
constexpr int SB_GAM = SB_GB2 + FD * 4;       // ttt_norm_weight of this head
constexpr int SB_BET = SB_GAM + FD * 4;       // ttt_norm_bias of this head
constexpr int SB_ETA = SB_BET + FD * 4;
constexpr int SB_DETA = SB_ETA + CS * 4;                  // [8 waves][64 tokens] partial dEta sums
constexpr int SB_RED = SB_DETA + BW_NWAVE * CS * 4;       // [8 waves][2][64] norm-gradient accumulators
constexpr int SB_FLAG = SB_RED + BW_NWAVE * 2 * FD * 4;   // outcome of a wait on the other workgroup
constexpr int SM_BWD_BYTES = SB_FLAG + 16;
static_assert(SM_BWD_BYTES <= 160 * 1024, "LDS budget of one gfx950 CU exceeded");

#define WAVE_SYNC() TTT_WAVE_SYNC()
#define MFMA(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_bf16((a), (b), (c), 0, 0, 0)

// ------------------------------------------------------------------ register images in HBM
// A [64 tok x 32 hid] (or [64 F x 32 hid]) bf16 operand as 4 chunks of 8 bf16 per lane; chunk n of
// thread tid sits at (n*512 + tid)*16 bytes, so every load/store instruction of a wave moves 1 KiB.
// `img` = byte offset of the image inside the buffer, `t16` = 16 * tid.
constexpr unsigned IMG_BYTES = CS * HID * 2;          // 32 KiB
constexpr unsigned CHUNK_BYTES = BW_THREADS * 16;     // 8 KiB
constexpr unsigned TILE_BYTES = CS * FD * 2;          // one [64][64] bf16 tile in HBM: 8 KiB
TTT_DEV void chunk_store(gptr_t b, unsigned img, int n, unsigned t16, bf16x8 v) { g_st8h(b, t16, img + n * CHUNK_BYTES, v); }
// The replay's images: written once and read a checkpoint group later, with streaming stores and loads, so that they do not push out
// lines that are re-used.  With one workgroup per (batch, head) those are the walk's parks: since they take 64 KiB instead of 128,
// 2 MiB of an XCD's 4 MiB L2 with every CU busy, streaming everything else keeps them there (backward, ms, 384 x 512 33.5 -> 32.0,
// 200 x 100 3.68 -> 3.51; it gave nothing while they took the whole of it).
// CACHED: few pairs with one workgroup each, whose groups the memory-side cache holds until they are walked (below).
template <bool CACHED = false>
TTT_DEV void image_store(gptr_t b, unsigned img, int n, unsigned t16, bf16x8 v) {
  if constexpr (CACHED) chunk_store(b, img, n, t16, v);
  else g_st_stream<bf16x8>(b, t16, img + n * CHUNK_BYTES, v);
}
TTT_DEV bf16x8 image_load(gptr_t b, unsigned img, int n, unsigned t16) { return g_ld_stream<bf16x8>(b, t16, img + n * CHUNK_BYTES); }
TTT_DEV bf16x8 chunk_load(gptr_t b, unsigned img, int n, unsigned t16) { return g_ld8h(b, t16, img + n * CHUNK_BYTES); }

// fp32 accumulator tile <-> HBM in the caller's row-major layout.  `ld` = row length, (r0, c0) =
// origin of this wave's block (wave-uniform); accumulator rows are tensor rows.
template <int RB, int CB>
TTT_DEV void acc_load_rows(AccT<RB, CB>& a, gptr_t g, unsigned off, int ld, int r0, int c0, int c, int h) {
  const unsigned vo = (4 * h * ld + c) * 4;
#pragma unroll
  for (int rb = 0; rb < RB; rb++)
#pragma unroll
    for (int cb = 0; cb < CB; cb++)
#pragma unroll
      for (int i = 0; i < 16; i++)
        a.b[rb][cb][i] = g_ldf(g, vo, off + ((r0 + 32 * rb + 8 * (i >> 2) + (i & 3)) * ld + c0 + 32 * cb) * 4);
}
template <int RB, int CB>
TTT_DEV void acc_store_rows(const AccT<RB, CB>& a, gptr_t g, unsigned off, int ld, int r0, int c0, int c, int h) {
  const unsigned vo = (4 * h * ld + c) * 4;
#pragma unroll
  for (int rb = 0; rb < RB; rb++)
#pragma unroll
    for (int cb = 0; cb < CB; cb++)
#pragma unroll
      for (int i = 0; i < 16; i++)
        g_stf(g, vo, off + ((r0 + 32 * rb + 8 * (i >> 2) + (i & 3)) * ld + c0 + 32 * cb) * 4, a.b[rb][cb][i]);
}
// ------------------------------------------------------------------ LayerNorm-lane helpers
// A lane of a LayerNorm stage owns token `tok` and the 8 features f0 .. f0+7.
TTT_DEV void ln_load(float (&x)[8], const bf16* p) {      // p 8-byte aligned
  const bf16x4 a = *reinterpret_cast<const bf16x4*>(p), b = *reinterpret_cast<const bf16x4*>(p + 4);
#pragma unroll
  for (int e = 0; e < 4; e++) { x[e] = (float)a[e]; x[4 + e] = (float)b[e]; }
}
TTT_DEV void ln_store_h(bf16* p, bf16x8 v) {
  *reinterpret_cast<bf16x4*>(p) = __builtin_shufflevector(v, v, 0, 1, 2, 3);
  *reinterpret_cast<bf16x4*>(p + 4) = __builtin_shufflevector(v, v, 4, 5, 6, 7);
}
template <bool PAIRS = false>
TTT_DEV void ln_store(bf16* p, const float (&x)[8]) { ln_store_h(p, cvt8<PAIRS>(x)); }
// 8 features of this lane's token to a [tok][F] bf16 tile in HBM (16 bytes per lane), which is read a checkpoint group later.
template <bool CACHED, bool PAIRS>
TTT_DEV void ln_store_g(gptr_t b, unsigned voff, unsigned soff, const float (&x)[8]) {
  const bf16x8 v = cvt8<PAIRS>(x);
  if constexpr (CACHED) g_st8h(b, voff, soff, v);
  else g_st_stream<bf16x8>(b, voff, soff, v);
}
TTT_DEV void ln_cvt8(float (&x)[8], bf16x8 v) {
#pragma unroll
  for (int e = 0; e < 8; e++) x[e] = (float)v[e];
}
TTT_DEV void ln_load_f32(float (&x)[8], const float* p) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
  for (int e = 0; e < 4; e++) { x[e] = a[e]; x[4 + e] = b[e]; }
}
// Sum of the four pair sums of this lane's token / features.  `row` points at this token's row of the
// first pair's region; the regions of successive pairs are 2 regions apart.
TTT_DEV void ln_gather(float (&z)[8], const float* row) {
  f32x4 a = *reinterpret_cast<const f32x4*>(row), b = *reinterpret_cast<const f32x4*>(row + 4);
#pragma unroll
  for (int pp = 1; pp < 4; pp++) {
    a += *reinterpret_cast<const f32x4*>(row + pp * 2 * RGN);
    b += *reinterpret_cast<const f32x4*>(row + pp * 2 * RGN + 4);
  }
#pragma unroll
  for (int e = 0; e < 4; e++) { z[e] = a[e]; z[4 + e] = b[e]; }
}
TTT_DEV float sum8(const float (&x)[8]) {
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) s += x[e];
  return s;
}
TTT_DEV float dot8(const float (&x)[8], const float (&y)[8]) {
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) s = __builtin_fmaf(x[e], y[e], s);
  return s;
}
// z -> x_hat in place, returns 1/std; *std_out = std.
TTT_DEV float ln_normalize(float (&z)[8], float* std_out) {
  const float mu = oct_sum(sum8(z)) * (1.f / FD);
  float var = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) { z[e] -= mu; var = __builtin_fmaf(z[e], z[e], var); }
  const float v = oct_sum(var) * (1.f / FD) + LN_EPS;
  const float rstd = __builtin_amdgcn_rsqf(v);
#pragma unroll
  for (int e = 0; e < 8; e++) z[e] *= rstd;
  *std_out = v * rstd;  // sqrt(v)
  return rstd;
}
// acc[f0 + e] += sum over this wave's tokens of x[e]   (wave-private LDS vector).  The 8 tokens sit in the lanes
// that share lane % 8: lanes 8 apart inside a row of 16 (one rotation), then the four rows, two values per swap
// (row_pair_sum2, half_sum2): in the end row r of one register holds the total of x[r], of the other that of
// x[4 + r], and lanes 0..7 of every row add their two totals to the vector.
TTT_DEV void ln_token_sum_add(float* s_acc, const float (&x)[8], int lane, int f0) {
  float y[8];
#pragma unroll
  for (int e = 0; e < 8; e++)
    y[e] = x[e] + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x[e]), 0x128, 0xF, 0xF, false));  // row_ror:8
  const float lo = half_sum2(row_pair_sum2(y[0], y[1]), row_pair_sum2(y[2], y[3]));
  const float hi = half_sum2(row_pair_sum2(y[4], y[5]), row_pair_sum2(y[6], y[7]));
  if ((lane & 8) == 0) {
    float* d = s_acc + f0 + (lane >> 4);
    d[0] += lo;
    d[4] += hi;
  }
}

// 16-byte chunk staging of one [64][64] bf16 tile from HBM into an LDS tile with row stride LDX
// (rows are 8-byte aligned): thread tid moves chunk tid.
// The same into a tile of row pairs (XQ, XK, XV: the layout LDS-direct loads deliver).
TTT_DEV void lds_put16x(bf16* s_tile, int tid, u32x4 v) {
  uint2* d = reinterpret_cast<uint2*>(s_tile + xrow(tid >> 3) + (tid & 7) * 8);
  d[0] = make_uint2(v[0], v[1]);
  d[1] = make_uint2(v[2], v[3]);
}
TTT_DEV void lds_put16(bf16* s_tile, int tid, u32x4 v) {
  uint2* d = reinterpret_cast<uint2*>(s_tile + (tid >> 3) * LDX + (tid & 7) * 8);
  d[0] = make_uint2(v[0], v[1]);
  d[1] = make_uint2(v[2], v[3]);
}

// ---------------------------------------------------------------- just-in-time operand pieces
// Piece (free block fb, k-step s) of the chained operand of an accumulator tile.
template <int RB, int CB>
TTT_DEV bf16x8 piece_state(const AccT<RB, CB>& x, int fb, int s) { return pack8(x.b[s >> 1][fb], s & 1); }
// Chained operand of an accumulator tile written as an LDS tile stored [free index][contraction index].
template <int LD, int RB, int CB>
TTT_DEV void store_state_rows(bf16* tile, const AccT<RB, CB>& x, int c, int h) {
#pragma unroll
  for (int fb = 0; fb < CB; fb++)
#pragma unroll
    for (int s = 0; s < 2 * RB; s++) store_piece_rows<LD>(tile, fb, s, c, h, piece_state(x, fb, s));
}
// s_vec[row] += sum over the 64-long contraction of the 32-row operand whose pieces fa(s) yields; the
// sum is formed on the matrix cores, lanes with c == 0 fold it into the LDS vector.
template <class FA>
TTT_DEV void lds_rowsum_add_jit(float* s_vec, FA fa, bf16x8 ones, int c, int h) {
  f32x16 t;
#pragma unroll
  for (int i = 0; i < 16; i++) t[i] = 0.f;
#pragma unroll
  for (int s = 0; s < 4; s++) t = MFMA(fa(s), ones, t);
  if (c == 0) {
#pragma unroll
    for (int g = 0; g < 4; g++) {
      f32x4* q = reinterpret_cast<f32x4*>(s_vec + 8 * g + 4 * h);
      f32x4 v = *q;
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] += t[4 * g + e];
      *q = v;
    }
  }
  // Other lanes of this wave read the vector next; without a fence the compiler may forward the
  // values each lane saw before the update.
  WAVE_SYNC();
}
// C-init of the rows of a Q-orientation tile from an LDS vector indexed by accumulator row (32 floats).
template <int CB>
TTT_DEV void acc_init_rows_lds(AccT<1, CB>& a, const float* s_vec, int h) {
#pragma unroll
  for (int g = 0; g < 4; g++) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(s_vec + 8 * g + 4 * h);
#pragma unroll
    for (int cb = 0; cb < CB; cb++)
#pragma unroll
      for (int e = 0; e < 4; e++) a.b[0][cb][4 * g + e] = v[e];
  }
}

TTT_DEV bf16x8 cvt8(const f32x4 lo, const f32x4 hi) {
  const float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return cvt8(x);
}
// Piece (kappa order) straight from a row-major fp32 matrix in HBM: lane = row row0 + c, contraction =
// columns col0 + 16 s ...; row0, col0, s wave-uniform.
TTT_DEV bf16x8 piece_from_f32(gptr_t g, unsigned off, int ld, int row0, int col0, int s, int c, int h) {
  const unsigned vo = (c * ld + 4 * h) * 4, so = off + (row0 * ld + col0 + 16 * s) * 4;
  return cvt8(g_ld4f(g, vo, so), g_ld4f(g, vo, so + 32));
}

// gelu, gelu', gelu'' of eight bf16 values, rounded to bf16.
template <bool PAIRS>
TTT_DEV void gelu_images(const bf16x8 z, bf16x8& g, bf16x8& a, bf16x8& b) {
#pragma unroll
  for (int jj = 0; jj < 8; jj += 2) {
    float g2[2], a2[2], b2[2];
#pragma unroll
    for (int q = 0; q < 2; q++) gelu_fdd((float)z[jj + q], g2[q], a2[q], b2[q]);
    put_cvt<PAIRS>(g, jj, g2[0], g2[1]);
    put_cvt<PAIRS>(a, jj, a2[0], a2[1]);
    put_cvt<PAIRS>(b, jj, b2[0], b2[1]);
  }
}

// Pair sum of a product z (rows F, column block 0 = the token block this wave keeps, column block 1 =
// the one it hands over): leaves the pair sum of the kept block in the PARTNER's region, stored
// [tok in block][F].  Contains two workgroup barriers; the caller makes sure that this wave's own
// reads of its region (the private tiles T1 / T2) are complete.
TTT_DEV void pair_sum(float* own, float* partner, const AccT<2, 2>& z, int c, int h) {
#pragma unroll
  for (int rb = 0; rb < 2; rb++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const f32x16& x = z.b[rb][1];
      f32x4 v = {x[4 * g], x[4 * g + 1], x[4 * g + 2], x[4 * g + 3]};
      *reinterpret_cast<f32x4*>(own + c * LDR + 32 * rb + 8 * g + 4 * h) = v;
    }
  __syncthreads();
#pragma unroll
  for (int rb = 0; rb < 2; rb++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      float* q = partner + c * LDR + 32 * rb + 8 * g + 4 * h;
      const f32x16& x = z.b[rb][0];
      f32x4 v = *reinterpret_cast<const f32x4*>(q);
      v[0] += x[4 * g]; v[1] += x[4 * g + 1]; v[2] += x[4 * g + 2]; v[3] += x[4 * g + 3];
      *reinterpret_cast<f32x4*>(q) = v;
    }
  __syncthreads();
}

// Three [64][64] bf16 tiles + the eta vector of one mini-batch in flight from HBM (per thread).
struct Staged3 {
  u32x4 a, b, c;
  bf16 eta;
};
// `mb` = mini-batch index inside this (batch, head); t16 = 16 * tid.
TTT_DEV void stage3_load(Staged3& s, gptr_t ga, gptr_t gb, gptr_t gc, gptr_t geta, int mb, int tid, unsigned t16) {
  s.a = g_ld_stream<u32x4>(ga, t16, mb * TILE_BYTES);
  s.b = g_ld_stream<u32x4>(gb, t16, mb * TILE_BYTES);
  s.c = g_ld_stream<u32x4>(gc, t16, mb * TILE_BYTES);
  s.eta = g_ldh(geta, 2 * (tid & (CS - 1)), mb * (CS * 2));   // in bounds for every thread; threads >= CS drop it
}
TTT_DEV void stage3_store(const Staged3& s, bf16* sa, bf16* sb, bf16* sc, bf16* s_eta, int tid) {
  lds_put16x(sa, tid, s.a);
  lds_put16x(sb, tid, s.b);
  lds_put16x(sc, tid, s.c);
  if (tid < CS) s_eta[tid] = s.eta;   // the replay keeps eta as bf16 in LDS
}

// Piece s of W2[shard] before mini-batch j of the group as an operand (lane = hid row, contraction =
// F): the image the replay stored after mini-batch j-1, or straight from the fp32 checkpoint.
// STREAM: the only read of the image on this CU, so it need not stay in the L2.
template <bool STREAM = false>
TTT_DEV bf16x8 w2_before(gptr_t img, gptr_t ck, unsigned ck_off, int j, int s, int hid0, int c, int h, unsigned t16) {
  // the image offset is clamped so that the load stays inside the buffer even if it is hoisted above the branch
  bf16x8 r = STREAM ? image_load(img, (j > 0 ? j - 1 : 0) * IMG_BYTES, s, t16) : chunk_load(img, (j > 0 ? j - 1 : 0) * IMG_BYTES, s, t16);
  if (j == 0) r = piece_from_f32(ck, ck_off, FD, hid0, 0, s, c, h);
  return r;
}
// Piece (row block rb, k-step s) of W1[:, shard]^T before mini-batch j (lane = F row, contraction = hid).
TTT_DEV bf16x8 w1_before(gptr_t img, gptr_t ck, unsigned ck_off, int j, int rb, int s, int hid0, int c, int h, unsigned t16) {
  bf16x8 r = image_load(img, (j > 0 ? j - 1 : 0) * IMG_BYTES, 2 * rb + s, t16);
  if (j == 0) r = piece_from_f32(ck, ck_off, HID, 32 * rb, hid0, s, c, h);
  return r;
}

constexpr int FIN_CHUNK = 8;   // mini-batches per hand-over to the grad_L_XK workgroup within the last group walked (a power of two)

// What a set's word has come to when group number `done` has been replayed into it, in all of its parts.
TTT_DEV int parts_until(const BwdParams& p, int done) {
  const int use = uni(done / p.n_sets);   // (only the first use of a set can be in parts)
  return use + (done - use * p.n_sets < p.n_shared ? p.n_parts : 1);
}

// ------------------------------------------------------------------ one workgroup per (batch, head), and helpers
// Between half and all of the CUs' number of pairs a workgroup each leaves CUs idle, and a second workgroup for each does not fit.  The idle ones
// replay checkpoint groups for whoever has most to do: one is free to take a group as soon as one of the pair's sets
// beyond the caller's is free, and writes it into that set; the pair's own workgroup, when it comes to a group, walks it from the set
// if it is taken and replays it itself if it is not.  Who takes what depends on the timing, the results do not.  A
// workgroup waits only for a group that a running one has taken, so nothing has to be resident at once.
constexpr int HELP_ONE = 24, HELP_TWO = 44;   // first bits of what is taken into sets 1 and 2
// The pair's workgroup comes to group number `done`: the set it is (being) replayed into, or 0.  Its sets of the group before
// are free again: every wave has what it read of them.
TTT_DEV int take_group(int* word, int done, int* s_flag, bool first_lane) {
  __syncthreads();
  if (first_lane) {
    uint64_t* const w = reinterpret_cast<uint64_t*>(word);
    uint64_t old = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), to;
    int set;
    do {
      uint64_t one = (old >> HELP_ONE) & 0xfffff, two = old >> HELP_TWO;
      const uint64_t here = done + 1;
      set = one == here ? 1 : two == here ? 2 : 0;
      if (one < here) one = 0;
      if (two < here) two = 0;
      to = (two << HELP_TWO) | (one << HELP_ONE) | (2 * (uint64_t)done + (set > 0 ? 1 : 0));
    } while (!__hip_atomic_compare_exchange_strong(w, &old, to, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    *s_flag = set;
  }
  __syncthreads();
  return uni(*s_flag);
}
// A helper takes a group: job[0] = pair (of the launch), job[1] = number of the group, job[2] = set; false: there is none left to
// take (or a wait gave up, or nothing came free for as long as one may wait: nobody waits for this workgroup).
// Taken is the group that the pair will come to next once this one could be ready: the one behind those taken already, else the
// next one while the pair replays, the one behind that while it walks.  With many helpers (up to 146 pairs on 256 CUs) also the next one while it
// walks: a helper is there as soon as the walk frees a set, and the pair waits for less than it would replay (in ms, 136 pairs x 512
// 14.77 -> 13.66, 144 x 512 15.1 -> 14.5).
TTT_DEV bool help_take(const BwdParams& p, int me, int* job) {
  const int lane = threadIdx.x & 63;
  const bool many = 4 * p.n_helpers >= 3 * p.nbh;
  __syncthreads();   // the last job has been read by every wave
  if (threadIdx.x < 64) {
    int* const words = p.sync + (size_t)p.bh0 * BWD_SYNC_STRIDE + BWD_HELP;
    const uint64_t t0 = wall_clock64();
    int took = 0;
    for (bool more = true; more;) {
      // what is left to do of a pair, in halves of a group: its replay is one, its walk the other
      int most = -1, pair = 0, group = 0, set = 0;
      uint64_t seen = 0;
      bool open = false;
      for (int i = lane; i < p.nbh; i += 64) {
        const int q = i + me < p.nbh ? i + me : i + me - p.nbh;   // (not all helpers the same one)
        const uint64_t w = __hip_atomic_load(reinterpret_cast<uint64_t*>(words + (size_t)q * BWD_SYNC_STRIDE), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int at = static_cast<int>(w & 0xffffff), done = at >> 1, walks = at & 1;
        const int one = static_cast<int>((w >> HELP_ONE) & 0xfffff), two = static_cast<int>(w >> HELP_TWO), last = max(one, two);
        const int ahead = (one > done + 1) + (two > done + 1);
        const int next = ahead > 0 ? last : min(done + 1 + (many ? 0 : walks), max(p.K - 1, done + 1));
        if (next >= p.K) continue;
        open = true;
        const int s = one == 0 ? 1 : two == 0 && p.n_sets > 2 ? 2 : 0;
        const int left = 2 * (p.K - done) - walks - ahead;
        if (s > 0 && left > most) { most = left; pair = q; group = next; set = s; seen = w; }
      }
      if (!__any(open)) break;
      int key = most < 0 ? -1 : most * 64 + 63 - lane, best = key;
#pragma unroll
      for (int d = 1; d < 64; d *= 2) best = max(best, __shfl_xor(best, d, 64));
      if (best < 0) {
        more = __hip_atomic_load(p.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0 && wall_clock64() - t0 <= p.wait_limit;
        __builtin_amdgcn_s_sleep(64);
        continue;
      }
      bool mine = false;
      if (key == best) {
        const uint64_t to = seen | ((uint64_t)(group + 1) << (set == 1 ? HELP_ONE : HELP_TWO));
        mine = __hip_atomic_compare_exchange_strong(reinterpret_cast<uint64_t*>(words + (size_t)pair * BWD_SYNC_STRIDE), &seen, to,
                                                    __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (mine) {
          job[0] = pair;
          job[1] = group;
          job[2] = set;
        }
      }
      if (__any(mine)) {
        took = 1;
        break;
      }
    }
    if (lane == 0) job[3] = took;
  }
  __syncthreads();
  return uni(job[3]) != 0;
}

// ------------------------------------------------------------------ several workgroups per (batch, head)
// The replay of a checkpoint group needs only the checkpoint, so it can run ahead of the reverse walk
// on other CUs: one or more workgroups replay group after group, in turn, into alternating sets of the per-group
// tensors, another walks each group backwards as soon as it is complete.  They signal through
// counters in HBM (agent scope); all are resident at once because the launcher uses this mode only
// when the grid fits the CUs of the device.  A wait that sees no progress for p.wait_limit ticks of the
// 100 MHz clock raises the status word and all of them leave, so every wave always exits.
// ROLE 0: replay and reverse walk of every group in one workgroup; 1: one replay (k_hi = k_lo); 2: the reverse walks only.
// IMG (two replaying workgroups per pair and the walk on one CU): the replay has time to spare and evaluates gelu,
// gelu', gelu'' of the rounded Z1 for the walk, which gets them as three images instead of the image of Z1.  Same values
// either way.
// FIN: grad_L_XK is a leaf of the walk - it needs the running gradients, but nothing needs it.  Where one more workgroup
// fits, the walk hands it dZ1 (a register image) and two fp32 tiles, g_y and the norm-weight gradient terms, and that
// workgroup (bwd_finish_dxk) forms grad_L_XK, grad_L_XV and the norm gradients.
// WIDE: the walk runs on two workgroups (ttt_mlp_bwd_wide.hip), which say separately how far they are.
// PARTS: several workgroups at once replay each of the p.n_shared groups walked first, a stretch of its mini-batches each.
// HELPED: a workgroup that replays and walks (ROLE 0) where others (ROLE 1) replay groups ahead of it.
// EIGHTHS: a replay hands over its norm-gradient sums by eighths of the group (eighth_done); needed with PARTS.
template <int ROLE, bool IMG, bool FIN, bool WIDE = false, bool PARTS = false, bool HELPED = false, bool EIGHTHS = PARTS, bool CACHED = false>
// k_hi, k_lo: the checkpoint groups k_hi, k_hi - 1, .. k_lo of the sequence (ROLE 0: a segment; ROLE 2: K - 1 .. 0).
// part (PARTS): which of the p.n_parts stretches of the group's mini-batches this workgroup replays; it takes the state there from
// the checkpoint itself, through the state-carrying half of the mini-batches before (`light`).  HELPED: the set it is replayed into.
// False: a wait gave up.
TTT_DEV bool bwd_body(const BwdParams& p, unsigned char* smem, const int bh, const int k_hi, const int k_lo, const int part = 0) {
  constexpr bool PAIRS = ROLE == 0;
  static_assert(!(ROLE == 0 && (IMG || FIN)), "one workgroup per (batch, head) does everything itself");
  bf16* s_xq = reinterpret_cast<bf16*>(smem + SB_XQ);
  bf16* s_xk = reinterpret_cast<bf16*>(smem + SB_XK);
  bf16* s_gz2 = reinterpret_cast<bf16*>(smem + SB_GZ2);
  bf16* s_e2 = reinterpret_cast<bf16*>(smem + SB_E2);
  bf16* s_a = reinterpret_cast<bf16*>(smem + SB_A);
  float* s_P = reinterpret_cast<float*>(smem + SB_P);
  float* s_b1 = reinterpret_cast<float*>(smem + SB_B1);     // replay: b1
  float* s_b2 = reinterpret_cast<float*>(smem + SB_B2);     // replay: b2
  float* s_gb1 = reinterpret_cast<float*>(smem + SB_GB1);   // running gradient wrt b1
  float* s_gb2 = reinterpret_cast<float*>(smem + SB_GB2);   // running gradient wrt b2
  float* s_gam = reinterpret_cast<float*>(smem + SB_GAM);
  float* s_bet = reinterpret_cast<float*>(smem + SB_BET);
  float* s_eta = reinterpret_cast<float*>(smem + SB_ETA);
  bf16* s_etah = reinterpret_cast<bf16*>(smem + SB_ETA);     // the replay's view: eta as it sits in HBM
  float* s_deta = reinterpret_cast<float*>(smem + SB_DETA);
  float* s_red = reinterpret_cast<float*>(smem + SB_RED);

  int tid0 = threadIdx.x;
  if constexpr (HELPED) asm volatile("" : "+v"(tid0));   // (what a helper and a pair's own workgroup derive from it is not to be shared)
  const int tid = tid0, lane = tid & 63, h = lane >> 5, c = lane & 31;
  const int v = __builtin_amdgcn_readfirstlane(tid >> 6);        // wave index, in a scalar register
  const int pp = v & 3, r = v >> 2;                              // pair, index inside the pair
  const int tb[2] = {r, 1 - r};                                  // token block held in column block 0 / 1 of a Q tile
  const int q8 = lane >> 3, tok = 8 * v + q8, f0 = 8 * (lane & 7);   // LayerNorm ownership (token block r)
  const int head = bh % p.NH;
  const int hid0 = BW_NS * v;
  float* s_own = s_P + (pp * 2 + r) * RGN;
  float* s_partner = s_P + (pp * 2 + (1 - r)) * RGN;
  // the pair sums of token block r sit in region 1-r of every pair
  const float* s_lnrow = s_P + (1 - r) * RGN + (tok & 31) * LDR + f0;
  bf16* const T0 = reinterpret_cast<bf16*>(smem + SB_BNC) + v * (64 * LDH);   // wave-private tiles: T0 = the bounce
  bf16* const T1 = reinterpret_cast<bf16*>(s_own);                            // tile; T1, T2 = the two halves of
  bf16* const T2 = T1 + 64 * LDH;                                             // this wave's pair-sum region
  float* s_b1w = s_b1 + hid0;
  float* s_gb1w = s_gb1 + hid0;
  const int cgs = p.cgs;
  // a segment that is not the first to run continues where the one before it stopped; one that is not the last leaves
  // what the next one needs instead of the norm gradients
  const bool seg_first = k_hi == p.K - 1, seg_last = k_lo == 0;

  if (tid < FD) {
    s_gam[tid] = p.ttt_norm_weight[head * FD + tid];
    s_bet[tid] = p.ttt_norm_bias[head * FD + tid];
    if (ROLE != 1) s_gb2[tid] = (seg_first ? p.grad_L_b2_last : p.grad_L_b2_init)[(size_t)bh * FD + tid];
  }
  if (ROLE != 1 && tid < HID) s_gb1[tid] = (seg_first ? p.grad_L_b1_last : p.grad_L_b1_init)[(size_t)bh * HID + tid];
  // Norm-weight / norm-bias gradients accumulate per wave in LDS (summed over the wave's 8 tokens
  // with cross-lane adds in a fixed order); summed over the waves at the end.  The replay and the
  // reverse walk each contribute, and their sums are kept apart (so that the result does not depend on
  // whether one workgroup does both): with one workgroup the sum that is not being added to waits in HBM.
  float* s_dgw = s_red + (v * 2 + 0) * FD;
  float* s_dbw = s_red + (v * 2 + 1) * FD;
  if (lane < FD) { s_dgw[lane] = 0.f; s_dbw[lane] = 0.f; }
  float* s_gy = reinterpret_cast<float*>(smem + SB_XQ) + tok * FD + f0;   // this lane's part of the g_y park
  bf16x8 ones;
#pragma unroll
  for (int j = 0; j < 8; j++) ones[j] = (bf16)1.0f;

  // Buffers: base = this (batch, head)'s part of each tensor; offsets inside stay below 2 GiB (checked
  // by the launcher).  Per-lane offsets: t16 = chunk / tile staging, vln = this LayerNorm lane's 8
  // features of its token in a [tok][F] bf16 tile, vtok = its token in a [tok] fp32 vector.
  // Element offsets of this (batch, head) inside each class of tensor.  A buffer descriptor is built
  // where it is used, from the kernel argument and one of these offsets; the offsets are made opaque
  // to the optimiser once per mini-batch (REFRESH_OFFSETS) so that the thirty descriptors are not all
  // hoisted out of the loops and kept in scalar registers at once.
  size_t ox = uni64((size_t)bh * p.NC * (CS * FD));     // [NC][64][64] inputs / outputs
  size_t oe = uni64((size_t)bh * p.NC * CS);            // [NC][64] eta, d eta
  size_t of = uni64((size_t)bh * cgs * (CS * FD));      // [cgs][64][64] scratch tiles
  size_t oh = uni64((size_t)bh * cgs * (CS * HID));     // [cgs][64][256] scratch tiles (register images)
  size_t ot = uni64((size_t)bh * cgs * CS);             // [cgs][64] scratch vectors
  size_t opk = uni64((size_t)bh * cgs * (FD * HID));    // W1_init_group / W2_init_group
  size_t ock = uni64((size_t)bh * p.K * (FD * HID));    // W1 / W2 checkpoints
  // The tensor pointers are read from the kernel-argument segment (scalar loads) where they are used,
  // through a pointer that is refreshed with the offsets, instead of all fifty living in scalar registers.
  typedef const __attribute__((address_space(4))) BwdParams* KernArgs;
  KernArgs ka = (KernArgs)__builtin_amdgcn_kernarg_segment_ptr();
#define REFRESH_OFFSETS()                                                                                                       \
  asm volatile("" : "+s"(ka), "+s"(ox), "+s"(oe), "+s"(of), "+s"(oh), "+s"(ot), "+s"(opk), "+s"(ock));                          \
  if constexpr (HELPED) asm volatile("" : "+s"(kg))
  // per-group tensors: the caller's (set 0) or, with several workgroups, one of the alternate sets
// (with helpers through a pointer to the set's: choosing between the two at every use costs the workgroup that does everything 3 %)
  typedef const __attribute__((address_space(4))) BwdSet* KernSets;
  KernSets kg = nullptr;
#define GRP(name) (HELPED ? kg->name : ROLE != 0 && set ? ka->alt_##name[ROLE != 0 && set ? set - 1 : 0] : ka->name)
#define bXQ gbuf(ka->XQ + ox)
#define bXK gbuf(ka->XK + ox)
#define bXV gbuf(ka->XV + ox)
#define bGO gbuf(ka->grad_L_XQW + ox)
#define bETA gbuf(ka->last_eta + oe)
#define bZ1 gbuf(GRP(Z1_group) + oh)
#define bGZ1B gbuf(GRP(Z1_bar_group) + oh)              // operand image of gZ1_bar = dL/dZ1_bar
#define bX2B gbuf(GRP(X2_bar_group) + oh)               // operand image of X2_bar
#define bGZB gbuf(GRP(grad_x_hat_fused_group) + of)     // gZ2_bar = dL/dZ2_bar, [tok][F] tiles
#define bIMG1 gbuf(GRP(X2_group) + oh)
#define bIMG2 gbuf(GRP(grad_l_wrt_Z1_group) + oh)
#define bXHF gbuf(GRP(x_hat_fused_group) + of)
#define bGOF gbuf(GRP(grad_output_fused_group) + of)
#define bGZ2 gbuf(GRP(grad_l_wrt_Z2_group) + of)
#define bSDF gbuf(GRP(std_fused_group) + ot)
  // While a group is replayed the running gradients are parked in W*_init_group; during the reverse
  // walk the same two 64 KiB slots park what must survive the LayerNorm stage (block 0's half of three 32 KiB images).
  // Several workgroups per (batch, head): slot j of W1_init_group (of the set) carries gelu'(Z1) and gelu''(Z1)
  // of mini-batch j as two register images, and Z1_group carries gelu(Z1) instead of Z1.
#define bDD gbuf(GRP(W1_init_group) + opk)
  // the walk's fourth parked image (-eta * (XK gW1 + gb1) * gelu'(Z1)): second half of slot 0 of W1_init_group,
  // or - where that tensor carries GELU images - the workspace
#define bPUH (ROLE == 0 ? gbuf(ka->W1_init_group + opk) + IMG_BYTES : gbuf(ka->walk_park + (size_t)bh * (CS * HID)))
#define bPW1 gbuf(ka->W1_init_group + opk)
#define bPW2 gbuf(ka->W2_init_group + opk)
  constexpr unsigned PARK_D1 = 0, PARK_T2 = IMG_BYTES, PARK_G1 = 0;   // d1 in bPW1 (one workgroup only); g1, t2 in bPW2
#define bCW1 gbuf(ka->W1_ck + ock)
#define bCW2 gbuf(ka->W2_ck + ock)
#define bDXQ gbuf(ka->grad_L_XQ + ox)
#define bDXK gbuf(ka->grad_L_XK + ox)
#define bDXV gbuf(ka->grad_L_XV + ox)
#define bDETA gbuf(ka->grad_L_last_eta + oe)
// what an accumulating output held before: the tile itself, or zeros when the outputs are overwritten
#define OLD_VALUE(buf, off) (ka->overwrite ? gbuf(zero_tile) : (buf)), vln, (ka->overwrite ? 0u : (off))
  const unsigned t16 = 16 * tid, vln = (tok * FD + f0) * 2, vtok = 4 * tok;
  // Everything derived from the lane index is cheap to recompute and expensive to keep: a value
  // computed once before the loops is held in a register (or spilled and reloaded) for the whole
  // kernel.  LANE_VARS re-derives the lot from a lane index the optimiser cannot see through, so
  // each stage that opens with it gets fresh, short-lived copies.
  int lane_v = lane;
#define LANE_VARS                                                                                       \
  asm volatile("" : "+v"(lane_v));                                                                      \
  const int lane = lane_v, h = lane >> 5, c = lane & 31, tid = (v << 6) | lane;                         \
  const int q8 = lane >> 3, tok = 8 * v + q8, f0 = 8 * (lane & 7);                                      \
  const unsigned t16 = 16 * tid, vln = (tok * FD + f0) * 2, vtok = 4 * tok;                             \
  const float* s_lnrow = s_P + (1 - r) * RGN + (tok & 31) * LDR + f0;                            \
  float* s_gy = reinterpret_cast<float*>(smem + SB_XQ) + tok * FD + f0;                                 \
  (void)h; (void)c; (void)tid; (void)q8; (void)t16; (void)vln; (void)vtok; (void)s_lnrow; (void)s_gy

  // running gradients wrt the state after the last mini-batch
  AccT<2, 1> gW1s;
  AccT<1, 2> gW2s;
  if constexpr (ROLE != 1) {
    acc_load_rows(gW1s, gbuf((seg_first ? p.grad_L_W1_last : p.grad_L_W1_init) + (size_t)bh * FD * HID), 0, HID, 0, hid0, c, h);
    acc_load_rows(gW2s, gbuf((seg_first ? p.grad_L_W2_last : p.grad_L_W2_init) + (size_t)bh * HID * FD), 0, FD, hid0, 0, c, h);
  }
  int* const w_sync = p.sync + (size_t)bh * BWD_SYNC_STRIDE;   // + s: the group last replayed into set s
  int* const w_walked = w_sync + (WIDE ? BWW_WALKED : 16);
  int* const w_finished = w_sync + 24;
  const int n_sets = ROLE == 0 ? 1 : p.n_sets;
  int* const w_status = p.status;
  int* const s_flag = reinterpret_cast<int*>(smem + SB_FLAG);

  // The replay's share of the norm gradients is formed by eighths of a group, which are summed, and added group by group to a
  // running sum, in that order, so it does not depend on who replays what.  The running sum sits in HBM (slot 0 of the park, 4 KiB): with one workgroup per
  // (batch, head) in the caller's x_hat_ln_group, where the walk's sum waits behind it (slot 1) while the LDS accumulators
  // serve a replay, otherwise in the workspace, added to by the walk (by the grad_L_XK workgroup where there is one).
  // (Its address is formed where it is used: kept over the loop it costs the walk two registers it does not have.)
  auto park = [&]() {
    size_t o = uni64(ROLE == 0 ? (size_t)bh * cgs * (CS * FD) : (size_t)bh * (BW_NWAVE * 2 * FD));
    asm volatile("" : "+s"(o));
    return ROLE == 0 ? gbuf(p.x_hat_ln_group + o) : gbuf(p.norm_park + o);
  };
  // (also formed where it is used) this lane's two words of the wave's accumulators: +0, +FD*4
  auto np_off = [&]() {
    LANE_VARS;
    return (v * 2 * FD + lane) * 4u;
  };
  const int eighth = (cgs + 7) / 8;   // mini-batches
  auto group_sums = [&](int set, int e) {   // of this wave
    size_t o = uni64((((size_t)bh * BWD_MAX_SETS + set) * 8 + e) * (BW_NWAVE * 2 * FD) + v * 2 * FD);
    asm volatile("" : "+s"(o));
    return gbuf(p.norm_partial + o);
  };
  constexpr unsigned PARK_BYTES = BW_NWAVE * 2 * FD * 4;
  if (ROLE == 0 ? seg_first : (ROLE == 2 && !FIN)) {   // the running sum starts at zero
    const gptr_t g = park();
    g_stf(g, (v * 2 * FD + lane) * 4, 0, 0.f);
    g_stf(g, (v * 2 * FD + lane) * 4, FD * 4, 0.f);
  }
  if (ROLE == 0 && !seg_first) {   // the walk's sum as the segment before this one left it
    s_dgw[lane] = g_ldf(park(), np_off(), PARK_BYTES);
    s_dbw[lane] = g_ldf(park(), np_off(), PARK_BYTES + FD * 4);
  }

  TTT_STAGES_BEGIN();
  for (int kk = k_hi; kk >= k_lo; kk--) {
    int k = kk;
    if constexpr (HELPED) asm volatile("" : "+s"(k));   // (no offsets that run with k in vector registers)
    const int n_mb = min(cgs, p.NC - k * cgs);
    const int done = p.K - 1 - k;                    // number of this group, counted from the end of the sequence
    const int in_set = HELPED ? (ROLE == 1 ? part : take_group(w_sync + BWD_HELP, done, s_flag, v == 0 && lane_v == 0)) : ROLE == 0 ? 0 : done % n_sets;
    int* const w_replayed = w_sync + in_set;
    if constexpr (HELPED) kg = (KernSets)((const __attribute__((address_space(4))) char*)ka + offsetof(BwdParams, help_sets)) + in_set;
    REFRESH_OFFSETS();
    const size_t slot = (size_t)bh * p.K + k;
    const unsigned ckW = static_cast<unsigned>(k) * (FD * HID * 4u);   // byte offset of this group's checkpoint in bCW1 / bCW2
    // ================================================================= replay
    if constexpr (ROLE != 2)
    if (ROLE == 1 || !HELPED || in_set == 0) {
      const int set = ROLE == 0 ? 0 : in_set;
      if constexpr (ROLE == 1 && !HELPED) {   // the set is free once the reverse walk is done with the group that used it last
        if (done >= n_sets && !wait_at_least(w_walked, done - n_sets + 1, w_status, s_flag, p.wait_limit)) return false;
        if (WIDE && done >= n_sets && !wait_at_least(w_walked + 4, done - n_sets + 1, w_status, s_flag, p.wait_limit)) return false;
        if constexpr (FIN) {   // ... and so is the workgroup that reads the before-state images for grad_L_XK
          if (done >= n_sets && !wait_at_least(w_finished, done - n_sets + 1, w_status, s_flag, p.wait_limit)) return false;
        }
      }
      if constexpr (ROLE == 1) {
        WAVE_SYNC();
        s_dgw[lane] = 0.f;   // (every lane its own words)
        s_dbw[lane] = 0.f;
      }
      // [j_first, j_end): what this workgroup replays of the group
      int j_first = 0, j_end = n_mb;
      if (PARTS && done < p.n_shared) {
        const int n_eighths = (n_mb + eighth - 1) / eighth;
        j_first = uni((p.part_start[part] * n_eighths / 8) * eighth);
        j_end = uni(min((p.part_start[part + 1] * n_eighths / 8) * eighth, n_mb));
        if (j_first >= j_end) {
          publish_part(w_replayed);
          continue;
        }
      }
      // park the running gradients while the forward state needs the registers
      if constexpr (ROLE == 0) {
        acc_store_rows(gW1s, bPW1, 0, HID, 0, hid0, c, h);
        acc_store_rows(gW2s, bPW2, 0, FD, hid0, 0, c, h);
        WAVE_SYNC();
        const gptr_t g = park();
        const unsigned o = np_off();
        g_stf(g, o, PARK_BYTES, s_dgw[lane]);   // the walk's sum out
        g_stf(g, o, PARK_BYTES + FD * 4, s_dbw[lane]);
        s_dgw[lane] = 0.f;
        s_dbw[lane] = 0.f;
      }
      AccT<2, 1> W1s;
      AccT<1, 2> W2s;
      acc_load_rows(W1s, bCW1, ckW, HID, 0, hid0, c, h);
      acc_load_rows(W2s, bCW2, ckW, FD, hid0, 0, c, h);
      __syncthreads();  // previous group's readers of the bias vectors are done
      if (tid < HID) s_b1[tid] = p.b1_ck[slot * HID + tid];
      if (tid < FD) s_b2[tid] = p.b2_ck[slot * FD + tid];

      // where XK of a mini-batch on the way to j_first sits: the two buffers in turn, so that the last one is in XQ's
      auto light_xk = [&](int j) { return (j_first - 1 - j) & 1 ? SB_XK : SB_XQ; };
      {
        Staged3 st;
        stage3_load(st, bXQ, bXK, bXV, bETA, k * cgs, tid, t16);
        const bool swap = PARTS && j_first > 0 && light_xk(0) == SB_XQ;
        stage3_store(st, swap ? s_xk : s_xq, swap ? s_xq : s_xk, s_e2, s_etah, tid);
      }
      TTT_STAGE(BS_GROUP);
      // The state through mini-batch j.  FULL: with everything the walk needs of it saved on the way.
      auto step_state = [&](auto full, const int j, bf16* const xk_tile) __attribute__((always_inline)) {
        constexpr bool FULL = decltype(full)::value;
        LANE_VARS;
        // Z1^T = W1s^T XK^T + b1  (rows hid, lane = tok); X2 rows [tok][hid] -> T0; gelu'(Z1) (fp32) and the
        // low-order term of X2 stay in registers.  The products that carry the state to the next mini-batch
        // take their fp32 operands in two bf16 terms (see split8).
        float d1f[2][16];
        bf16x8 x2lo[2][2];
        {
          LANE_VARS;
          AccT<1, 2> x2;
          acc_init_rows_lds(x2, s_b1w, h);
#pragma unroll
          for (int s = 0; s < 4; s++) {
            bf16x8 wh, wl, xk[2];
            split8(W1s.b[s >> 1][0], s & 1, wh, wl);
#pragma unroll
            for (int i = 0; i < 2; i++) xk[i] = xpiece_rows(xk_tile, tb[i], s, c, h);
#pragma unroll
            for (int i = 0; i < 2; i++) {
              x2.b[0][i] = MFMA(wl, xk[i], x2.b[0][i]);
              x2.b[0][i] = MFMA(wh, xk[i], x2.b[0][i]);
            }
          }
#pragma unroll
          for (int i = 0; i < 2; i++)
#pragma unroll
            for (int t = 0; t < 2; t++) {
              const bf16x8 zr = pack8<PAIRS>(x2.b[0][i], t);
              if constexpr (FULL && !IMG) {
                image_store<CACHED>(bZ1, j * IMG_BYTES, 2 * tb[i] + t, t16, zr);
              } else if constexpr (FULL) {
                // The walk needs gelu, gelu' and gelu'' of the ROUNDED Z1 (what it would compute from the image
                // of Z1); a replaying workgroup has the time to do that for it.
                bf16x8 gv, av, bv;
                gelu_images<PAIRS>(zr, gv, av, bv);
                image_store(bZ1, j * IMG_BYTES, 2 * tb[i] + t, t16, gv);
                image_store(bDD, j * (2 * IMG_BYTES), 2 * tb[i] + t, t16, av);
                image_store(bDD, j * (2 * IMG_BYTES) + IMG_BYTES, 2 * tb[i] + t, t16, bv);
              }
              bf16x8 xv;
#pragma unroll
              for (int jj = 0; jj < 8; jj += 2) {
                float g[2];
#pragma unroll
                for (int q = 0; q < 2; q++) {
                  float d;
                  gelu_fd(x2.b[0][i][8 * t + jj + q], g[q], d);
                  d1f[i][8 * t + jj + q] = d;
                  // pinned: left to itself the compiler finishes gelu' only where it is used, two stages on, and keeps
                  // three values per element alive until then instead of one (a dozen of them in scratch memory)
                  asm volatile("" : "+v"(d1f[i][8 * t + jj + q]));
                }
                put_split<PAIRS>(xv, x2lo[i][t], jj, g[0], g[1]);
              }
              store_piece_rows<LDH>(T0, tb[i], t, c, h, xv);
            }
        }
        TTT_STAGE(BS_R_F1_GELU);
        WAVE_SYNC();
        {
          LANE_VARS;
          AccT<2, 2> z2;
          acc_zero(z2);
#pragma unroll
          for (int s = 0; s < 2; s++) {                      // W2s: lane = F, contraction = hid, two terms; X2: lane = tok
            bf16x8 wh[2], wl[2], xb[2];
#pragma unroll
            for (int rb = 0; rb < 2; rb++) split8(W2s.b[0][rb], s, wh[rb], wl[rb]);
#pragma unroll
            for (int i = 0; i < 2; i++) xb[i] = piece_rows<LDH>(T0, tb[i], s, c, h);
#pragma unroll
            for (int rb = 0; rb < 2; rb++)
#pragma unroll
              for (int i = 0; i < 2; i++) {
                z2.b[rb][i] = MFMA(wl[rb], xb[i], z2.b[rb][i]);
                z2.b[rb][i] = MFMA(wh[rb], xb[i], z2.b[rb][i]);
              }
          }
          pair_sum(s_own, s_partner, z2, c, h);
        }
        TTT_STAGE(BS_R_F2_PAIRSUM);
        // fused LayerNorm + reconstruction-loss gradient; saves for the reverse walk
        {
          LANE_VARS;
          float z[8], gam[8];
          {
            float b2v[8];
            ln_gather(z, s_lnrow);
            ln_load_f32(b2v, s_b2 + f0);
#pragma unroll
            for (int e = 0; e < 8; e++) z[e] += b2v[e];
          }
          ln_load_f32(gam, s_gam + f0);
          float sd;
          const float rstd = ln_normalize(z, &sd);
          float go[8], gx[8];
          {
            float kv[8], vv[8], bet[8];
            ln_load(kv, xk_tile + xrow(tok) + f0);
            ln_load(vv, s_e2 + xrow(tok) + f0);
            ln_load_f32(bet, s_bet + f0);
#pragma unroll
            for (int e = 0; e < 8; e++) {
              go[e] = __builtin_fmaf(gam[e], z[e], bet[e]) - (vv[e] - kv[e]);
              gx[e] = go[e] * gam[e];
            }
          }
          if constexpr (FULL) {
            ln_store_g<CACHED, PAIRS>(bXHF, vln, j * TILE_BYTES, z);
            ln_store_g<CACHED, PAIRS>(bGOF, vln, j * TILE_BYTES, go);
          }
          const float s1 = oct_sum(sum8(gx)), s2 = oct_sum(dot8(gx, z));
          const float sc = rstd * (1.f / FD), neg_eta = -bf2f(s_etah[tok]);
#pragma unroll
          for (int e = 0; e < 8; e++) gx[e] = (FD * gx[e] - s1 - z[e] * s2) * sc;   // dl/dZ2
          if constexpr (FULL) ln_store_g<CACHED, PAIRS>(bGZ2, vln, j * TILE_BYTES, gx);
#pragma unroll
          for (int e = 0; e < 8; e++) gx[e] *= neg_eta;                             // G2, in two terms (the second in
          ln_token_sum_store(s_deta + v * CS, gx, lane, f0);   // b2's step: this wave's share (s_deta is the walk's otherwise)
          {                                                                          // the tile gZ2_bar takes later)
            bf16x8 gh, gl;
            split8(gx, gh, gl);
            ln_store_h(s_gz2 + tok * LDX + f0, gh);
            ln_store_h(s_a + tok * LDX + f0, gl);
          }
          if (FULL && (lane & 7) == 0) g_stf(bSDF, vtok, j * (CS * 4), sd);
        }
        if (PARTS && FULL && j == j_first && j > 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // XQ (see below)
        __syncthreads();
        if constexpr (!FULL) {   // XV and eta have been read: the next ones'
          LANE_VARS;
          tile_to_lds<CPOL_NT>(bXV, (k * cgs + j + 1) * TILE_BYTES, smem + SB_E2, v, lane);
          eta_to_lds(bETA, (k * cgs + j + 1) * (CS * 2), smem + SB_ETA, v, lane);
        }
        if (v == 0) {   // b2 += sum over the tokens of G2: the eight waves' fp32 shares in a fixed order (next read: the output LayerNorm)
          LANE_VARS;
          float b = s_b2[lane];
#pragma unroll
          for (int u = 0; u < BW_NWAVE; u++) b += s_deta[u * CS + lane];
          s_b2[lane] = b;
        }
        TTT_STAGE(BS_R_LN);
        // G1 = (W2 G2^T) * gelu'(Z1)  (rows hid, lane = tok) -> T1 rows [tok][hid]; weight step
        {
          LANE_VARS;
          AccT<1, 2> g1;
          acc_zero(g1);
          // W2[shard, :] with F contracted (lane = hid): the two terms of W2s, written as rows [F][hid] into T1 / T2
          // and read back transposed
#pragma unroll
          for (int fb = 0; fb < 2; fb++)
#pragma unroll
            for (int s = 0; s < 2; s++) {
              bf16x8 ph, pl;
              split8(W2s.b[0][fb], s, ph, pl);
              store_piece_rows<LDH>(T1, fb, s, c, h, ph);
              store_piece_rows<LDH>(T2, fb, s, c, h, pl);
            }
          WAVE_SYNC();
#pragma unroll
          for (int s = 0; s < 4; s++) {                      // W2: lane = hid, contraction = F; G2: lane = tok; two terms each
            const bf16x8 wh = piece_tr<LDH>(T1, 0, s, lane), wl = piece_tr<LDH>(T2, 0, s, lane);
            bf16x8 gh[2], gl[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
              gh[i] = piece_rows<LDX>(s_gz2, tb[i], s, c, h);
              gl[i] = piece_rows<LDX>(s_a, tb[i], s, c, h);
            }
#pragma unroll
            for (int i = 0; i < 2; i++) {
              g1.b[0][i] = MFMA(wh, gl[i], g1.b[0][i]);
              g1.b[0][i] = MFMA(wl, gh[i], g1.b[0][i]);
              g1.b[0][i] = MFMA(wh, gh[i], g1.b[0][i]);
            }
          }
          WAVE_SYNC();   // W2's terms are read before G1 takes their place
#pragma unroll
          for (int i = 0; i < 2; i++)
#pragma unroll
            for (int t = 0; t < 2; t++) {
              bf16x8 gv, gvl;
#pragma unroll
              for (int jj = 0; jj < 8; jj += 2) {
                const int k0 = 8 * t + jj, k1 = k0 + 1;
                put_split<PAIRS>(gv, gvl, jj, g1.b[0][i][k0] * d1f[i][k0], g1.b[0][i][k1] * d1f[i][k1]);
              }
              store_piece_rows<LDH>(T1, tb[i], t, c, h, gv);      // G1 rows [tok][hid], two terms
              store_piece_rows<LDH>(T2, tb[i], t, c, h, gvl);
            }
        }
        WAVE_SYNC();
        TTT_STAGE(BS_R_F3);
        {   // weight step
          LANE_VARS;
#pragma unroll
          for (int s = 0; s < 4; s++) {                        // W1[:, shard] += XK^T G1
            bf16x8 xk[2];
#pragma unroll
            for (int fb = 0; fb < 2; fb++) xk[fb] = xpiece_tr(xk_tile, fb, s, lane);               // XK^T: lane = F
            const bf16x8 gh = piece_tr<LDH>(T1, 0, s, lane), gl = piece_tr<LDH>(T2, 0, s, lane);   // G1: lane = hid
#pragma unroll
            for (int fb = 0; fb < 2; fb++) {
              W1s.b[fb][0] = MFMA(xk[fb], gl, W1s.b[fb][0]);
              W1s.b[fb][0] = MFMA(xk[fb], gh, W1s.b[fb][0]);
            }
          }
          lds_rowsum_add_jit(s_b1w, [&](int s) { return piece_tr<LDH>(T2, 0, s, lane); }, ones, c, h);
          lds_rowsum_add_jit(s_b1w, [&](int s) { return piece_tr<LDH>(T1, 0, s, lane); }, ones, c, h);
          // the low-order term of X2 takes G1's place in T1 (rows [tok][hid])
#pragma unroll
          for (int i = 0; i < 2; i++)
#pragma unroll
            for (int t = 0; t < 2; t++) store_piece_rows<LDH>(T1, tb[i], t, c, h, x2lo[i][t]);
          WAVE_SYNC();
#pragma unroll
          for (int s = 0; s < 4; s++) {                        // W2[shard, :] += X2^T G2
            const bf16x8 xh = piece_tr<LDH>(T0, 0, s, lane), xl = piece_tr<LDH>(T1, 0, s, lane);   // X2^T: lane = hid
            bf16x8 gh[2], gl[2];
#pragma unroll
            for (int fb = 0; fb < 2; fb++) {
              gh[fb] = piece_tr<LDX>(s_gz2, fb, s, lane);                                        // G2: lane = F
              gl[fb] = piece_tr<LDX>(s_a, fb, s, lane);
            }
#pragma unroll
            for (int fb = 0; fb < 2; fb++) {
              W2s.b[0][fb] = MFMA(xl, gh[fb], W2s.b[0][fb]);
              W2s.b[0][fb] = MFMA(xh, gl[fb], W2s.b[0][fb]);
              W2s.b[0][fb] = MFMA(xh, gh[fb], W2s.b[0][fb]);
            }
          }
          WAVE_SYNC();   // this wave's readers of T1 / T2 are done
        }
        TTT_STAGE(BS_R_WSTEP);
      };
      if constexpr (PARTS) {
        for (int j = 0; j < j_first; j++) {
          REFRESH_OFFSETS();
          __syncthreads();   // the staged inputs (and, for j = 0, the biases) are visible
          TTT_STAGE(BS_R_TOP);
          {
            LANE_VARS;
            tile_to_lds<CPOL_NT>(bXK, (k * cgs + j + 1) * TILE_BYTES, smem + light_xk(j + 1), v, lane);   // (read last a mini-batch ago)
          }
          step_state(std::false_type{}, j, reinterpret_cast<bf16*>(smem + light_xk(j)));
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the next mini-batch's inputs are in LDS before the barrier
        }
      }
      // The norm-gradient sums of an eighth of the group end at the top of the next one.  Where a group may be replayed in parts they go
      // out on their own, otherwise they are added up here, in the same order, and one sum goes out with the group: two registers (which
      // spill) instead of two stores an eighth and of as many trips to HBM for whoever adds them (ms: 96 x 64 in groups of 8 1.443 ->
      // 1.427, 72 x 64 in 4 1.417 -> 1.366, 51 x 77 in 10 1.205 -> 1.183, 128 x 128 in 16 3.207 -> 3.179).  Of one workgroup per (batch, head)
      // they go out, and the last eighth's stay in LDS.
      float sum0 = 0.f, sum1 = 0.f;
      auto eighth_done = [&](int e) {
        WAVE_SYNC();
        LANE_VARS;
        if constexpr (ROLE == 1 && !EIGHTHS) {
          sum0 = e > 0 ? sum0 + s_dgw[lane] : s_dgw[lane];
          sum1 = e > 0 ? sum1 + s_dbw[lane] : s_dbw[lane];
        } else {
          const gptr_t g = ROLE == 1 ? group_sums(set, e) : park();
          const unsigned o = ROLE == 1 ? 4 * lane : np_off(), so = ROLE == 1 ? 0 : (2 + e) * PARK_BYTES;
          g_stf(g, o, so, s_dgw[lane]);
          g_stf(g, o, so + FD * 4, s_dbw[lane]);
        }
        s_dgw[lane] = 0.f;
        s_dbw[lane] = 0.f;
        WAVE_SYNC();
      };
      int e = uni(PARTS ? j_first / eighth : 0), e_end = j_first + eighth;   // the eighth of the group that mini-batch j is in, and its end
      for (int j = j_first; j < j_end; j++) {
        const int mb = k * cgs + j;
        REFRESH_OFFSETS();
        LANE_VARS;
        __syncthreads();   // the staged inputs (and, for j = 0, the biases) are visible
        TTT_STAGE(BS_R_TOP);
        if (j == e_end) {
          eighth_done(e++);
          e_end += eighth;
        }
        if (PARTS && j == j_first && j > 0) tile_to_lds<CPOL_NT>(bXQ, mb * TILE_BYTES, smem + SB_XQ, v, lane);   // XK was there until now
        step_state(std::true_type{}, j, s_xk);
        // operand images of the state after this step, for the reverse walk; the image of W2 (lane = hid,
        // contraction = F) also serves the output branch below
        bf16x8 w2a[4];
        bf16x8 gO_n;   // LayerNorm lanes: the upstream gradient of their 8 features, asked for two stages ahead
        {
          LANE_VARS;
          gO_n = g_ld_stream<bf16x8>(bGO, vln, mb * TILE_BYTES);
          // bIMG2: W2, lane = hid, contraction = F;  bIMG1: W1^T, lane = F, contraction = hid
          store_state_rows<LDF>(T2, W1s, c, h);                                 // rows [hid][F]
          store_state_rows<LDH>(T1, W2s, c, h);                                 // rows [F][hid]
          WAVE_SYNC();
#pragma unroll
          for (int s = 0; s < 4; s++) {
            w2a[s] = piece_tr<LDH>(T1, 0, s, lane);
            image_store<CACHED>(bIMG2, j * IMG_BYTES, s, t16, w2a[s]);
          }
#pragma unroll
          for (int fb = 0; fb < 2; fb++)
#pragma unroll
            for (int s = 0; s < 2; s++) image_store<CACHED>(bIMG1, j * IMG_BYTES, 2 * fb + s, t16, piece_tr<LDF>(T2, fb, s, lane));
        }
        TTT_STAGE(BS_R_IMAGES);
        // post-update forward on XQ; X2_bar rows [tok][hid] -> T0, gelu'(Z1_bar) packed
        bf16x8 d1b[2][2];
        {
          LANE_VARS;
          AccT<1, 2> z1b;
          acc_init_rows_lds(z1b, s_b1w, h);
          // W1 after the step in two terms: its rounding pattern persists over many mini-batches, so the error it
          // leaves in Z1_bar - and through it in every gradient the output branch feeds - does not average out
#pragma unroll
          for (int s = 0; s < 4; s++) {
            bf16x8 wh, wl, xq[2];
            split8(W1s.b[s >> 1][0], s & 1, wh, wl);
#pragma unroll
            for (int i = 0; i < 2; i++) xq[i] = xpiece_rows(s_xq, tb[i], s, c, h);
#pragma unroll
            for (int i = 0; i < 2; i++) {
              z1b.b[0][i] = MFMA(wl, xq[i], z1b.b[0][i]);
              z1b.b[0][i] = MFMA(wh, xq[i], z1b.b[0][i]);
            }
          }
          bf16x8 x2bQ[2][2];
          WAVE_SYNC();   // the weight step's readers of T0 are done
#pragma unroll
          for (int i = 0; i < 2; i++)
#pragma unroll
            for (int t = 0; t < 2; t++) {
#pragma unroll
              for (int jj = 0; jj < 8; jj += 2) {
                float g[2], d[2];
#pragma unroll
                for (int q = 0; q < 2; q++) gelu_fd(z1b.b[0][i][8 * t + jj + q], g[q], d[q]);
                put_cvt<PAIRS>(x2bQ[i][t], jj, g[0], g[1]);
                put_cvt<PAIRS>(d1b[i][t], jj, d[0], d[1]);
              }
              asm volatile("" : "+v"(d1b[i][t]));   // finished here, not where it is used (see gelu'(Z1) above)
              store_piece_rows<LDH>(T0, tb[i], t, c, h, x2bQ[i][t]);
            }
          AccT<2, 2> z2;
          acc_zero(z2);
          mma_jit<2>(z2, [&](int rb, int s) { return piece_state(W2s, rb, s); },
                     [&](int i, int s) { return x2bQ[i][s]; });
          WAVE_SYNC();   // this wave's readers of T1 / T2 are done
          pair_sum(s_own, s_partner, z2, c, h);
        }
        TTT_STAGE(BS_R_OUT_FORWARD);
        // ---- the output branch, backwards: it needs the state after this step, which is in registers
        //      right now, and nothing of the running gradients.  Output LayerNorm forward and backward:
        float gO[8];
        bf16x8 dxq_old;
        Staged3 next;
        {
          LANE_VARS;
          float z[8], gx[8], gam[8];
          {
            float b2v[8];
            ln_gather(z, s_lnrow);
            ln_load_f32(b2v, s_b2 + f0);
#pragma unroll
            for (int e = 0; e < 8; e++) z[e] += b2v[e];
          }
          asm volatile("" : "+v"(gO_n));   // not converted, and waited for, as soon as it is asked for
          ln_cvt8(gO, gO_n);
          // The next mini-batch's tiles: in registers until every reader of this one's is done, at the end (the last one's come again,
          // unread).  Straight to LDS they were waited for at this stage's barrier, together with every store of images before them.
          stage3_load(next, bXQ, bXK, bXV, bETA, j + 1 < j_end ? mb + 1 : mb, tid, t16);
          float sd;
          ln_normalize(z, &sd);   // z = x_hat
          ln_load_f32(gam, s_gam + f0);
#pragma unroll
          for (int e = 0; e < 8; e++) gx[e] = gO[e] * z[e];
          ln_token_sum_add(s_dbw, gO, lane, f0);
          ln_token_sum_add(s_dgw, gx, lane, f0);
#pragma unroll
          for (int e = 0; e < 8; e++) gx[e] = gO[e] * gam[e];
          const float s1 = oct_sum(sum8(gx)), s2 = oct_sum(dot8(gx, z));
          const float sc = 1.f / (FD * sd);
#pragma unroll
          for (int e = 0; e < 8; e++) gx[e] = (FD * gx[e] - s1 - z[e] * s2) * sc;
          ln_store<PAIRS>(s_a + tok * LDX + f0, gx);            // gZ2_bar
          ln_store_g<CACHED, PAIRS>(bGZB, vln, j * TILE_BYTES, gx);
        }
        __syncthreads();
        TTT_STAGE(BS_R_OUT_LN);
        {
          LANE_VARS;
          dxq_old = g_ld_stream<bf16x8>(OLD_VALUE(bDXQ, mb * TILE_BYTES));   // ahead of the images' stores, which it would have to wait for
          // W1 after the step (lane = F, contraction = hid).  Beside a walk it is the image stored above, fetched ahead of its use; where
          // the same workgroup walks, and every CU is busy, that is a trip to HBM, and it goes through T2 once more (backward,
          // ms, 384 x 512 33.5 -> 33.3, 200 x 100 3.68 -> 3.65 or the same; 96 x 128, with 64 CUs idle, 2.65 -> 2.67).
          constexpr bool W1_AGAIN = ROLE == 0 && !CACHED;
          bf16x8 w1a[2][2];
          if constexpr (!W1_AGAIN)
#pragma unroll
            for (int rb = 0; rb < 2; rb++)
#pragma unroll
              for (int s = 0; s < 2; s++) w1a[rb][s] = chunk_load(bIMG1, j * IMG_BYTES, 2 * rb + s, t16);
          {
            LANE_VARS;
            AccT<1, 2> gz1b;   // (gZ2_bar W2^T) * gelu'(Z1_bar): rows hid, lane = tok
            acc_zero(gz1b);
            // W2 after the step in two terms here as well (see W1 above): the low-order term goes through T2 like the
            // high-order one went through T1 for the image
#pragma unroll
            for (int fb = 0; fb < 2; fb++)
#pragma unroll
              for (int s = 0; s < 2; s++) {
                bf16x8 ph, pl;
                split8(W2s.b[0][fb], s, ph, pl);
                store_piece_rows<LDH>(T2, fb, s, c, h, pl);
              }
            WAVE_SYNC();
#pragma unroll
            for (int s = 0; s < 4; s++) {
              const bf16x8 wl = piece_tr<LDH>(T2, 0, s, lane);
              bf16x8 gb[2];
#pragma unroll
              for (int i = 0; i < 2; i++) gb[i] = piece_rows<LDX>(s_a, tb[i], s, c, h);
#pragma unroll
              for (int i = 0; i < 2; i++) {
                gz1b.b[0][i] = MFMA(wl, gb[i], gz1b.b[0][i]);
                gz1b.b[0][i] = MFMA(w2a[s], gb[i], gz1b.b[0][i]);
              }
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
              for (int t = 0; t < 2; t++) {
                bf16x8 gzb;
#pragma unroll
                for (int jj = 0; jj < 8; jj += 2)
                  put_cvt<PAIRS>(gzb, jj, gz1b.b[0][i][8 * t + jj] * (float)d1b[i][t][jj], gz1b.b[0][i][8 * t + jj + 1] * (float)d1b[i][t][jj + 1]);
                store_piece_rows<LDH>(T1, tb[i], t, c, h, gzb);    // gZ1_bar rows [tok][hid]
              }
          }
          WAVE_SYNC();   // (W2's low-order term is read)
          if constexpr (W1_AGAIN) {
            store_state_rows<LDF>(T2, W1s, c, h);   // rows [hid][F]
            WAVE_SYNC();
          }
          AccT<2, 2> dq;
          acc_zero(dq);
          mma_jit<2>(dq, [&](int rb, int s) { return W1_AGAIN ? piece_tr<LDF>(T2, rb, s, lane) : w1a[rb][s]; },
                     [&](int i, int s) { return piece_rows<LDH>(T1, tb[i], s, c, h); });                   // gZ1_bar: lane = tok
          // what the reverse walk adds to the running gradients, as ready-made operands (lane = hid, contraction = tok)
#pragma unroll
          for (int s = 0; s < 4; s++) {
            image_store<CACHED>(bX2B, j * IMG_BYTES, s, t16, piece_tr<LDH>(T0, 0, s, lane));
            image_store<CACHED>(bGZ1B, j * IMG_BYTES, s, t16, piece_tr<LDH>(T1, 0, s, lane));
          }
          WAVE_SYNC();   // every reader of T1 / T2 is done before the pair sum takes their place
          pair_sum(s_own, s_partner, dq, c, h);
        }
        {
          LANE_VARS;
          float z[8];
          ln_gather(z, s_lnrow);
          asm volatile("" : "+v"(dxq_old));
#pragma unroll
          for (int e = 0; e < 8; e++) z[e] = (float)dxq_old[e] + (z[e] + gO[e]);
          g_st_stream<bf16x8>(bDXQ, vln, mb * TILE_BYTES, cvt8<PAIRS>(z));
        }
        stage3_store(next, s_xq, s_xk, s_e2, s_etah, tid);   // (read last ahead of the output branch's pair sum)
        TTT_STAGE(BS_R_OUT_BACKWARD);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if constexpr (ROLE == 1) eighth_done(e);
      if constexpr (ROLE == 1 && !EIGHTHS) {
        LANE_VARS;
        const gptr_t g = group_sums(set, 0);
        g_stf(g, 4 * lane, 0, sum0);
        g_stf(g, 4 * lane, FD * 4, sum1);
      }
      // running gradients back into registers
      if constexpr (ROLE == 0) {
        LANE_VARS;
        // one round trip to HBM for the words and the gradients (200 pairs x 100 mini-batches, 7 groups: 5.42 ms forward +
        // backward with a word at a time and their address kept over the loops, 5.36 so)
        const gptr_t g = park();
        const unsigned o = np_off();
        const float r0 = g_ldf(g, o, 0), r1 = g_ldf(g, o, FD * 4), w0 = g_ldf(g, o, PARK_BYTES), w1 = g_ldf(g, o, PARK_BYTES + FD * 4);
        float e0[7], e1[7];
        const int n_out = (n_mb + eighth - 1) / eighth - 1;   // eighths that are out
#pragma unroll
        for (int e = 0; e < 7; e++) {
          e0[e] = e < n_out ? g_ldf(g, o, (2 + e) * PARK_BYTES) : 0.f;
          e1[e] = e < n_out ? g_ldf(g, o, (2 + e) * PARK_BYTES + FD * 4) : 0.f;
        }
        acc_load_rows(gW1s, bPW1, 0, HID, 0, hid0, c, h);
        acc_load_rows(gW2s, bPW2, 0, FD, hid0, 0, c, h);
        WAVE_SYNC();
        float a0 = s_dgw[lane], a1 = s_dbw[lane];
        if (n_out > 0) {
          float t0 = e0[0], t1 = e1[0];
#pragma unroll
          for (int e = 1; e < 7; e++)
            if (e < n_out) { t0 += e0[e]; t1 += e1[e]; }
          a0 = t0 + a0;
          a1 = t1 + a1;
        }
        s_dgw[lane] = w0;
        s_dbw[lane] = w1;
        g_stf(g, o, 0, r0 + a0);   // the running sum
        g_stf(g, o, FD * 4, r1 + a1);
        WAVE_SYNC();
      }
      if constexpr (ROLE == 1 && !HELPED) publish_part(w_replayed);
      if constexpr (ROLE == 1 && HELPED) publish(w_replayed, done + 1);
      if constexpr (ROLE == 0 && HELPED) {
        if (v == 0 && lane_v == 0) __hip_atomic_fetch_add(reinterpret_cast<uint64_t*>(w_sync + BWD_HELP), 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      TTT_STAGE(BS_PUBLISH);
    }
    const int set = in_set;

    // ================================================================= reverse walk
    // Operands are fetched from HBM right where they are consumed: with two waves per SIMD the other
    // wave covers the latency, while holding requests in registers across stages costs more in spills
    // than it gains (measured).
    // adds the replay's share of the norm gradients of the group in `set` to the running sum
    auto add_norm_sums = [&]() {
      LANE_VARS;
      const gptr_t g = park();
      const unsigned o = (v * 2 * FD + lane) * 4;
      const gptr_t gs = group_sums(set, 0);
      const float r0 = g_ldf(g, o, 0), r1 = g_ldf(g, o, FD * 4), a0 = g_ldf(gs, 4 * lane, 0), a1 = g_ldf(gs, 4 * lane, FD * 4);
      g_stf(g, o, 0, r0 + a0);
      g_stf(g, o, FD * 4, r1 + a1);
    };
    if constexpr (ROLE == 0 && HELPED) {
      if (set > 0) {
        if (uni(wait_at_least(w_replayed, done + 1, w_status, s_flag, p.wait_limit)) == 0) return false;
        add_norm_sums();
      }
    }
    if constexpr (ROLE == 2) {
      if (!wait_at_least(w_replayed, parts_until(p, done), w_status, s_flag, p.wait_limit)) return false;
      if constexpr (FIN) {   // the hand-over set of this group's parity is free once the group before last is finished
        if (done >= 2 && !wait_at_least(w_finished, done - 1, w_status, s_flag, p.wait_limit)) return false;
      } else {
        add_norm_sums();
      }
    }
    // hand-over buffers of this group for the grad_L_XK workgroup (set = parity of the group)
    const size_t ofin = uni64(((size_t)bh * 2 + (done & 1)) * cgs);
#define bFDZ gbuf(ka->fin_dz + ofin * (CS * HID))
#define bFGY gbuf(ka->fin_gy + ofin * (2 * CS * FD))
    TTT_STAGE(BS_GROUP);
    // What a mini-batch of the walk needs first - its two input tiles, the two tiles the replay left for it (gZ2 and
    // gZ2_bar) and eta - is requested during the updates of the mini-batch walked before it and held in registers
    // until the barrier that opens the mini-batch (the very first one of a group is requested here).  The walk is the
    // longest chain of the backward pass; with the lines in the L2 already, a request a stage earlier hides the rest.
    u32x4 n_xq, n_xk, n_gz, n_gzb;
    bf16 n_eta, n_etai[2];
    // What the output branch adds to the running gradients: the replay has taken that branch backwards already
    // and left gZ2_bar (a tile) and X2_bar^T, gZ1_bar^T as operand images.
    bf16x8 x2b[4], g1b[4];   // lane = hid, contraction = tok
#define WALK_FETCH(jn)                                                                                   \
    {                                                                                                    \
      LANE_VARS;                                                                                         \
      const int jf = __builtin_amdgcn_readfirstlane(jn), mbf = k * cgs + jf;                             \
      const unsigned xo = mbf * TILE_BYTES, so = jf * TILE_BYTES;                                        \
      n_etai[0] = g_ldh(bETA, 2 * c, mbf * (CS * 2) + 64 * tb[0]);                                       \
      n_etai[1] = g_ldh(bETA, 2 * c, mbf * (CS * 2) + 64 * tb[1]);                                       \
      n_xq = g_ld_stream<u32x4>(bXQ, t16, xo);                                                           \
      n_xk = g_ld_stream<u32x4>(bXK, t16, xo);                                                           \
      n_gz = g_ld_stream<u32x4>(bGZ2, t16, so);                                                          \
      n_gzb = g_ld_stream<u32x4>(bGZB, t16, so);                                                         \
      n_eta = g_ldh(bETA, 2 * (tid & (CS - 1)), mbf * (CS * 2));                                         \
    }
    if constexpr (ROLE != 1) WALK_FETCH(n_mb - 1);
    if constexpr (ROLE != 1)
    for (int jj = n_mb - 1; jj >= 0; jj--) {
      // (in a scalar register: left to itself the compiler keeps sums of the images' offsets in vector registers over the whole
      // mini-batch and spills them, up to 14 reloads, each of which waits for every load under way; 51 pairs x 77: 1.60 ms)
      const int j = ROLE == 2 ? __builtin_amdgcn_readfirstlane(jj) : jj;
      const int mb = k * cgs + j;
      REFRESH_OFFSETS();
      LANE_VARS;
      const unsigned xo = mb * TILE_BYTES;       // this mini-batch in the input / output tensors
      const unsigned so = j * TILE_BYTES;        // its slot in the [cgs][64][64] scratch tensors
      const unsigned ho = j * IMG_BYTES;         // its slot in the [cgs][64][256] scratch tensors
      // eta of the token this lane holds in column block i of a Q-orientation tile
      const float eta_i[2] = {bf2f(n_etai[0]), bf2f(n_etai[1])};
      {
        LANE_VARS;
        // the two operand images of the next stage are asked for here: on their way across both barriers
#pragma unroll
        for (int s = 0; s < 4; s++) {
          x2b[s] = image_load(bX2B, ho, s, t16);
          g1b[s] = image_load(bGZ1B, ho, s, t16);
        }
        __syncthreads();   // the previous mini-batch's readers of these tiles are done
        lds_put16x(s_xq, tid, n_xq);
        lds_put16x(s_xk, tid, n_xk);
        lds_put16(s_gz2, tid, n_gz);
        lds_put16(s_a, tid, n_gzb);
        if (tid < CS) s_eta[tid] = bf2f(n_eta);
      }
      __syncthreads();

      TTT_STAGE(BS_W_TOP);
      bf16x8 w2bf[4];   // W2 before this step (lane = hid, contraction = F): fetched now, needed by the next stage
      bf16x8 gq[2][2], aq[2][2], bq[2][2];
      {
        LANE_VARS;
#pragma unroll
        for (int s = 0; s < 4; s++) w2bf[s] = w2_before<ROLE == 2>(bIMG2, bCW2, ckW, j, s, hid0, c, h, t16);
        if constexpr (IMG) {   // the three GELU images of the next stage, under way during this one
#pragma unroll
          for (int i = 0; i < 2; i++)
#pragma unroll
            for (int t = 0; t < 2; t++) {
              gq[i][t] = image_load(bZ1, ho, 2 * tb[i] + t, t16);
              aq[i][t] = chunk_load(bDD, j * (2 * IMG_BYTES), 2 * tb[i] + t, t16);   // read again two stages on
              bq[i][t] = image_load(bDD, j * (2 * IMG_BYTES) + IMG_BYTES, 2 * tb[i] + t, t16);
            }
        } else {               // the image of Z1 (gq takes it), from which the next stage evaluates the three
#pragma unroll
          for (int i = 0; i < 2; i++)
#pragma unroll
            for (int t = 0; t < 2; t++) gq[i][t] = image_load(bZ1, ho, 2 * tb[i] + t, t16);
        }
        mma_jit<4>(gW2s, [&](int, int s) { return x2b[s]; },                                   // X2_bar^T: lane = hid
                   [&](int fb, int s) { return piece_tr<LDX>(s_a, fb, s, lane); });            // gZ2_bar: lane = F
        if (v < 2) lds_rowsum_add_jit(s_gb2 + 32 * v, [&](int s) { return piece_tr<LDX>(s_a, v, s, lane); }, ones, c, h);
        mma_jit<4>(gW1s, [&](int fb, int s) { return xpiece_tr(s_xq, fb, s, lane); },         // XQ^T: lane = F
                   [&](int, int s) { return g1b[s]; });                                        // gZ1_bar: lane = hid
        lds_rowsum_add_jit(s_gb1w, [&](int s) { return g1b[s]; }, ones, c, h);
      }
      // gb2 holds its value after the first update

      TTT_STAGE(BS_W_BAR_TERMS);
      // ---- the weight step, backwards (uses the state BEFORE this mini-batch).
      //      Kept across the LayerNorm stage: X2 in T0; packed d1 = gelu'(Z1), g1 = -eta * dl/dZ1 and
      //      t2 = -eta * (gZ2 W2^T) * (XK gW1 + gb1) * gelu''(Z1).
      bf16x8 dxv_old;            // LayerNorm lanes: the two outputs the stage accumulates into
      bf16 deta_old;
      bf16x8 xhf_n, gof_n;       // and the saved x_hat, grad_output, std of the fused LayerNorm
      float sdf_n;
      bf16x8 w2b[4];             // W2 before the step: lane = hid, contraction = F
      // Block 1's of what block 0 parks across the LayerNorm stage (below).  With the GELU images, twelve of which are held while the
      // blocks are computed, both blocks' are parked.
      constexpr bool KEEP = !IMG;
      bf16x8 k_uh[2], k_d1[2], k_t2[2], k_g1[2];
      {
        LANE_VARS;
        // T1 = W2 before the step, rows [hid][F]; T2 = gW1, rows [hid][F]
#pragma unroll
        for (int s = 0; s < 4; s++)
          store_piece_rows<LDF>(T1, 0, s, c, h, w2bf[s]);
        store_state_rows<LDF>(T2, gW1s, c, h);
        WAVE_SYNC();
        AccT<2, 2> pz;
        acc_zero(pz);
        float de[2] = {0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 2; i++) {
          AccT<1, 1> R, S;   // R = gZ2 W2^T, S = XK gW1 + gb1   (rows hid, lane = tok)
          acc_zero(R);
          acc_init_rows_lds(S, s_gb1w, h);
          mma_jit<4>(R, [&](int, int s) { return piece_rows<LDF>(T1, 0, s, c, h); },
                     [&](int, int s) { return piece_rows<LDX>(s_gz2, tb[i], s, c, h); });
          mma_jit<4>(S, [&](int, int s) { return piece_rows<LDF>(T2, 0, s, c, h); },
                     [&](int, int s) { return xpiece_rows(s_xk, tb[i], s, c, h); });
          bf16x8 x2c[2], uc[2];
          // gelu(Z1), gelu'(Z1), gelu''(Z1), each rounded to bf16: computed here from the image of Z1, or
          // fetched as three images that a replaying workgroup computed the same way
          bf16x8 ac[2], bc[2];
          if constexpr (!IMG) {
#pragma unroll
            for (int t = 0; t < 2; t++) gelu_images<PAIRS>(gq[i][t], x2c[t], ac[t], bc[t]);
          } else {
#pragma unroll
            for (int t = 0; t < 2; t++) {
              x2c[t] = gq[i][t];
              ac[t] = aq[i][t];
              bc[t] = bq[i][t];
            }
          }
#pragma unroll
          for (int t = 0; t < 2; t++) {
            bf16x8 t2c, g1c, uhc;
#pragma unroll
            for (int jj = 0; jj < 8; jj += 2) {
              float u[2], uh[2], g[2], t2[2];
#pragma unroll
              for (int q = 0; q < 2; q++) {
                const float a = (float)ac[t][jj + q], b = (float)bc[t][jj + q];
                const float r0 = R.b[0][0][8 * t + jj + q], sv = S.b[0][0][8 * t + jj + q];
                const float gz1 = r0 * a;                                   // dl/dZ1
                de[i] = __builtin_fmaf(gz1, sv, de[i]);
                u[q] = sv * a;
                uh[q] = -eta_i[i] * sv * a;
                g[q] = -eta_i[i] * gz1;
                t2[q] = -eta_i[i] * r0 * sv * b;
              }
              put_cvt<PAIRS>(uc[t], jj, u[0], u[1]);
              put_cvt<PAIRS>(uhc, jj, uh[0], uh[1]);
              put_cvt<PAIRS>(g1c, jj, g[0], g[1]);
              put_cvt<PAIRS>(t2c, jj, t2[0], t2[1]);
            }
            // Block 0's go to their parks across the LayerNorm stage (rewritten every mini-batch): held as well, they are more than
            // there are registers for while block 1 is computed (two of the four held: 14 registers spilled for 16).  Block 1's take the
            // place of its R and S and stay, half of 256 KiB per mini-batch that 32 workgroups an L2 mostly sent through HBM (ms,
            // forward + backward: 384 x 512 45.6 -> 43.2, 200 x 100 5.20 -> 5.01).
            // Only grad_L_XK needs G1: its workgroup, where there is one, forms G1 itself.
            if (KEEP && i == 1) {
              k_uh[t] = uhc;
              k_d1[t] = ac[t];
              k_t2[t] = t2c;
              asm volatile("" : "+v"(k_uh[t]), "+v"(k_d1[t]), "+v"(k_t2[t]));   // finished here, not where they are used
              if constexpr (!FIN) {
                k_g1[t] = g1c;
                asm volatile("" : "+v"(k_g1[t]));
              }
            } else {
              chunk_store(bPUH, 0, 2 * tb[i] + t, t16, uhc);
              if constexpr (!IMG) chunk_store(bPW1, PARK_D1, 2 * tb[i] + t, t16, ac[t]);
              chunk_store(bPW2, PARK_T2, 2 * tb[i] + t, t16, t2c);
              if constexpr (!FIN) chunk_store(bPW2, PARK_G1, 2 * tb[i] + t, t16, g1c);
            }
            store_piece_rows<LDH>(T0, tb[i], t, c, h, x2c[t]);             // X2 rows [tok][hid]
          }
          // pz[:, i] = gW2^T X2^T ; dEta partial ; + W2^T u^T
#pragma unroll
          for (int t = 0; t < 2; t++)
#pragma unroll
            for (int rb = 0; rb < 2; rb++) pz.b[rb][i] = MFMA(piece_state(gW2s, rb, t), x2c[t], pz.b[rb][i]);
#pragma unroll
          for (int s = 0; s < 4; s++) {
            const bf16x8 gzv = piece_rows<LDX>(s_gz2, tb[i], s, c, h);
#pragma unroll
            for (int jj = 0; jj < 8; jj++) de[i] = __builtin_fmaf((float)gzv[jj], pz.b[s >> 1][i][8 * (s & 1) + jj], de[i]);
          }
#pragma unroll
          for (int t = 0; t < 2; t++)
#pragma unroll
            for (int rb = 0; rb < 2; rb++) pz.b[rb][i] = MFMA(piece_tr<LDF>(T1, rb, t, lane), uc[t], pz.b[rb][i]);
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const float a = half_sum_valu(de[i]);   // (a shuffle keeps a lane index over the loop, and reloads it here)
          if (h == 0) s_deta[v * CS + 32 * tb[i] + c] = a;
        }
        // W2 is needed once more, behind the LayerNorm stage.  With several workgroups per pair it comes from T1, which is about to go:
        // its image, read 25 k clocks ago, has left the L2 (backward, ms, 96 x 512 10.28 -> 9.91, 128 x 128 2.99 -> 2.89).  One workgroup
        // per pair has no registers for it here (sixteen spilled, read twice) and asks for the image again.
        if constexpr (ROLE == 2)
#pragma unroll
          for (int s = 0; s < 4; s++) {
            w2b[s] = piece_rows<LDF>(T1, 0, s, c, h);
            asm volatile("" : "+v"(w2b[s]));
          }
        WAVE_SYNC();   // this wave's readers of T1 / T2 are done
        TTT_STAGE(BS_W_STEP_BACK);
        {   // what the LayerNorm stage reads from HBM is under way during the pair sum
          LANE_VARS;
          if constexpr (!FIN) dxv_old = g_ld_stream<bf16x8>(OLD_VALUE(bDXV, xo));
          deta_old = g_ldh(ka->overwrite ? gbuf(zero_tile) : bDETA, 2 * tok, ka->overwrite ? 0u : mb * (CS * 2));
          xhf_n = g_ld_stream<bf16x8>(bXHF, vln, so);
          gof_n = g_ld_stream<bf16x8>(bGOF, vln, so);
          sdf_n = g_ldf(bSDF, vtok, j * (CS * 4));
        }
        pair_sum(s_own, s_partner, pz, c, h);
      }
      TTT_STAGE(BS_W_PAIRSUM);
      // all pair sums of ggZ2 and the dEta partial sums are in LDS

      // ---- second-order pass through the fused LayerNorm loss (LayerNorm lanes)
      {
        LANE_VARS;
        float gy[8];
        float gg[8], xh[8], go[8], gz[8], gam[8], gb[8];
        const bf16x8 xhf = xhf_n, gof = gof_n;
        const float sdf = sdf_n;
        ln_gather(gg, s_lnrow);
        ln_load_f32(gb, s_gb2 + f0);
        ln_cvt8(xh, xhf);
        ln_cvt8(go, gof);
        ln_load(gz, s_gz2 + tok * LDX + f0);
        ln_load_f32(gam, s_gam + f0);
        const float neg_eta = -s_eta[tok];
#pragma unroll
        for (int e = 0; e < 8; e++) gg[e] = (gg[e] + gb[e]) * neg_eta;   // grad wrt dl/dZ2
        const float rsd = 1.f / sdf;
        // dEta: -(sum_F gZ2*(X2 gW2 + gb2) + sum_H gZ1*(XK gW1 + gb1))
        {
          LANE_VARS;
          float d[BW_NWAVE / 2];
#pragma unroll
          for (int u = 0; u < BW_NWAVE / 2; u++) d[u] = s_deta[u * CS + tok] + s_deta[(u + BW_NWAVE / 2) * CS + tok];
          const float tot = oct_sum(dot8(gz, gb)) + ((d[0] + d[1]) + (d[2] + d[3]));
          if ((lane & 7) == 0) g_sth(bDETA, 2 * tok, mb * (CS * 2), (bf16)((float)deta_old - tot));
        }
        // (the expressions are walk_layernorm's, ttt_mlp_bwd_wide.hip, which writes out what the compiler fuses here)
        const float s0 = oct_sum(sum8(gg)), a = oct_sum(dot8(gg, xh));
        float bb = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) bb = __builtin_fmaf(go[e] * gam[e], xh[e], bb);
        bb = oct_sum(bb);
        float gx[8], dg[8];
        const float inv = rsd * (1.f / FD);
        float sg = 0.f, sx = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float ggx = (gg[e] - (s0 + xh[e] * a) * (1.f / FD)) * rsd;
          gy[e] = gam[e] * ggx;
          dg[e] = go[e] * ggx + gy[e] * xh[e];
          gx[e] = gy[e] * gam[e] - (go[e] * gam[e] * a + gg[e] * bb) * inv;
          sg += (-gx[e] * xh[e] - gg[e] * gz[e]) * rsd;
          sx += gx[e];
        }
        sg = oct_sum(sg);
        sx = oct_sum(sx);
        if constexpr (!FIN) {   // with a grad_L_XK workgroup these token sums and grad_L_XV are formed there, from g_y and dg
          ln_token_sum_add(s_dgw, dg, lane, f0);
          ln_token_sum_add(s_dbw, gy, lane, f0);
        }
#pragma unroll
        for (int e = 0; e < 8; e++) {
          gx[e] = gx[e] * rsd + (sg * xh[e] - sx * rsd) * (1.f / FD);   // dZ2
        }
        if constexpr (!FIN) {
          float x[8];
#pragma unroll
          for (int e = 0; e < 8; e++) x[e] = (float)dxv_old[e] - gy[e];   // dXV accumulates -g_y
          dxv_old = cvt8<PAIRS>(x);
        }
        // g_y is needed again for dXK: park it (the XQ / E2 tiles are dead by now), or hand it over
        {
          LANE_VARS;
          f32x4 lo = {gy[0], gy[1], gy[2], gy[3]}, hi = {gy[4], gy[5], gy[6], gy[7]};
          if constexpr (FIN) {
            g_st_stream<f32x4>(bFGY, 2 * vln, 4 * so, lo);
            g_st_stream<f32x4>(bFGY, 2 * vln + 16, 4 * so, hi);
            f32x4 dlo = {dg[0], dg[1], dg[2], dg[3]}, dhi = {dg[4], dg[5], dg[6], dg[7]};
            g_st_stream<f32x4>(bFGY, 2 * vln, 4 * so + 2 * TILE_BYTES, dlo);
            g_st_stream<f32x4>(bFGY, 2 * vln + 16, 4 * so + 2 * TILE_BYTES, dhi);
          } else {
            *reinterpret_cast<f32x4*>(s_gy) = lo;
            *reinterpret_cast<f32x4*>(s_gy + 4) = hi;
          }
        }
        ln_store<PAIRS>(s_a + tok * LDX + f0, gx);
        if constexpr (!FIN) g_st_stream<bf16x8>(bDXV, vln, xo, dxv_old);
      }
      TTT_STAGE(BS_W_LN);
      __syncthreads();  // dZ2 tile complete; regions (T1 / T2) free again
      TTT_STAGE(BS_W_LN_BARRIER);

      // ---- inner MLP, backwards (uses the state BEFORE this mini-batch)
      bf16x8 dxk_old;
      {
        LANE_VARS;
        if constexpr (ROLE == 0)
#pragma unroll
          for (int s = 0; s < 4; s++) w2b[s] = w2_before<true>(bIMG2, bCW2, ckW, j, s, hid0, c, h, t16);   // second and last read
        // converted anew: kept from the weight step backwards, the bf16 gradients are 32 registers (and spilled) for 32 instructions
        if constexpr (KEEP)
#pragma unroll
          for (int fb = 0; fb < 2; fb++) asm volatile("" : "+v"(gW1s.b[fb][0]), "+v"(gW2s.b[0][fb]));
        // T2 = gW1 rows [hid][F] (for gW1 G1^T), T1 = gW2 rows [F][hid] (transposed read gives lane = hid)
        if constexpr (!FIN) store_state_rows<LDF>(T2, gW1s, c, h);
        store_state_rows<LDH>(T1, gW2s, c, h);
        WAVE_SYNC();
        AccT<2, 2> dk;
        acc_zero(dk);
        bf16x8 dzp[2][2], uhp[2][2];
#pragma unroll
        for (int ib = 0; ib < 2; ib++) {
          const int i = KEEP ? 1 - ib : ib;   // block 1 first, which has what it needs
          AccT<1, 1> dx2;
          acc_zero(dx2);
          mma_jit<4>(dx2, [&](int, int s) { return piece_tr<LDH>(T1, 0, s, lane); },           // gW2: lane = hid, contraction = F
                     [&](int, int s) { return piece_rows<LDX>(s_gz2, tb[i], s, c, h); });      // P2 = gZ2 gW2^T
#pragma unroll
          for (int e = 0; e < 16; e++) dx2.b[0][0][e] *= -eta_i[i];
          mma_jit<4>(dx2, [&](int, int s) { return w2b[s]; },                                  // + dZ2 W2^T
                     [&](int, int s) { return piece_rows<LDX>(s_a, tb[i], s, c, h); });
          // dk[:, i] = gW1 G1^T  (gW1: lane = F, contraction = hid)
          bf16x8 g1c[2], d1c[2], t2c[2];
#pragma unroll
          for (int t = 0; t < 2; t++) {
            const int n = 2 * tb[i] + t;
            if (KEEP && i == 1) {
              if constexpr (!FIN) g1c[t] = k_g1[t];
              d1c[t] = k_d1[t];
              t2c[t] = k_t2[t];
            } else {
              if constexpr (!FIN) g1c[t] = chunk_load(bPW2, PARK_G1, n, t16);
              if constexpr (!IMG) d1c[t] = chunk_load(bPW1, PARK_D1, n, t16);
              else d1c[t] = image_load(bDD, j * (2 * IMG_BYTES), n, t16);   // its last reader on this XCD
              t2c[t] = chunk_load(bPW2, PARK_T2, n, t16);
            }
          }
          if constexpr (!FIN) {
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
              for (int rb = 0; rb < 2; rb++) dk.b[rb][i] = MFMA(piece_tr<LDF>(T2, rb, t, lane), g1c[t], dk.b[rb][i]);
          }
          // dZ1 = dX2*gelu' + t2 ;  -eta * S * gelu'   (kept as pieces until T1 / T2 may be overwritten)
#pragma unroll
          for (int t = 0; t < 2; t++)
#pragma unroll
            for (int jj = 0; jj < 8; jj += 2)
              put_cvt<PAIRS>(dzp[i][t], jj, __builtin_fmaf(dx2.b[0][0][8 * t + jj], (float)d1c[t][jj], (float)t2c[t][jj]),
                                       __builtin_fmaf(dx2.b[0][0][8 * t + jj + 1], (float)d1c[t][jj + 1], (float)t2c[t][jj + 1]));
#pragma unroll
          for (int t = 0; t < 2; t++) uhp[i][t] = KEEP && i == 1 ? k_uh[t] : chunk_load(bPUH, 0, 2 * tb[i] + t, t16);   // -eta * S * gelu', formed with S two stages back
        }
        bf16x8 w1bf[2][2];   // W1^T before the step (lane = F, contraction = hid), for the product after the next fence
        if constexpr (!FIN) {
#pragma unroll
          for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int s = 0; s < 2; s++) w1bf[rb][s] = w1_before(bIMG1, bCW1, ckW, j, rb, s, hid0, c, h, t16);
        } else {   // dZ1 leaves for the other workgroup (which keeps its own copy of gW1: it sees every term added to it)
#pragma unroll
          for (int i = 0; i < 2; i++)
#pragma unroll
            for (int t = 0; t < 2; t++) image_store(bFDZ, ho, 2 * tb[i] + t, t16, dzp[i][t]);
        }
        TTT_STAGE(BS_W_MLP_BACK);
        WAVE_SYNC();   // S, P2 and gW1 G1^T have consumed T2 / T1
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int t = 0; t < 2; t++) {
            store_piece_rows<LDH>(T1, tb[i], t, c, h, dzp[i][t]);   // dZ1 rows [tok][hid]
            store_piece_rows<LDH>(T2, tb[i], t, c, h, uhp[i][t]);   // -eta u rows [tok][hid]
          }
        WAVE_SYNC();
        WALK_FETCH(j > 0 ? j - 1 : 0);   // the next mini-batch's tiles (the last step of a group asks for its own again)
        if constexpr (!FIN)
          mma_jit<2>(dk, [&](int rb, int s) { return w1bf[rb][s]; },                           // + W1 dZ1^T, W1 before the step
                     [&](int i, int s) { return dzp[i][s]; });
        mma_jit<4>(gW2s, [&](int, int s) { return piece_tr<LDH>(T2, 0, s, lane); },            // (-eta u)^T: lane = hid
                   [&](int fb, int s) { return piece_tr<LDX>(s_gz2, fb, s, lane); });          // gZ2: lane = F
        mma_jit<4>(gW2s, [&](int, int s) { return piece_tr<LDH>(T0, 0, s, lane); },            // X2^T: lane = hid
                   [&](int fb, int s) { return piece_tr<LDX>(s_a, fb, s, lane); });            // dZ2: lane = F
        if (v < 2) lds_rowsum_add_jit(s_gb2 + 32 * v, [&](int s) { return piece_tr<LDX>(s_a, v, s, lane); }, ones, c, h);
        mma_jit<4>(gW1s, [&](int fb, int s) { return xpiece_tr(s_xk, fb, s, lane); },         // XK^T: lane = F
                   [&](int, int s) { return piece_tr<LDH>(T1, 0, s, lane); });                 // dZ1: lane = hid
        lds_rowsum_add_jit(s_gb1w, [&](int s) { return piece_tr<LDH>(T1, 0, s, lane); }, ones, c, h);
        TTT_STAGE(BS_W_UPDATES);
        WAVE_SYNC();   // this wave's readers of T1 / T2 are done
        if constexpr (!FIN) {
          {
            LANE_VARS;
            dxk_old = g_ld_stream<bf16x8>(OLD_VALUE(bDXK, xo));   // under way during the pair sum
          }
          pair_sum(s_own, s_partner, dk, c, h);
        }
      }
      // pair sums of dXK complete
      if constexpr (!FIN) {
        LANE_VARS;
        float z[8], gyv[8];
        ln_gather(z, s_lnrow);
        ln_load_f32(gyv, s_gy);
#pragma unroll
        for (int e = 0; e < 8; e++) z[e] = (float)dxk_old[e] + (z[e] + gyv[e]);
        g_st_stream<bf16x8>(bDXK, vln, xo, cvt8<PAIRS>(z));
      }
      TTT_STAGE(BS_W_DXK);
      if constexpr (ROLE == 2 && FIN) {
        // The last group to be walked is handed to the grad_L_XK workgroup in chunks, so that that workgroup follows
        // FIN_CHUNK mini-batches behind instead of ending a whole group after the walk.
        if (k == 0 && (j & (FIN_CHUNK - 1)) == 0) {
          publish(w_sync + 12, n_mb - j);
          TTT_STAGE(BS_PUBLISH);
        }
      }
    }
    if constexpr (ROLE == 2) publish(w_walked, done + 1);
    TTT_STAGE(BS_PUBLISH);
#undef bFDZ
#undef bFGY
#undef WALK_FETCH
  }
  TTT_STAGES_END(bh, ROLE == 1 ? 0 : STAGE_ROLE_WALK);
  if constexpr (ROLE == 1) return true;

  // ---- outputs that are written once
  acc_store_rows(gW1s, gbuf(p.grad_L_W1_init + (size_t)bh * FD * HID), 0, HID, 0, hid0, c, h);
  acc_store_rows(gW2s, gbuf(p.grad_L_W2_init + (size_t)bh * HID * FD), 0, FD, hid0, 0, c, h);
  __syncthreads();
  if (tid < HID) p.grad_L_b1_init[(size_t)bh * HID + tid] = s_gb1[tid];
  if (tid < FD) p.grad_L_b2_init[(size_t)bh * FD + tid] = s_gb2[tid];
  // norm-weight / norm-bias gradients: sum the per-wave LDS accumulators
  if constexpr (FIN) return true;   // with a grad_L_XK workgroup the walk holds no share of these sums: they are written there
  if (ROLE == 0 && !seg_last) {   // the next segment goes on with the walk's sum (the replay's is in place already)
    g_stf(park(), np_off(), PARK_BYTES, s_dgw[lane]);
    g_stf(park(), np_off(), PARK_BYTES + FD * 4, s_dbw[lane]);
    return true;
  }
  if (tid < 2 * FD) {
    const int which = tid / FD, f = tid % FD;
    const float* rp = ROLE == 0 ? reinterpret_cast<const float*>(p.x_hat_ln_group + (size_t)bh * cgs * (CS * FD))
                                : p.norm_park + (size_t)bh * (BW_NWAVE * 2 * FD);
    float s = 0.f, sr = 0.f;
#pragma unroll
    for (int u = 0; u < BW_NWAVE; u++) {
      s += s_red[(u * 2 + which) * FD + f];
      sr += rp[(u * 2 + which) * FD + f];   // the other waves' stores: before the barrier above
    }
    (which == 0 ? p.grad_L_ttt_norm_weight : p.grad_L_ttt_norm_bias)[(size_t)bh * FD + f] = sr + s;
  }
  return true;
}
#undef REFRESH_OFFSETS
#undef LANE_VARS
#undef GRP
#undef bXQ
#undef bXK
#undef bXV
#undef bGO
#undef bETA
#undef bZ1
#undef bGZ1B
#undef bX2B
#undef bGZB
#undef bIMG1
#undef bIMG2
#undef bXHF
#undef bGOF
#undef bGZ2
#undef bSDF
#undef bDD
#undef bPUH
#undef bPW1
#undef bPW2
#undef bCW1
#undef bCW2
#undef bDXQ
#undef bDXK
#undef bDXV
#undef bDETA

#ifndef TTT_BWD_ROLES_ONLY   // ttt_mlp_bwd_wide.hip takes the roles above and below without these kernels
__global__ __launch_bounds__(BW_THREADS) void ttt_mlp_bwd_kernel(const BwdParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  int bh = p.bh0 + blockIdx.x, k_hi = p.K - 1, k_lo = 0;
  if (p.seg_groups > 0) {
    const int pairs = p.B * p.NH, job = p.job0 + blockIdx.x, seg = job / pairs;
    bh = job - seg * pairs;
    k_hi = p.K - 1 - seg * p.seg_groups;
    k_lo = k_hi - p.seg_groups + 1 > 0 ? k_hi - p.seg_groups + 1 : 0;
  }
  // With few pairs a group's images stay in the memory-side cache until they are walked unless they are streamed there; with many they
  // do not, and streamed they leave the L2 to the parks.  The line lies between 64 pairs (x 64 mini-batches in groups of 16: 2.24 ms
  // streamed, 2.19 cached; 48 x 256 8.85, 8.65) and 96 (2.26, 2.29).
  if (p.nbh < 80) bwd_body<0, false, false, false, false, false, false, true>(p, smem, bh, k_hi, k_lo);
  else bwd_body<0, false, false>(p, smem, bh, k_hi, k_lo);
}
#endif

// grad_L_XK on a workgroup of its own: for every mini-batch of every group, as soon as the walk is done with the
// group, dk = gW1 G1^T + W1 dZ1^T (W1 before the step: from the replay's image, or the checkpoint), its sum over
// the hidden dimension, + g_y, accumulated into grad_L_XK.  Same wave / lane roles and the same order of every
// sum as in the walk, so the result is the same to the bit.  OWN: the whole sequence (k_hi = K - 1); otherwise fewer such
// workgroups than pairs take the groups in turn and this is group k_hi, with what is carried from group to group (the copy of
// the gradient wrt W1 and the norm-gradient sums) parked in between.  EIGHTHS: as in the replay.  False: a wait gave up.
template <bool IMG, bool WIDE, bool OWN, bool EIGHTHS>
TTT_DEV bool bwd_finish_dxk(const BwdParams& p, unsigned char* smem, const int bh, const int k_hi) {
  float* s_P = reinterpret_cast<float*>(smem + SB_P);
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));   // nothing derived from it is kept over the caller's loop over groups
  const int lane = tid & 63, h = lane >> 5, c = lane & 31;
  const int v = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pp = v & 3, r = v >> 2;
  const int tb[2] = {r, 1 - r};
  const int q8 = lane >> 3, tok = 8 * v + q8, f0 = 8 * (lane & 7);
  const int hid0 = BW_NS * v;
  float* s_own = s_P + (pp * 2 + r) * RGN;
  float* s_partner = s_P + (pp * 2 + (1 - r)) * RGN;
  const float* s_lnrow = s_P + (1 - r) * RGN + (tok & 31) * LDR + f0;
  const int cgs = p.cgs, n_sets = p.n_sets;
  const unsigned t16 = 16 * tid, vln = (tok * FD + f0) * 2;
  int* const w_sync = p.sync + (size_t)bh * BWD_SYNC_STRIDE;
  int* const w_walked = w_sync + 16;
  int* const w_finished = w_sync + 24;
  int* const s_flag = reinterpret_cast<int*>(smem + SB_FLAG);
  const gptr_t gDXK = gbuf(p.grad_L_XK + uni64((size_t)bh * p.NC * (CS * FD)));
  const gptr_t gDXV = gbuf(p.grad_L_XV + uni64((size_t)bh * p.NC * (CS * FD)));
  const gptr_t gCW1 = gbuf(p.W1_ck + uni64((size_t)bh * p.K * (FD * HID)));
  const gptr_t gXQ = gbuf(p.XQ + uni64((size_t)bh * p.NC * (CS * FD))), gXK = gbuf(p.XK + uni64((size_t)bh * p.NC * (CS * FD)));
  bf16* const s_xq = reinterpret_cast<bf16*>(smem + SB_XQ);
  bf16* const s_xk = reinterpret_cast<bf16*>(smem + SB_XK);
  bf16* const s_gz2 = reinterpret_cast<bf16*>(smem + SB_GZ2);
  const gptr_t gETA = gbuf(p.last_eta + uni64((size_t)bh * p.NC * CS));
  const gptr_t gCW2 = gbuf(p.W2_ck + uni64((size_t)bh * p.K * (FD * HID)));
  bf16* const T1 = reinterpret_cast<bf16*>(s_own);   // wave-private tiles in this wave's pair-sum region, as in the walk
  bf16* const T2 = T1 + 64 * LDH;
  // This workgroup keeps its own copy of the running gradient wrt W1: both terms the walk adds to it per
  // mini-batch (XQ^T gZ1_bar and XK^T dZ1) are formed from data that reaches this workgroup anyway, in the walk's order.
  AccT<2, 1> gW1s;
  const bool first = OWN || k_hi == p.K - 1;
  float* const park = p.fin_park + (size_t)bh * FIN_PARK_FLOATS;
  if (!first && !wait_at_least(w_finished, p.K - 1 - k_hi, p.status, s_flag, p.wait_limit)) return false;   // the group before is parked
  acc_load_rows(gW1s, gbuf(first ? p.grad_L_W1_last + (size_t)bh * FD * HID : park), 0, HID, 0, hid0, c, h);
  // the walk's share of the norm-weight / norm-bias gradients: per wave, summed in the walk's order
  float* s_red = reinterpret_cast<float*>(smem + SB_RED);
  float* s_dgw = s_red + (v * 2 + 0) * FD;
  float* s_dbw = s_red + (v * 2 + 1) * FD;
  float nr0 = 0.f, nr1 = 0.f;   // the replay's share: this lane's two words of the wave's running sum
  {
    float w0 = 0.f, w1 = 0.f;
    if (!first) {
      const float* const q = park + FD * HID + v * 4 * FD + lane;
      w0 = q[0]; w1 = q[FD]; nr0 = q[2 * FD]; nr1 = q[3 * FD];
    }
    s_dgw[lane] = w0;
    s_dbw[lane] = w1;
  }
  // mini-batches walked before group k_hi (the ragged group is the first), and how many of them are known to have been
  int n_step = first ? 0 : p.NC - (k_hi + 1) * cgs, n_seen = 0;
  int lane_v = lane;
#define FIN_LANE                                                                                  \
  asm volatile("" : "+v"(lane_v));                                                                \
  const int lane = lane_v, h = lane >> 5, c = lane & 31, tid = (v << 6) | lane;                   \
  const int tok = 8 * v + (lane >> 3), f0 = 8 * (lane & 7);                                       \
  const unsigned t16 = 16 * tid, vln = (tok * FD + f0) * 2;                                       \
  const float* s_lnrow = s_P + (1 - r) * RGN + (tok & 31) * LDR + f0;                             \
  (void)h; (void)c; (void)t16; (void)vln; (void)s_lnrow
  TTT_STAGES_BEGIN();
  int k = k_hi;
  do {
    const int n_mb = min(cgs, p.NC - k * cgs);
    const int done = p.K - 1 - k, set = done % n_sets;
    // the walk hands over whole groups, except the last one it walks (k = 0): that one in chunks of FIN_CHUNK mini-batches
    // (WIDE: every mini-batch is announced by both halves of the walk)
    if (!WIDE && k > 0 && !wait_at_least(w_walked, done + 1, p.status, s_flag, p.wait_limit)) return false;
    TTT_STAGE(BS_X_GROUP);
    const size_t ofin = uni64(((size_t)bh * 2 + (done & 1)) * cgs);
    const size_t o_img = uni64((size_t)bh * cgs * (CS * HID)), o_tile = uni64((size_t)bh * cgs * (CS * FD));
    const gptr_t gIMG2 = gbuf((set ? p.alt_grad_l_wrt_Z1_group[set - 1] : p.grad_l_wrt_Z1_group) + o_img);   // W2 after each step
    const gptr_t gGZ2 = gbuf((set ? p.alt_grad_l_wrt_Z2_group[set - 1] : p.grad_l_wrt_Z2_group) + o_tile);   // dl/dZ2
    // gelu'(Z1) images, or (without IMG) the images of Z1
    const gptr_t gDD = IMG ? gbuf((set ? p.alt_W1_init_group[set - 1] : p.W1_init_group) + uni64((size_t)bh * cgs * (FD * HID)))
                           : gbuf((set ? p.alt_Z1_group[set - 1] : p.Z1_group) + o_img);
    const gptr_t gGZ1B = gbuf((set ? p.alt_Z1_bar_group[set - 1] : p.Z1_bar_group) + uni64((size_t)bh * cgs * (CS * HID)));
    const gptr_t gDZ = gbuf(p.fin_dz + ofin * (CS * HID)), gGY = gbuf(p.fin_gy + ofin * (2 * CS * FD));
    const gptr_t gIMG1 = gbuf((set ? p.alt_X2_group[set - 1] : p.X2_group) + uni64((size_t)bh * cgs * (CS * HID)));
    const unsigned ckW = static_cast<unsigned>(k) * (FD * HID * 4u);
    // What a mini-batch takes from the replay's images and the inputs is asked for during the mini-batch before it, each operand
    // as soon as its registers are free (the first mini-batch of a group: here): fetched where it is used, this workgroup
    // spent 18 k of its 22 k clocks per mini-batch waiting, and the walk on two CUs is faster than that.
    u32x4 xq, xk, gz;
    bf16 eta_n[2];
    bf16x8 g1b[4];   // gZ1_bar^T of the output branch: lane = hid, contraction = tok
    bf16x8 w2bf[4];  // W2 before the step: lane = hid, contraction = F
    bf16x8 d1[2][2], w1b[2][2];
    auto ask_tiles = [&](int jn) {
      FIN_LANE;
      const unsigned xo = (k * cgs + jn) * TILE_BYTES;
      xq = g_ld_stream<u32x4>(gXQ, t16, xo);
      xk = g_ld_stream<u32x4>(gXK, t16, xo);
      gz = g_ld_stream<u32x4>(gGZ2, t16, jn * TILE_BYTES);
      eta_n[0] = g_ldh(gETA, 2 * c, (k * cgs + jn) * (CS * 2) + 64 * tb[0]);
      eta_n[1] = g_ldh(gETA, 2 * c, (k * cgs + jn) * (CS * 2) + 64 * tb[1]);
    };
    auto ask_g1b = [&](int jn) {
      FIN_LANE;
#pragma unroll
      for (int s = 0; s < 4; s++) g1b[s] = image_load(gGZ1B, jn * IMG_BYTES, s, t16);
    };
    auto ask_w2 = [&](int jn) {
      FIN_LANE;
      if (jn > 0) {
#pragma unroll
        for (int s = 0; s < 4; s++) w2bf[s] = image_load(gIMG2, (jn - 1) * IMG_BYTES, s, t16);
      } else {
#pragma unroll
        for (int s = 0; s < 4; s++) w2bf[s] = piece_from_f32(gCW2, ckW, FD, hid0, 0, s, c, h);
      }
    };
    auto ask_d1 = [&](int jn) {   // gelu'(Z1)
      FIN_LANE;
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int t = 0; t < 2; t++) d1[a][t] = image_load(gDD, jn * (IMG ? 2 * IMG_BYTES : IMG_BYTES), 2 * tb[a] + t, t16);
    };
    auto ask_w1 = [&](int jn) {   // W1 before the step
      FIN_LANE;
      if (jn > 0) {
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
          for (int t = 0; t < 2; t++) w1b[a][t] = image_load(gIMG1, (jn - 1) * IMG_BYTES, 2 * a + t, t16);
      } else {
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
          for (int t = 0; t < 2; t++) w1b[a][t] = piece_from_f32(gCW1, ckW, HID, 32 * a, hid0, t, c, h);
      }
    };
    for (int j = n_mb - 1; j >= 0; j--) {
      const int jn = j > 0 ? j - 1 : 0;
      FIN_LANE;
      if constexpr (WIDE) {
        if (++n_step > n_seen) {
          n_seen = wait_for_both(w_sync + BWW_GIVEN, w_sync + BWW_GIVEN + 4, n_step, p.status, s_flag, p.wait_limit);
          if (n_seen < 0) return false;
        }
        TTT_STAGE(BS_X_GROUP);
      } else if (k == 0 && (j == n_mb - 1 || (j & (FIN_CHUNK - 1)) == FIN_CHUNK - 1)) {
        if (!wait_at_least(w_sync + 12, n_mb - (j & ~(FIN_CHUNK - 1)), p.status, s_flag, p.wait_limit)) return false;
        TTT_STAGE(BS_X_GROUP);
      }
      if (j == n_mb - 1) {   // the group's norm-gradient sum, or its eighths': published with it, and the walk has acquired it
        const float* np = p.norm_partial + ((size_t)bh * BWD_MAX_SETS + set) * (8 * BW_NWAVE * 2 * FD) + v * 2 * FD + lane;
        const int eighth = (cgs + 7) / 8;
        float a0 = np[0], a1 = np[FD];
        for (int e = 1; EIGHTHS && e * eighth < n_mb; e++) {
          a0 += np[e * (BW_NWAVE * 2 * FD)];
          a1 += np[e * (BW_NWAVE * 2 * FD) + FD];
        }
        nr0 += a0;
        nr1 += a1;
        ask_tiles(j);
        ask_g1b(j);
        ask_w2(j);
        ask_d1(j);
        ask_w1(j);
      }
      const unsigned xo = (k * cgs + j) * TILE_BYTES, so = j * TILE_BYTES, ho = j * IMG_BYTES;
      const bf16x8 dxk_ld = g_ld_stream<bf16x8>(p.overwrite ? gbuf(zero_tile) : gDXK, vln, p.overwrite ? 0u : xo);
      const bf16x8 dxv_ld = g_ld_stream<bf16x8>(p.overwrite ? gbuf(zero_tile) : gDXV, vln, p.overwrite ? 0u : xo);
      const f32x4 gy_lo = g_ld_stream<f32x4>(gGY, 2 * vln, 4 * so), gy_hi = g_ld_stream<f32x4>(gGY, 2 * vln + 16, 4 * so);
      const f32x4 dg_lo = g_ld_stream<f32x4>(gGY, 2 * vln, 4 * so + 2 * TILE_BYTES);
      const f32x4 dg_hi = g_ld_stream<f32x4>(gGY, 2 * vln + 16, 4 * so + 2 * TILE_BYTES);
      bf16x8 g1[2][2], dz[2][2];
#pragma unroll
      for (int a = 0; a < 2; a++)
#pragma unroll
        for (int t = 0; t < 2; t++) dz[a][t] = image_load(gDZ, ho, 2 * tb[a] + t, t16);
      const float eta_i[2] = {bf2f(eta_n[0]), bf2f(eta_n[1])};
      lds_put16x(s_xq, tid, xq);
      lds_put16x(s_xk, tid, xk);
      lds_put16(s_gz2, tid, gz);
      ask_tiles(jn);
      __syncthreads();
      {
      FIN_LANE;
      mma_jit<4>(gW1s, [&](int fb, int s) { return xpiece_tr(s_xq, fb, s, lane); },         // + XQ^T gZ1_bar
                 [&](int, int s) { return g1b[s]; });
      ask_g1b(jn);
      }
      AccT<2, 2> dk;
      {
      FIN_LANE;
      store_state_rows<LDF>(T2, gW1s, c, h);                                                  // gW1 rows [hid][F]
#pragma unroll
      for (int s = 0; s < 4; s++) store_piece_rows<LDF>(T1, 0, s, c, h, w2bf[s]);            // W2 before the step, rows [hid][F]
      ask_w2(jn);
      WAVE_SYNC();
      acc_zero(dk);
#pragma unroll
      for (int i = 0; i < 2; i++) {
        // G1 = -eta * dl/dZ1 with dl/dZ1 = (gZ2 W2^T) * gelu'(Z1), as the walk forms it
        AccT<1, 1> R;
        acc_zero(R);
        mma_jit<4>(R, [&](int, int s) { return piece_rows<LDF>(T1, 0, s, c, h); },
                   [&](int, int s) { return piece_rows<LDX>(s_gz2, tb[i], s, c, h); });
#pragma unroll
        for (int t = 0; t < 2; t++) {
#pragma unroll
          for (int jj = 0; jj < 8; jj++) {
            float a = (float)d1[i][t][jj];
            if constexpr (!IMG) {
              float g, b;
              gelu_fdd(a, g, a, b);
              a = (float)(bf16)a;
            }
            const float gz1 = R.b[0][0][8 * t + jj] * a;
            g1[i][t][jj] = (bf16)(-eta_i[i] * gz1);
          }
#pragma unroll
          for (int rb = 0; rb < 2; rb++) dk.b[rb][i] = MFMA(piece_tr<LDF>(T2, rb, t, lane), g1[i][t], dk.b[rb][i]);
        }
      }
      ask_d1(jn);
      }
      {
      FIN_LANE;
      WAVE_SYNC();   // the readers of T1 (W2 rows) are done
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int t = 0; t < 2; t++) store_piece_rows<LDH>(T1, tb[i], t, c, h, dz[i][t]);     // dZ1 rows [tok][hid]
      WAVE_SYNC();
      mma_jit<2>(dk, [&](int rb, int s) { return w1b[rb][s]; }, [&](int i, int s) { return dz[i][s]; });
      ask_w1(jn);
      mma_jit<4>(gW1s, [&](int fb, int s) { return xpiece_tr(s_xk, fb, s, lane); },         // + XK^T dZ1
                 [&](int, int s) { return piece_tr<LDH>(T1, 0, s, lane); });
      WAVE_SYNC();   // this wave's readers of T1 / T2 are done
      TTT_STAGE(BS_X_PRODUCTS);
      pair_sum(s_own, s_partner, dk, c, h);
      }
      float z[8];
      ln_gather(z, s_lnrow);
      const float gyv[8] = {gy_lo[0], gy_lo[1], gy_lo[2], gy_lo[3], gy_hi[0], gy_hi[1], gy_hi[2], gy_hi[3]};
      const float dgv[8] = {dg_lo[0], dg_lo[1], dg_lo[2], dg_lo[3], dg_hi[0], dg_hi[1], dg_hi[2], dg_hi[3]};
      float dxv_new[8];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        z[e] = (float)dxk_ld[e] + (z[e] + gyv[e]);
        dxv_new[e] = (float)dxv_ld[e] - gyv[e];                         // dXV accumulates -g_y
      }
      g_st_stream<bf16x8>(gDXK, vln, xo, cvt8(z));
      g_st_stream<bf16x8>(gDXV, vln, xo, cvt8(dxv_new));
      ln_token_sum_add(s_dgw, dgv, lane, f0);
      ln_token_sum_add(s_dbw, gyv, lane, f0);
      __syncthreads();   // the readers of the pair sums are done before the next mini-batch's take their place
      TTT_STAGE(BS_X_SUMS);
    }
    if (!OWN && k > 0) {   // another workgroup goes on with the next group
      FIN_LANE;
      acc_store_rows(gW1s, gbuf(park), 0, HID, 0, hid0, c, h);
      float* const q = park + FD * HID + v * 4 * FD + lane;
      q[0] = s_dgw[lane]; q[FD] = s_dbw[lane]; q[2 * FD] = nr0; q[3 * FD] = nr1;
    }
    publish(w_finished, done + 1);
    TTT_STAGE(BS_PUBLISH);
  } while (OWN && --k >= 0);
  TTT_STAGES_END(bh, STAGE_ROLE_DXK);
  if (!OWN && k > 0) return true;
  // norm-weight / norm-bias gradients: the replay's sum + the walk's, in the order of the other launch shapes
  __syncthreads();
  s_P[v * 2 * FD + lane] = nr0;
  s_P[v * 2 * FD + FD + lane] = nr1;
  __syncthreads();
  if (tid < 2 * FD) {
    const int which = tid / FD, f = tid % FD;
    float s = 0.f, sr = 0.f;
#pragma unroll
    for (int u = 0; u < BW_NWAVE; u++) {
      s += s_red[(u * 2 + which) * FD + f];
      sr += s_P[(u * 2 + which) * FD + f];
    }
    (which == 0 ? p.grad_L_ttt_norm_weight : p.grad_L_ttt_norm_bias)[(size_t)bh * FD + f] = sr + s;
  }
  return true;
}
#undef FIN_LANE

#ifndef TTT_BWD_ROLES_ONLY
// NREPLAY + 1 workgroups per (batch, head): one walks.  Workgroups are dealt to the 8 XCDs in turn, so with a
// multiple of 8 (batch, head) pairs the workgroups of a pair are placed 8 apart: same XCD, same L2.
template <int NREPLAY>
__global__ __launch_bounds__(BW_THREADS) void ttt_mlp_bwd_split_kernel(const BwdParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int PER = NREPLAY + 1;
  constexpr bool IMG = NREPLAY == 2;   // two replaying workgroups also evaluate the GELU family for the walk
  const int b = blockIdx.x;
  int bh, role;
  if (p.nbh % 8 == 0) {
    bh = (b / (8 * PER)) * 8 + (b & 7);
    role = (b >> 3) % PER;
  } else {
    bh = b / PER;
    role = b % PER;
  }
  bh += p.bh0;
  if (role == NREPLAY) {
    bwd_body<2, IMG, false>(p, smem, bh, p.K - 1, 0);
    return;
  }
  for (int k = p.K - 1 - role; k >= 0; k -= NREPLAY)
    if (!bwd_body<1, IMG, false>(p, smem, bh, k, k)) return;
}

// nbh workgroups with a pair each, n_helpers that replay for them.
__global__ __launch_bounds__(BW_THREADS) void ttt_mlp_bwd_helped_kernel(const BwdParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int b = blockIdx.x;
  if (b < p.nbh) {
    bwd_body<0, false, false, false, false, true>(p, smem, p.bh0 + b, p.K - 1, 0);
    return;
  }
  int* const job = reinterpret_cast<int*>(smem + SB_FLAG);
  const int me = uni((b - p.nbh) * (p.nbh / p.n_helpers));
  while (help_take(p, me, job)) {
    const int k = uni(p.K - 1 - job[1]);
    bwd_body<1, false, false, false, false, true>(p, smem, uni(p.bh0 + job[0]), k, k, uni(job[2]));
  }
}

__global__ void ttt_mlp_zero_words(int* w, int n, const int* report) { clear_word(w, n, blockIdx.x * blockDim.x + threadIdx.x, report); }

}  // namespace ttt

extern "C" int ttt_mlp_bwd_threads() { return ttt::BW_THREADS; }
extern "C" int ttt_mlp_bwd_lds_bytes() { return ttt::SM_BWD_BYTES; }

hipError_t ttt_mlp_bwd_enqueue(const ttt::BwdParams& p, TttKernel kernel, int grid, hipStream_t stream) {
  auto launch = [&](auto k) -> hipError_t {
    if (p.sync != nullptr) {
      const int n = static_cast<int>(ttt::bwd_sync_ints(p.nbh));
      int* const words = p.status - (size_t)p.nbh * ttt::BWD_SYNC_STRIDE;   // p.sync itself is moved back by bh0 entries
      hipLaunchKernelGGL(ttt::ttt_mlp_zero_words, dim3((n + 255) / 256), dim3(256), 0, stream, words, n, p.report);
    }
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, ttt::SM_BWD_BYTES);   // (while that runs)
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k, dim3(grid), dim3(ttt::BW_THREADS), ttt::SM_BWD_BYTES, stream, p);
    return hipGetLastError();
  };
  switch (kernel) {
    TTT_BWD_KERNELS(TTT_KERNEL_LAUNCH)
    default: return hipErrorInvalidValue;
  }
}
#else
}  // namespace ttt
#endif
