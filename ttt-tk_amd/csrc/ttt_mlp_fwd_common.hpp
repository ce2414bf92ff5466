// What the forward kernels share: LDS carve-up, pair sums, the two LayerNorm stages and the output branch.
#pragma once
#include "ttt_mlp_common.hpp"
#include "ttt_mlp_kernels.hpp"

namespace ttt {

constexpr int FW_NWAVE = 8;
constexpr int FW_THREADS = 64 * FW_NWAVE;
constexpr int FW_NS = HID / FW_NWAVE;                  // hidden columns per wave: 32
// Row stride (elements) of every bf16 tile in LDS.  136-byte rows put the 32 row-wise 8-byte reads of
// an operand piece on 64 distinct banks (measured: 8.6 clocks per piece against 16 with 144-byte
// rows); rows are 8-byte aligned, so 16-byte accesses are made as two 8-byte ones.
constexpr int FLD = 68;
#define MFMA(a, b, c) __builtin_amdgcn_mfma_f32_32x32x16_bf16((a), (b), (c), 0, 0, 0)
TTT_DEV OpdT<2, 4> x_rows_kappa(const bf16* tile, int c, int h) {
  OpdT<2, 4> o;
#pragma unroll
  for (int fb = 0; fb < 2; fb++)
#pragma unroll
    for (int s = 0; s < 4; s++) o.v[fb][s] = xpiece_rows(tile, fb, s, c, h);
  return o;
}

// LDS carve-up (bytes)
constexpr int SM_TILE = 64 * FLD * 2;                   // one bf16 tile: 8704
static_assert(32 * 132 * 2 <= SM_TILE, "a tile of row pairs fits a tile slot");
constexpr int SM_XQ = 0;                                // two buffers, alternating per mini-batch
constexpr int SM_XK = SM_XQ + 2 * SM_TILE;
constexpr int SM_XV = SM_XK + SM_TILE;
constexpr int SM_G2 = SM_XV + SM_TILE;
constexpr int SM_G2L = SM_G2 + SM_TILE;                  // low-order bf16 term of G2
constexpr int SM_P = SM_G2L + SM_TILE;                   // 4 fp32 pair-sum tiles [tok][F]
constexpr int SM_PTILE = 64 * LDP * 4;
constexpr int SM_X2T = SM_P + 4 * SM_PTILE;             // per wave: X2 shard stored [hid][tok], bf16
constexpr int SM_X2T_TILE = FW_NS * FLD * 2;
constexpr int SM_B1 = SM_X2T + FW_NWAVE * SM_X2T_TILE;
constexpr int SM_B2 = SM_B1 + HID * 4;
constexpr int SM_ETA = SM_B2 + FD * 4;
constexpr int SM_GAM = SM_ETA + CS * 4;
constexpr int SM_BET = SM_GAM + FD * 4;
constexpr int SM_B2P = SM_BET + FD * 4;                  // per wave: the sum of G2 over its 8 LayerNorm tokens (the step of b2)
constexpr int SM_FLAG = SM_B2P + FW_NWAVE * FD * 4;      // outcome of a wait on the other workgroup
constexpr int SM_FWD_BYTES = SM_FLAG + 16;
static_assert(SM_FWD_BYTES <= 160 * 1024, "forward LDS budget");

// 16 bytes to / from an 8-byte aligned LDS address.
TTT_DEV void lds_put16(void* p, u32x4 v) {
  uint2* d = reinterpret_cast<uint2*>(p);
  d[0] = make_uint2(v[0], v[1]);
  d[1] = make_uint2(v[2], v[3]);
}
TTT_DEV bf16x8 lds_get8h(const bf16* p) { return cat(*reinterpret_cast<const bf16x4*>(p), *reinterpret_cast<const bf16x4*>(p + 4)); }

struct Staged {  // one mini-batch of inputs in flight from HBM: one 16-byte chunk per tile per thread
  u32x4 q, k, v;
  bf16 eta;
};

// gq / gk / gv / ge = this (batch, head)'s XQ, XK, XV, last_eta; thread tid moves 16-byte chunk tid
// (row tid / 8, 8 chunks per row) of each tile of mini-batch mb.
constexpr unsigned TILE_BYTES = CS * FD * 2;
TTT_DEV void stage_load(Staged& s, gptr_t gq, gptr_t gk, gptr_t gv, gptr_t ge, int mb, int tid) {
  s.q = g_ld16(gq, 16 * tid, mb * TILE_BYTES);
  s.k = g_ld16(gk, 16 * tid, mb * TILE_BYTES);
  s.v = g_ld16(gv, 16 * tid, mb * TILE_BYTES);
  s.eta = g_ldh(ge, 2 * (tid & (CS - 1)), mb * (CS * 2));   // threads >= CS drop it
}

TTT_DEV void stage_store(const Staged& s, unsigned char* smem, int xq_buf, int tid) {
  const int off = (xrow(tid >> 3) + (tid & 7) * 8) * 2;
  lds_put16(smem + SM_XQ + xq_buf * SM_TILE + off, s.q);
  lds_put16(smem + SM_XK + off, s.k);
  lds_put16(smem + SM_XV + off, s.v);
  if (tid < CS) reinterpret_cast<bf16*>(smem + SM_ETA)[tid] = s.eta;   // eta stays bf16 in LDS
}

// Two-step sum over the wave pair (v, v ^ 4) of a partial tile z (rows F, columns tok): the wave
// with pair index r gives away row block 1-r, then adds the partner's row block r to its own and
// leaves the pair sum in the pair's LDS tile, stored [tok][F].  Contains two workgroup barriers.
template <int R>
TTT_DEV void pair_give(float* tile, const AccT<2, 2>& z, int c, int h) {
#pragma unroll
  for (int cb = 0; cb < 2; cb++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const f32x16& x = z.b[1 - R][cb];
      f32x4 v = {x[4 * g], x[4 * g + 1], x[4 * g + 2], x[4 * g + 3]};
      *reinterpret_cast<f32x4*>(tile + (32 * cb + c) * LDP + 32 * (1 - R) + 8 * g + 4 * h) = v;
    }
}
template <int R>
TTT_DEV void pair_take(float* tile, const AccT<2, 2>& z, int c, int h) {
#pragma unroll
  for (int cb = 0; cb < 2; cb++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      float* q = tile + (32 * cb + c) * LDP + 32 * R + 8 * g + 4 * h;
      const f32x16& x = z.b[R][cb];
      f32x4 v = *reinterpret_cast<const f32x4*>(q);
      v[0] += x[4 * g]; v[1] += x[4 * g + 1]; v[2] += x[4 * g + 2]; v[3] += x[4 * g + 3];
      *reinterpret_cast<f32x4*>(q) = v;
    }
}
TTT_DEV void pair_sum_to_lds(float* tile, const AccT<2, 2>& z, int r, int c, int h) {
  if (r == 0) pair_give<0>(tile, z, c, h); else pair_give<1>(tile, z, c, h);
  __syncthreads();
  if (r == 0) pair_take<0>(tile, z, c, h); else pair_take<1>(tile, z, c, h);
  __syncthreads();
}

// The same sum with the product formed one F block at a time - `half(rb)` returns rows [32 rb, 32 rb + 32) of
// the partial tile - so that 32 accumulator registers are live instead of 64: first the block that is given away,
// then the one that is kept.
template <int R, class HALF>
TTT_DEV void pair_sum_halves_r(float* tile, HALF half, int c, int h) {
  {
    const AccT<1, 2> z = half(1 - R);
#pragma unroll
    for (int cb = 0; cb < 2; cb++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const f32x16& x = z.b[0][cb];
        f32x4 v = {x[4 * g], x[4 * g + 1], x[4 * g + 2], x[4 * g + 3]};
        *reinterpret_cast<f32x4*>(tile + (32 * cb + c) * LDP + 32 * (1 - R) + 8 * g + 4 * h) = v;
      }
  }
  const AccT<1, 2> z = half(R);
  __syncthreads();
#pragma unroll
  for (int cb = 0; cb < 2; cb++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      float* q = tile + (32 * cb + c) * LDP + 32 * R + 8 * g + 4 * h;
      const f32x16& x = z.b[0][cb];
      f32x4 v = *reinterpret_cast<const f32x4*>(q);
      v[0] += x[4 * g]; v[1] += x[4 * g + 1]; v[2] += x[4 * g + 2]; v[3] += x[4 * g + 3];
      *reinterpret_cast<f32x4*>(q) = v;
    }
  __syncthreads();
}
template <class HALF0, class HALF1>
TTT_DEV void pair_sum_halves(float* tile, HALF0 half0, HALF1 half1, int r, int c, int h) {
  // half0 / half1: the product's F block 0 / 1 (two callables so that each indexes the state registers statically)
  if (r == 0) pair_sum_halves_r<0>(tile, [&](int rb) { return rb == 0 ? half0() : half1(); }, c, h);
  else pair_sum_halves_r<1>(tile, [&](int rb) { return rb == 0 ? half0() : half1(); }, c, h);
}

// Output LayerNorm + residual for 8 features of a token: XQ + LN(z).  8 lanes per token.
TTT_DEV bf16x8 output_layernorm_row(float (&z)[8], const float* s_gam, const float* s_bet, const bf16x8 qv) {
  float sum = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) sum += z[e];
  const float mu = oct_sum(sum) * (1.f / FD);
  float var = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) { z[e] -= mu; var = __builtin_fmaf(z[e], z[e], var); }
  const float rstd = __builtin_amdgcn_rsqf(oct_sum(var) * (1.f / FD) + LN_EPS);
  float gam[8], bet[8];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const f32x4 gq = *reinterpret_cast<const f32x4*>(s_gam + 4 * q);
    const f32x4 bq = *reinterpret_cast<const f32x4*>(s_bet + 4 * q);
#pragma unroll
    for (int e = 0; e < 4; e++) { gam[4 * q + e] = gq[e]; bet[4 * q + e] = bq[e]; }
  }
  bf16x8 o;
#pragma unroll
  for (int e = 0; e < 8; e++) o[e] = (bf16)(bf2f(qv[e]) + __builtin_fmaf(gam[e], z[e] * rstd, bet[e]));
  return o;
}

// Out = XQ + LN(sum of the four pair sums + b2) for the features [f0, f0+8) of token `tok`; 8 tokens per wave.
TTT_DEV void output_layernorm(const float* s_P, const float* s_b2, const float* s_gam, const float* s_bet,
                              const bf16* s_xq, gptr_t gOut, int mb, int tok, int f0) {
  float z[8];
  {
    f32x4 a0 = *reinterpret_cast<const f32x4*>(s_b2 + f0);
    f32x4 a1 = *reinterpret_cast<const f32x4*>(s_b2 + f0 + 4);
#pragma unroll
    for (int t = 0; t < 4; t++) {
      a0 += *reinterpret_cast<const f32x4*>(s_P + t * 64 * LDP + tok * LDP + f0);
      a1 += *reinterpret_cast<const f32x4*>(s_P + t * 64 * LDP + tok * LDP + f0 + 4);
    }
#pragma unroll
    for (int e = 0; e < 4; e++) { z[e] = a0[e]; z[4 + e] = a1[e]; }
  }
  const bf16x8 o = output_layernorm_row(z, s_gam + f0, s_bet + f0, lds_get8h(s_xq + xrow(tok) + f0));
  g_st8h(gOut, (tok * FD + f0) * 2, mb * TILE_BYTES, o);
}

// LayerNorm-fused gradient of the reconstruction loss for the 8 features of this lane's token (8 lanes per token):
// z = Z2 in, target = XV - XK; gx times the returned scale is G2 = -eta * dl/dZ2.
TTT_DEV float ln_loss_gradient(float (&z)[8], const float (&target)[8], const float eta, const float* s_gam, const float* s_bet,
                              float (&gx)[8]) {
  float sum = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) sum += z[e];
  const float mu = oct_sum(sum) * (1.f / FD);
  float var = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) { z[e] -= mu; var = __builtin_fmaf(z[e], z[e], var); }
  const float rstd = __builtin_amdgcn_rsqf(oct_sum(var) * (1.f / FD) + LN_EPS);
  float gam[8], bet[8];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const f32x4 gq = *reinterpret_cast<const f32x4*>(s_gam + 4 * q);
    const f32x4 bq = *reinterpret_cast<const f32x4*>(s_bet + 4 * q);
#pragma unroll
    for (int e = 0; e < 4; e++) { gam[4 * q + e] = gq[e]; bet[4 * q + e] = bq[e]; }
  }
  float s1 = 0.f, s2 = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const float xh = z[e] * rstd;
    const float go = __builtin_fmaf(gam[e], xh, bet[e]) - target[e];
    z[e] = xh;
    gx[e] = go * gam[e];
    s1 += gx[e];
    s2 = __builtin_fmaf(gx[e], xh, s2);
  }
  s1 = oct_sum(s1);
  s2 = oct_sum(s2);
  const float scale = -eta * rstd * (1.f / FD);
#pragma unroll
  for (int e = 0; e < 8; e++) gx[e] = FD * gx[e] - s1 - z[e] * s2;
  return scale;
}

TTT_DEV float ln_loss_gradient(float (&z)[8], const bf16x8 kv, const bf16x8 vv, const float eta, const float* s_gam, const float* s_bet,
                              float (&gx)[8]) {
  float target[8];
#pragma unroll
  for (int e = 0; e < 8; e++) target[e] = bf2f(vv[e]) - bf2f(kv[e]);
  return ln_loss_gradient(z, target, eta, s_gam, s_bet, gx);
}

// Everything derived from the lane index is cheap to recompute and expensive to keep in a register
// (or spilled) for the whole scan: LANE_VARS re-derives it from a lane index the optimiser cannot see
// through, so each stage that opens with it gets fresh, short-lived copies.
#define LANE_VARS                                                               \
  asm volatile("" : "+v"(lane_v));                                              \
  const int lane = lane_v, h = lane >> 5, c = lane & 31, tid = (v << 6) | lane; \
  const int tok = 8 * v + (lane >> 3), f0 = 8 * (lane & 7);                     \
  (void)h; (void)c; (void)tid; (void)tok; (void)f0

// The output branch of the forward on its own workgroup: Out[mb] = XQ + LN(gelu(XQ W1' + b1') W2' + b2')
// with the state after mini-batch mb, taken from the operand images the recurrence leaves behind.  Nothing
// is carried from one mini-batch to the next here.
// WIDE: the recurrence runs on two workgroups, which hand over every mini-batch (RING = 1).
template <int RING, bool WIDE>
TTT_DEV void fwd_output_branch(const FwdParams& p, unsigned char* smem, const int bh) {
  float* s_P = reinterpret_cast<float*>(smem + SM_P);
  float* s_b1 = reinterpret_cast<float*>(smem + SM_B1);
  float* s_b2 = reinterpret_cast<float*>(smem + SM_B2);   // two buffers: the second takes the place of the eta vector
  static_assert(SM_ETA == SM_B2 + FD * 4, "the second b2 buffer aliases the eta vector");
  float* s_gam = reinterpret_cast<float*>(smem + SM_GAM);
  float* s_bet = reinterpret_cast<float*>(smem + SM_BET);
  const int tid = threadIdx.x, lane = tid & 63;
  const int v = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pr = v >> 2;
  const int head = bh % p.NH;
  const int hid0 = FW_NS * v;
  float* s_Pp = s_P + (v & 3) * 64 * LDP;
  int lane_v = lane;
  if (tid < FD) {
    s_gam[tid] = p.ttt_norm_weight[head * FD + tid];
    s_bet[tid] = p.ttt_norm_bias[head * FD + tid];
  }
  const size_t x_base = uni64((size_t)bh * p.NC * (CS * FD));
  const gptr_t gXQ = gbuf(p.XQ + x_base), gOut = gbuf(p.Out + x_base);
  int* const w_given = p.sync + (size_t)bh * BWD_SYNC_STRIDE;
  int* const w_taken = w_given + 16;
  int* const w_status = p.status;
  int* const s_flag = reinterpret_cast<int*>(smem + SM_FLAG);

  TTT_STAGES_BEGIN();
  for (int mb = 0; mb < p.NC; mb++) {
    LANE_VARS;
    constexpr int ring = RING; const int grp = mb / ring, at = mb % ring, slot = WIDE ? mb % FWD_WIDE_RING : (grp & 1) * ring + at;
    const int buf = mb & 1;
    if (at == 0) {
      if (!wait_at_least(w_given, grp + 1, w_status, s_flag, p.wait_limit)) return;
      if (WIDE && !wait_at_least(w_given + 8, grp + 1, w_status, s_flag, p.wait_limit)) return;
    }
    bf16* s_xq = reinterpret_cast<bf16*>(smem + SM_XQ + buf * SM_TILE);
    const size_t at_slot = WIDE ? (size_t)bh * FWD_WIDE_RING + slot : (size_t)bh * 2 * FWD_RING_MAX + slot;
    const gptr_t gImg = gbuf(p.state_img + at_slot * (FWD_IMG_BYTES / 2));
    const float* gB = p.bias_img + at_slot * FWD_BIAS_FLOATS;
    {
      LANE_VARS;
      // XQ and b2 alternate between two LDS buffers: other waves may still be in the previous mini-batch's
      // LayerNorm, which reads both.  (b1 is read before the pair sum's barriers only.)
      const u32x4 q = g_ld16(gXQ, 16 * tid, mb * TILE_BYTES);
      float bv = 0.f;
      if (tid < FWD_BIAS_FLOATS) bv = gB[tid];
      lds_put16(smem + SM_XQ + buf * SM_TILE + (xrow(tid >> 3) + (tid & 7) * 8) * 2, q);
      if (tid < HID) s_b1[tid] = bv;
      else if (tid < FWD_BIAS_FLOATS) s_b2[buf * FD + tid - HID] = bv;
    }
    __syncthreads();   // XQ and the biases are visible; the previous mini-batch's readers of s_P are done
    TTT_STAGE(FS_TOP);
    {
      LANE_VARS;
      OpdT<1, 4> w1A;
      OpdT<2, 2> w2A;
#pragma unroll
      for (int s = 0; s < 4; s++) w1A.v[0][s] = g_ld_stream<bf16x8>(gImg, 16 * tid, s * 8192);
#pragma unroll
      for (int fb = 0; fb < 2; fb++)
#pragma unroll
        for (int s = 0; s < 2; s++) w2A.v[fb][s] = g_ld_stream<bf16x8>(gImg, 16 * tid, (4 + 2 * fb + s) * 8192);
      const OpdT<2, 4> xqB = x_rows_kappa(s_xq, c, h);
      AccT<1, 2> z1b;
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const f32x4 bv = *reinterpret_cast<const f32x4*>(s_b1 + hid0 + 8 * g + 4 * h);
#pragma unroll
        for (int cb = 0; cb < 2; cb++)
#pragma unroll
          for (int e = 0; e < 4; e++) z1b.b[0][cb][4 * g + e] = bv[e];
      }
      mma(z1b, w1A, xqB);
#pragma unroll
      for (int cb = 0; cb < 2; cb++)
#pragma unroll
        for (int i = 0; i < 16; i++) z1b.b[0][cb][i] = gelu_f(z1b.b[0][cb][i]);
      const OpdT<2, 2> x2bB = cvt_chain(z1b);      // lane = tok, contraction = hid
      AccT<2, 2> z2;
      acc_zero(z2);
      mma(z2, w2A, x2bB);                          // rows F, lane = tok
      pair_sum_to_lds(s_Pp, z2, pr, c, h);
    }
    TTT_STAGE(FS_OUT_FORWARD);
    {
      LANE_VARS;
      output_layernorm(s_P, s_b2 + buf * FD, s_gam, s_bet, s_xq, gOut, mb, tok, f0);
    }
    TTT_STAGE(FS_OUT_LN);
    if constexpr (WIDE) {   // every wave has read its operands (the pair sum's barriers are behind it); nothing else is ordered by this count
      if (threadIdx.x == 0) __hip_atomic_store(w_taken, mb + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else if (at == ring - 1 || mb == p.NC - 1) publish(w_taken, grp + 1);
    TTT_STAGE(FS_PUBLISH);
  }
  TTT_STAGES_END(bh, STAGE_ROLE_OUT);
}

}  // namespace ttt
