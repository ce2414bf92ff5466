// Forward scan with the recurrence of one (batch, head) spread over four CUs, which compute Out as well (up to an eighth of
// the CUs' number of pairs per XCD: 64 pairs on 256 CUs).
//
// Four workgroups of the same XCD hold one wave pair of the one-workgroup kernel each: the 64 hidden columns of its waves k and
// k + 4.  Inside a workgroup:
//   waves 0-3 (one per SIMD)  32 hidden columns (number w % 2 of the two) x 32 tokens (block w / 2): every matrix product.  Of the
//                             state of its columns a wave holds the half with the features of its block; a step forms that half, and
//                             the wave with the other block gets the bf16 terms of it through LDS
//   waves 4-7                 the sums over the hidden dimension, their exchange with the other CUs, the LayerNorm lanes
// so all 64 tokens of a mini-batch pass through the chain at once.  The sums of 16 tokens go to one CU, whose helpers normalise them
// and send G2 of them to the other three.  While the sums cross and are normalised, the compute waves form the output branch of the
// mini-batch before from the operands of the state that they hold anyway: no state leaves the CUs.  Its sums go to one CU per
// 16 tokens too, whose other two helpers finish Out a mini-batch later.
// Every sum has the order of the one-workgroup kernel - here CU k holds the whole of pair sum P_k - and results are the same
// to the bit.
//
// The exchange has no flags (ttt_mlp_exchange.hpp); slots are used in turn by mini-batch.  A message with one reader - sums, Out's sums -
// is marked empty again by it.  G2 and the shares of b2's step are written once and read by three CUs, so only their writer can do that:
// a CU that has the others' sums of mini-batch m knows that they have read its G2 of m - 1.  Marks are acknowledged before the
// barrier behind which the next mini-batch's sums and G2 are sent, and whoever writes a slot again, or reads it for another mini-batch,
// has received one of those first: with two slots for the sums and three for G2.  Out's last sums have no exchange behind
// them, hence three slots there as well.
//
// What bounds it: the chain of 11.2 k clocks per mini-batch (stage clocks, 12 pairs x 512): the new state's terms read back, Z1, GELU and
// partial sums 2.6 k, the sums gathered and sent 0.7 k, 1.2 k under way, LayerNorm 1.2 k, G2 under way 1.3 - 1.6 k, G1 and most of W2's step
// 1.5 k, W1's step and the split of the new state 1.5 k, barriers.  Against the recurrence on two CUs with two more for Out (14.2 k
// clocks, as many CUs): 2 pairs x 4 mini-batches 38.0 -> 29.1 us, 12 x 32 196 -> 162 us, 24 x 256 1.487 -> 1.216 ms, 48 x 256
// 1.519 -> 1.236, 64 x 256 1.533 -> 1.274, 48 x 1024 5.99 -> 4.86.
// What did not pay: all 64 tokens normalised on each of the four CUs, one exchange instead of two (12.2 k clocks: 48 KB to take per CU at
// 64 B a clock, and two tokens per lane); the output branch on the helper waves (14.7 k: they are what the step waits for then).
#pragma once
#include "ttt_mlp_exchange.hpp"
#include "ttt_mlp_fwd_common.hpp"

namespace ttt {

constexpr int QD_CUS = 4;
// LDS carve-up (bytes)
constexpr int QD_XK = 0;                                 // two buffers, alternating per mini-batch
constexpr int QD_XQ = QD_XK + 2 * SM_TILE;               // of the mini-batch before
constexpr int QD_G2 = QD_XQ + SM_TILE;
constexpr int QD_G2L = QD_G2 + SM_TILE;
constexpr int QD_X2T = QD_G2L + SM_TILE;                 // per shard: X2, [hid][tok], and its low-order term
constexpr int QD_X2L = QD_X2T + 2 * SM_X2T_TILE;
constexpr int QD_P = QD_X2L + 2 * SM_X2T_TILE;           // per compute wave: its partial sum, [32 tok][F] fp32; behind block
constexpr int QD_PTILE = 32 * LDP * 4;                   // sums' readers: the terms of G1 as operand pieces, [shard][term][4] of 1 KiB
constexpr int QD_OUT = QD_P + 4 * QD_PTILE;              // the same for Out; behind its readers: the terms of W1, the same way
constexpr int QD_W2T = QD_OUT + 4 * QD_PTILE;            // per shard: the two terms of W2 as [F][hid], row stride QD_LDT elements
constexpr int QD_LDT = 36;
constexpr int QD_W2TILE = FD * QD_LDT * 2;
constexpr int QD_B1 = QD_W2T + 4 * QD_W2TILE;            // [shard][32]
constexpr int QD_COLSUM = QD_B1 + 2 * FW_NS * 4;         // [shard][64 lanes]: the step of b1, block 0's share
constexpr int QD_GAM = QD_COLSUM + 2 * 64 * 4;
constexpr int QD_BET = QD_GAM + FD * 4;
constexpr int QD_B2 = QD_BET + FD * 4;
constexpr int QD_B2P = QD_B2 + FD * 4;                   // [8 groups of 8 tokens][F]: shares of the step of b2
constexpr int QD_FLAG = QD_B2P + 8 * FD * 4;             // non-zero: a wait gave up
constexpr int QD_BYTES = QD_FLAG + 16;
static_assert(2 * 2 * 4 * 1024 <= 4 * QD_PTILE, "operand pieces in the place of partial sums");
static_assert(QD_BYTES <= SM_FWD_BYTES, "the launch asks for SM_FWD_BYTES");
// Words of the exchange (FWD_QUAD_XCHG_WORDS): the sums as [2 slots][to CU][from CU][2 halves of its 16 tokens][4 words][lane], Out's as [3 slots]
// .. the same, G2's terms as [3 slots][CU][2 halves][4 words][lane], shares of the step of b2 as [3 slots][CU][2 halves][lane].
constexpr int QD_XOUT = 2 * QD_CUS * QD_CUS * 512;
constexpr int QD_XG2 = QD_XOUT + 3 * QD_CUS * QD_CUS * 512;
constexpr int QD_XB2 = QD_XG2 + 3 * QD_CUS * 2 * 256;
static_assert(QD_XB2 + 3 * QD_CUS * 2 * 64 <= FWD_QUAD_XCHG_WORDS, "exchange of four CUs");
constexpr int QDW_XCD = 24;   // synchronisation words of a pair: 24 .. the XCD each workgroup runs on (+ 1)

TTT_DEV void fwd_quad_recurrence(const FwdParams& p, unsigned char* smem, const int bh, const int part) {
  bf16* const s_g2 = reinterpret_cast<bf16*>(smem + QD_G2);
  bf16* const s_g2l = reinterpret_cast<bf16*>(smem + QD_G2L);
  bf16* const s_xq = reinterpret_cast<bf16*>(smem + QD_XQ);
  float* const s_b1 = reinterpret_cast<float*>(smem + QD_B1);
  float* const s_gam = reinterpret_cast<float*>(smem + QD_GAM);
  float* const s_bet = reinterpret_cast<float*>(smem + QD_BET);
  float* const s_b2 = reinterpret_cast<float*>(smem + QD_B2);
  float* const s_b2p = reinterpret_cast<float*>(smem + QD_B2P);
  typedef __attribute__((address_space(3))) int* lint_t;
  const lint_t s_flag = (lint_t)reinterpret_cast<int*>(smem + QD_FLAG);
  auto flag = [&]() { return __hip_atomic_load(s_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, c = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave of the workgroup
  const bool compute = w < 4;
  const int head = bh % p.NH;

  int* const words = p.sync + (size_t)bh * BWD_SYNC_STRIDE;
  int* const w_status = p.status;
  if (tid == 0) say_xcd(words + QDW_XCD + part);
  if (tid < FD) {
    s_b1[tid] = p.b1[(size_t)bh * HID + FW_NS * (part + 4 * (tid >> 5)) + (tid & 31)];
    s_b2[tid] = p.b2[(size_t)bh * FD + tid];
    s_gam[tid] = p.ttt_norm_weight[head * FD + tid];
    s_bet[tid] = p.ttt_norm_bias[head * FD + tid];
  }
  if (tid == 0) *s_flag = 0;
  const size_t x_base = uni64((size_t)bh * p.NC * (CS * FD));

  if (compute) {
    const int sh = w & 1, tb = w >> 1;                      // shard of this CU's two; token block, and half of the features
    const int hid0 = FW_NS * (part + 4 * sh);
    f32x16 W1, W2;                                          // W1[32 tb .., hid0 ..] (rows F), W2[hid0 .., 32 tb ..] (rows hid)
    {
      const gptr_t gW1 = gbuf(p.W1 + (size_t)bh * FD * HID), gW2 = gbuf(p.W2 + (size_t)bh * HID * FD);
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int row = 8 * (i >> 2) + (i & 3);             // + 4h in the lane offset
        W1[i] = g_ldf(gW1, (4 * h * HID + c) * 4, ((32 * tb + row) * HID + hid0) * 4);
        W2[i] = g_ldf(gW2, (4 * h * FD + c) * 4, ((hid0 + row) * FD + 32 * tb) * 4);
      }
    }
    bf16* const s_x2t = reinterpret_cast<bf16*>(smem + QD_X2T + sh * SM_X2T_TILE);
    bf16* const s_x2l = reinterpret_cast<bf16*>(smem + QD_X2L + sh * SM_X2T_TILE);
    float* const s_Pw = reinterpret_cast<float*>(smem + QD_P + w * QD_PTILE);
    float* const s_Ow = reinterpret_cast<float*>(smem + QD_OUT + w * QD_PTILE);
    bf16* const t_hi = reinterpret_cast<bf16*>(smem + QD_W2T + sh * 2 * QD_W2TILE);
    bf16* const t_lo = t_hi + QD_W2TILE / 2;
    float* const s_cs = reinterpret_cast<float*>(smem + QD_COLSUM) + sh * 64;
    int lane_v = lane;
#define QD_LANE                                             \
  asm volatile("" : "+v"(lane_v));                          \
  const int lane = lane_v & 63, h = lane >> 5, c = lane & 31; \
  (void)h; (void)c
    // Operand piece s of term t (0: high order) of this shard, as it is.
    auto piece_at = [&](int base, int t, int s) {
      return reinterpret_cast<bf16x8*>(smem + base + ((sh * 2 + t) * 4 + s) * 1024) + lane_v;
    };
    // The terms of this wave's half of the state, for both waves of the shard.
    auto give_w1 = [&]() {
#pragma unroll
      for (int t = 0; t < 2; t++) {
        bf16x8 ph, pl;
        split8(W1, t, ph, pl);
        *piece_at(QD_OUT, 0, 2 * tb + t) = ph;
        *piece_at(QD_OUT, 1, 2 * tb + t) = pl;
      }
    };
    auto give_w2 = [&](int t) {
      QD_LANE;
      bf16x8 ph, pl;
      split8(W2, t, ph, pl);
      store_piece_rows<QD_LDT>(t_hi, tb, t, c, h, ph);
      store_piece_rows<QD_LDT>(t_lo, tb, t, c, h, pl);
    };
    bf16x8 w1h[4], w1l[4], w2h[2][2], w2l[2][2], xk[4];
    auto take_w1 = [&]() {
#pragma unroll
      for (int s = 0; s < 4; s++) w1l[s] = *piece_at(QD_OUT, 1, s);
#pragma unroll
      for (int s = 0; s < 4; s++) w1h[s] = *piece_at(QD_OUT, 0, s);
    };
    auto take_w2 = [&]() {
      QD_LANE;
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int fb = 0; fb < 2; fb++) {
          w2l[fb][s] = piece_rows<QD_LDT>(t_lo, fb, s, c, h);
          w2h[fb][s] = piece_rows<QD_LDT>(t_hi, fb, s, c, h);
        }
    };
    // XK of this wave's tokens in mini-batch m (lane = tok)
    auto load_xk = [&](int m) {
      QD_LANE;
      const bf16* const x = reinterpret_cast<const bf16*>(smem + QD_XK + (m & 1) * SM_TILE);
#pragma unroll
      for (int s = 0; s < 4; s++) xk[s] = xpiece_rows(x, tb, s, c, h);
    };
    auto store_partial = [&](float* tile, int fb, const f32x16& z) {
      QD_LANE;
#pragma unroll
      for (int g = 0; g < 4; g++) {
        f32x4 q = {z[4 * g], z[4 * g + 1], z[4 * g + 2], z[4 * g + 3]};
        *reinterpret_cast<f32x4*>(tile + c * LDP + 32 * fb + 8 * g + 4 * h) = q;
      }
    };
    // The output branch of the last mini-batch, whose state the operands are, up to this shard's share of the sum.
    auto output_partial = [&]() {
      QD_LANE;
      f32x16 z1;   // rows hid, lane = tok
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const f32x4 bv = *reinterpret_cast<const f32x4*>(s_b1 + FW_NS * sh + 8 * g + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; e++) z1[4 * g + e] = bv[e];
      }
#pragma unroll
      for (int s = 0; s < 4; s++) z1 = MFMA(w1h[s], xpiece_rows(s_xq, tb, s, c, h), z1);
#pragma unroll
      for (int i = 0; i < 16; i++) z1[i] = gelu_f(z1[i]);
      const bf16x8 x2[2] = {pack8(z1, 0), pack8(z1, 1)};
      f32x16 z[2];
#pragma unroll
      for (int fb = 0; fb < 2; fb++)
#pragma unroll
        for (int i = 0; i < 16; i++) z[fb][i] = 0.f;
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int fb = 0; fb < 2; fb++) z[fb] = MFMA(w2h[fb][s], x2[s], z[fb]);
#pragma unroll
      for (int fb = 0; fb < 2; fb++) store_partial(s_Ow, fb, z[fb]);
    };
    give_w1();
    give_w2(0);
    give_w2(1);
    __syncthreads();   // the flag is clear
    __syncthreads();   // XK of mini-batch 0, the state's terms, b1, norm parameters; the helpers know where the other workgroups are
    if (flag() != 0) return;
    load_xk(0);
    __builtin_amdgcn_s_setprio(1);
    TTT_STAGES_BEGIN();
    for (int mb = 0; mb < p.NC; mb++) {
      const bf16* const s_xk = reinterpret_cast<const bf16*>(smem + QD_XK + (mb & 1) * SM_TILE);
      float b1L;
      {
        QD_LANE;
        b1L = s_b1[FW_NS * sh + c];
      }
      __builtin_amdgcn_sched_barrier(0);   // (the accumulators are set while the operands are on their way)
      take_w1();
      f32x16 d1;
      {
        QD_LANE;
        // Z1 = XK W1 + b1 (rows tok, lane = hid)
        f32x16 x2;
#pragma unroll
        for (int i = 0; i < 16; i++) x2[i] = b1L;
#pragma unroll
        for (int s = 0; s < 4; s++) x2 = MFMA(xk[s], w1l[s], x2);
#pragma unroll
        for (int s = 0; s < 4; s++) x2 = MFMA(xk[s], w1h[s], x2);
        take_w2();
#pragma unroll
        for (int i = 0; i < 16; i++) {
          float g, d;
          gelu_fd(x2[i], g, d);
          x2[i] = g;
          d1[i] = d;
        }
#pragma unroll
        for (int t = 0; t < 2; t++) {
          bf16x8 ph, pl;
          split8_plain(x2, t, ph, pl);
          store_piece_rows<FLD>(s_x2t, 0, 2 * tb + t, c, h, ph);
          store_piece_rows<FLD>(s_x2l, 0, 2 * tb + t, c, h, pl);
        }
        TTT_WAVE_SYNC();
      }
      {
        QD_LANE;
        // Z2^T partial (rows F, lane = tok)
        bf16x8 xb[2];
#pragma unroll
        for (int s = 0; s < 2; s++) xb[s] = piece_tr<FLD>(s_x2t, tb, s, lane);
        f32x16 z[2];
#pragma unroll
        for (int fb = 0; fb < 2; fb++)
#pragma unroll
          for (int i = 0; i < 16; i++) z[fb][i] = 0.f;
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
          for (int o = 0; o < 2; o++)
#pragma unroll
            for (int fb = 0; fb < 2; fb++) z[fb] = MFMA(o == 0 ? w2l[fb][s] : w2h[fb][s], xb[s], z[fb]);
#pragma unroll
        for (int fb = 0; fb < 2; fb++) store_partial(s_Pw, fb, z[fb]);
      }
      __builtin_amdgcn_sched_barrier(0);
      TTT_STAGE(FQC_SUMS);
      __syncthreads();                                    // B1: the partial sums
      TTT_STAGE(FQC_B1);
      __builtin_amdgcn_sched_barrier(0);
      // While they cross and are normalised: the output branch, what the step takes that does not wait for them, checkpoints.
      if (mb > 0) output_partial();
      if (mb % p.cgs == 0) {   // checkpoint: the state before this mini-batch
        QD_LANE;
        const gptr_t gW1 = gbuf(p.W1_ck + uni64((size_t)bh * p.K * FD * HID)), gW2 = gbuf(p.W2_ck + uni64((size_t)bh * p.K * HID * FD));
        const int ck_slot = mb / p.cgs;
        const unsigned ck = static_cast<unsigned>(ck_slot) * (FD * HID * 4u);
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int row = 8 * (i >> 2) + (i & 3);
          g_stf(gW1, (4 * h * HID + c) * 4, ck + ((32 * tb + row) * HID + hid0) * 4, W1[i]);
          g_stf(gW2, (4 * h * FD + c) * 4, ck + ((hid0 + row) * FD + 32 * tb) * 4, W2[i]);
        }
        if (tb == 0 && h == 0) p.b1_ck[((size_t)bh * p.K + ck_slot) * HID + hid0 + c] = b1L;
      }
      bf16x8 wh[4], wl[4], xkt[4], xh[4], xl[4];
      __builtin_amdgcn_sched_barrier(0);   // (not ahead of what the helpers read)
      {
        QD_LANE;
#pragma unroll
        for (int s = 0; s < 4; s++) {
          wh[s] = piece_tr<QD_LDT>(t_hi, 0, s, lane);        // W2 with F contracted (lane = hid)
          wl[s] = piece_tr<QD_LDT>(t_lo, 0, s, lane);
          xkt[s] = xpiece_tr(s_xk, tb, s, lane);             // XK with tokens contracted (lane = F)
          xh[s] = piece_rows<FLD>(s_x2t, 0, s, c, h);        // X2 with tokens contracted (lane = hid)
          xl[s] = piece_rows<FLD>(s_x2l, 0, s, c, h);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      TTT_STAGE(FQC_OUTPUT);
      __syncthreads();                                    // B2: G2
      TTT_STAGE(FQC_B2);
      __builtin_amdgcn_sched_barrier(0);
      const int gone = flag();   // (asked for here, looked at behind G1)
      f32x16 g1;
      bf16x8 gh[4], gl[4];
      float colsum = 0.f;
      auto w2_product = [&](int k) {   // number k of the twelve of W2[shard, 32 tb ..] += X2^T G2
        const int s = k / 3, o = k % 3;
        W2 = MFMA(o == 0 ? xl[s] : xh[s], o == 1 ? gl[s] : gh[s], W2);
        asm volatile("" : "+v"(W2));   // (here, not in a row behind the vector instructions)
      };
      {
        QD_LANE;
        // G1 = (G2 W2^T) * gelu'(Z1) of this wave's tokens; W2's step, which does not need it, keeps the matrix pipe busy while it is split
#pragma unroll
        for (int i = 0; i < 16; i++) g1[i] = 0.f;
        bf16x8 ah[4], al[4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
          ah[s] = piece_rows<FLD>(s_g2, tb, s, c, h);
          al[s] = piece_rows<FLD>(s_g2l, tb, s, c, h);
        }
#pragma unroll
        for (int s = 0; s < 4; s++) {
          __builtin_amdgcn_sched_barrier(0);
          g1 = MFMA(al[s], wh[s], g1);
          g1 = MFMA(ah[s], wl[s], g1);
          g1 = MFMA(ah[s], wh[s], g1);
          __builtin_amdgcn_sched_barrier(0);
          gh[s] = piece_tr<FLD>(s_g2, tb, s, lane);          // G2 with tokens contracted (lane = F)
          gl[s] = piece_tr<FLD>(s_g2l, tb, s, lane);
        }
        bf16x8 g1h[2], g1l[2];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 8; k++) {
          w2_product(k);
          __builtin_amdgcn_sched_barrier(0);
          bf16x2 h2, l2;
          split2_product(g1[2 * k], d1[2 * k], g1[2 * k + 1], d1[2 * k + 1], h2, l2);
          colsum = __builtin_fmaf(g1[2 * k + 1], d1[2 * k + 1], __builtin_fmaf(g1[2 * k], d1[2 * k], colsum));
          const int j = (2 * k) % 8;
          g1h[k / 4][j] = h2[0]; g1h[k / 4][j + 1] = h2[1];
          g1l[k / 4][j] = l2[0]; g1l[k / 4][j + 1] = l2[1];
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int t = 0; t < 2; t++) {
          *piece_at(QD_P, 0, 2 * tb + t) = g1h[t];
          *piece_at(QD_P, 1, 2 * tb + t) = g1l[t];
        }
        if (gone != 0) return;
        if (tb == 0) s_cs[lane] = colsum;   // (block 1's tokens are added to it, behind B3)
      }
      __builtin_amdgcn_sched_barrier(0);
      TTT_STAGE(FQC_G1);
      __syncthreads();                                    // B3: the terms of G1
      TTT_STAGE(FQC_B3);
      __builtin_amdgcn_sched_barrier(0);
      {
        bf16x8 g1h[4], g1l[4];
#pragma unroll
        for (int s = 0; s < 4; s++) {
          g1l[s] = *piece_at(QD_P, 1, s);
          g1h[s] = *piece_at(QD_P, 0, s);
        }
        float cs0 = s_cs[lane_v];
#pragma unroll
        for (int k = 8; k < 12; k++) w2_product(k);
        load_xk(mb + 1);   // (put there before B2)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 4; s++) {   // W1[32 tb .., shard] += XK^T G1, the split of W2 between the products
          W1 = MFMA(xkt[s], g1l[s], W1);
          W1 = MFMA(xkt[s], g1h[s], W1);
          __builtin_amdgcn_sched_barrier(0);
          if (s == 1) give_w2(0);
          if (s == 2) give_w2(1);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (tb == 1) {
          QD_LANE;
#pragma unroll
          for (int k = 0; k < 8; k++) cs0 = __builtin_fmaf(g1[2 * k + 1], d1[2 * k + 1], __builtin_fmaf(g1[2 * k], d1[2 * k], cs0));
          const float b1n = b1L + half_sum_valu(cs0);
          if (h == 0) s_b1[FW_NS * sh + c] = b1n;
        }
        give_w1();
      }
      __builtin_amdgcn_sched_barrier(0);
      TTT_STAGE(FQC_STEP);
      __syncthreads();                                    // B4: the terms of the new state
      TTT_STAGE(FQC_B4);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (part < 2) TTT_STAGES_END(bh, STAGE_ROLE_HALF + part);
    take_w1();
    take_w2();
    __syncthreads();   // (the last state's terms have been read)
    output_partial();
    __syncthreads();
#undef QD_LANE
    return;
  }

  // ------------------------------------------------------------------ helper waves
  const int u = w - 4;                                // number among them
  const int q8 = lane >> 3, f0 = 8 * (lane & 7);
  const int t_in = 8 * u + q8;                        // the rows that this lane sums, sends and brings in: token t_in of both blocks
  // This CU's 16 tokens (half u & 1 of them, as rows of 8 lanes each): two waves, whose rows they are anyway, normalise their sums and
  // form G2; the other two finish Out of them.
  const bool owns = (u >> 1) == (part & 1);
  const int half = u & 1, own_blk = part >> 1, own_tok = 16 * part + 8 * half + q8;
  const gptr_t gXQ = gbuf(p.XQ + x_base), gXK = gbuf(p.XK + x_base), gXV = gbuf(p.XV + x_base), gOut = gbuf(p.Out + x_base);
  const gptr_t gEta = gbuf(p.last_eta + uni64((size_t)bh * p.NC * CS));
  const unsigned voff = (t_in * FD + f0) * 2, own_off = (own_tok * FD + f0) * 2;
  struct Tile2 {
    bf16x8 v[2];
  };
  auto load2 = [&](gptr_t g, int m) {
    Tile2 x;
#pragma unroll
    for (int k = 0; k < 2; k++) x.v[k] = g_ld8h(g, voff, m * TILE_BYTES + k * (TILE_BYTES / 2));
    return x;
  };
  auto put2 = [&](bf16* tile, const Tile2& x) {
#pragma unroll
    for (int k = 0; k < 2; k++) lds_put16(tile + xrow(32 * k + t_in) + f0, __builtin_bit_cast(u32x4, x.v[k]));
  };
  // Inputs: XK a mini-batch ahead, XQ of the one at hand (for the output branch behind it); XK, XV (`kv`) and eta of this lane's own
  // token in it, or - the waves that finish Out - XQ of its token two mini-batches ago.
  const int last = p.NC - 1;
  Tile2 xk_n = load2(gXK, 0), xq = load2(gXQ, 0);
  bf16x8 kv[2];
  bf16 eta;
  auto load_own = [&](int m) {
    if (owns) {
      kv[0] = g_ld8h(gXK, own_off, m * TILE_BYTES);
      kv[1] = g_ld8h(gXV, own_off, m * TILE_BYTES);
      eta = g_ldh(gEta, 2 * own_tok, m * (CS * 2));
    } else {
      kv[0] = g_ld8h(gXQ, own_off, max(m - 2, 0) * TILE_BYTES);
    }
  };
  kv[1] = g_ld8h(gXV, own_off, 0);
  eta = g_ldh(gEta, 2 * own_tok, 0);
  load_own(0);
  put2(reinterpret_cast<bf16*>(smem + QD_XK), xk_n);
  xk_n = load2(gXK, min(1, last));
  __syncthreads();   // the flag is clear
  bool alive = true;
  const bool near = on_one_xcd(words + QDW_XCD, QD_CUS, lane, w_status, p.wait_limit, alive);
  if (!alive && lane == 0) *s_flag = 1;
  __syncthreads();
  if (flag() != 0) {
    if (lane == 0) report_status(w_status);
    return;
  }
  const gptr_t xch = gbuf(p.xchg + (size_t)bh * FWD_QUAD_XCHG_WORDS);
  auto words_at = [&](unsigned first) {   // (a scalar base and the lane's offset, as in g_ld)
    gptr_t q = xch + static_cast<uint64_t>(uni(8 * first));
    unsigned o = 8 * lane;
    asm("" : "+s"(q), "+v"(o));
    return (gword64_t)(q + static_cast<uint64_t>(o));
  };
  auto p_slot = [&](int slot, int to, int from, int half) { return words_at(((slot * QD_CUS + to) * QD_CUS + from) * 512 + half * 256); };
  auto o_slot = [&](int slot, int to, int from, int half) { return words_at(QD_XOUT + ((slot * QD_CUS + to) * QD_CUS + from) * 512 + half * 256); };
  auto g_slot = [&](int slot, int cu, int half) { return words_at(QD_XG2 + ((slot * QD_CUS + cu) * 2 + half) * 256); };
  auto b_slot = [&](int slot, int cu, int half) { return words_at(QD_XB2 + ((slot * QD_CUS + cu) * 2 + half) * 64); };
  bool gave_up = false;
  alignas(16) float gam[8], bet[8];
  float b2v[8], b2L = s_b2[lane];                     // b2 of this lane's features, and (the wave that steps it) of feature `lane`
#pragma unroll
  for (int e = 0; e < 8; e++) { gam[e] = s_gam[f0 + e]; bet[e] = s_bet[f0 + e]; b2v[e] = 0.f; }
  auto load_b2 = [&]() {
#pragma unroll
    for (int e = 0; e < 8; e++) b2v[e] = s_b2[f0 + e];
  };
  // Sum over this CU's hidden columns for token row `t` of block blk.
  auto gather = [&](int base, int blk, int t, float (&m)[8]) {
    const float* const row = reinterpret_cast<const float*>(smem + base + 2 * blk * QD_PTILE) + t * LDP + f0;
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const f32x4 s = *reinterpret_cast<const f32x4*>(row + 4 * q) + *reinterpret_cast<const f32x4*>(row + QD_PTILE / 4 + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; e++) m[4 * q + e] = s[e];
    }
  };
  auto put4 = [&](gword64_t dst, const uint64_t (&x)[4]) {   // (one branch for the four)
    if (near) {
#pragma unroll
      for (int k = 0; k < 4; k++) wd_put(dst + 64 * k, x[k], true);
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++) wd_put(dst + 64 * k, x[k], false);
    }
  };
  auto send = [&](gword64_t dst, const float (&m)[8]) {
    const uint64_t x[4] = {wd_pack(m[0], m[1]), wd_pack(m[2], m[3]), wd_pack(m[4], m[5]), wd_pack(m[6], m[7])};
    put4(dst, x);
  };
  auto mark = [&](gword64_t dst) {
    const uint64_t x[4] = {~0ull, ~0ull, ~0ull, ~0ull};
    put4(dst, x);
  };
  auto other = [&](int o) { return o + (o >= part ? 1 : 0); };   // the CUs but this one
  // z += the four CUs' shares in their order, this CU's own and what came from the others
  auto add_shares = [&](float (&z)[8], const float (&own)[8], const uint64_t (&x)[QD_CUS - 1][4]) {
    auto add_own = [&]() {
#pragma unroll
      for (int e = 0; e < 8; e++) z[e] += own[e];
    };
#pragma unroll
    for (int o = 0; o < QD_CUS - 1; o++) {
      if (part == o) add_own();
#pragma unroll
      for (int k = 0; k < 4; k++) { z[2 * k] += wd_lo(x[o][k]); z[2 * k + 1] += wd_hi(x[o][k]); }
    }
    if (part == QD_CUS - 1) add_own();
  };
  // Waits for N messages of W words per lane, number i at at(i); `meanwhile` once, between the first request and its answer.
  auto take = [&](auto at, auto& x, auto meanwhile) __attribute__((always_inline)) {
    constexpr int N = sizeof(x) / sizeof(x[0]), W = sizeof(x[0]) / sizeof(uint64_t);
    uint64_t t0 = 0;
    for (unsigned n = 0;; n++) {
#pragma unroll
      for (int i = 0; i < N; i++) {
        const gword64_t src = at(i);
#pragma unroll
        for (int k = 0; k < W; k++) x[i][k] = __hip_atomic_load(src + 64 * k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      if (n == 0) meanwhile();
      uint32_t most = 0;   // (the mark is the largest of all words)
#pragma unroll
      for (int i = 0; i < N; i++)
#pragma unroll
        for (int k = 0; k < W; k++) most = max(most, max(static_cast<uint32_t>(x[i][k]), static_cast<uint32_t>(x[i][k] >> 32)));
      if (__all(most != WD_EMPTY)) return;
      if (n == 1 || (n & 7) == 0) {   // (the clock is not asked every time: its answer takes as long as the words')
        const uint64_t now = wall_clock64();
        if (n == 0) t0 = now;
        else if (now - t0 > p.wait_limit || ((n & 63) == 0 && __hip_atomic_load(w_status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
          raise_status(w_status);
          gave_up = true;
          return;
        }
      }
    }
  };
  auto nothing = []() {};
  // Out's sums of the mini-batch at hand, gathered between B2 and B3 and sent behind it: of the rows of the other CUs' tokens; of this CU's
  // own tokens the waves that finish Out keep them (mo).
  float so[2][8], mo[8];
#pragma unroll
  for (int e = 0; e < 8; e++) mo[e] = 0.f;
  auto gather_output = [&]() {
    gather(QD_OUT, 0, t_in, so[0]);
    gather(QD_OUT, 1, t_in, so[1]);
    if (!owns) gather(QD_OUT, own_blk, own_tok & 31, mo);
  };
  auto give_output = [&](int slot) {
#pragma unroll
    for (int blk = 0; blk < 2; blk++) {
      const int to = 2 * blk + (u >> 1);
      if (to != part) send(o_slot(slot, to, part, half), so[blk]);
    }
  };
  // (b2v: b2 after mini-batch m; kv[0]: its XQ)
  auto finish_output = [&](int m, int slot, const float (&own)[8]) {
    uint64_t x[QD_CUS - 1][4];
    auto from = [&](int o) { return o_slot(slot, part, other(o), half); };
    take(from, x, nothing);
#pragma unroll
    for (int o = 0; o < QD_CUS - 1; o++) mark(from(o));
    float z[8];
#pragma unroll
    for (int e = 0; e < 8; e++) z[e] = b2v[e];
    add_shares(z, own, x);
    g_st8h(gOut, own_off, m * TILE_BYTES, output_layernorm_row(z, gam, bet, kv[0]));
  };
  TTT_STAGES_BEGIN();

  int slot = 0;   // mb % 3
  for (int mb = 0; mb < p.NC; mb++, slot = slot == 2 ? 0 : slot + 1) {
    const int before = slot == 0 ? 2 : slot - 1;      // the slot of mini-batch mb - 1
    if (owns) load_b2();
    if (u == 0 && part == 0 && mb % p.cgs == 0) p.b2_ck[((size_t)bh * p.K + mb / p.cgs) * FD + lane] = s_b2[lane];
    float target[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      target[e] = bf2f(kv[1][e]) - bf2f(kv[0][e]);
      asm volatile("" : "+v"(target[e]));   // formed here, before anything waits for these waves
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the marks put back so far are in place
    TTT_STAGE(FQH_TOP);
    __builtin_amdgcn_s_setprio(2);   // from here to B2 these waves' instructions are what the other four wait for
    __syncthreads();   // B1
    TTT_STAGE(FQH_B1);
    float m[2][8];
    gather(QD_P, 0, t_in, m[0]);
    gather(QD_P, 1, t_in, m[1]);
#pragma unroll
    for (int blk = 0; blk < 2; blk++) {
      const int to = 2 * blk + (u >> 1);
      if (to != part) send(p_slot(mb & 1, to, part, half), m[blk]);
    }
    TTT_STAGE(FQH_SEND);
    auto put_g2 = [&](int tok, u32x4 hi, u32x4 lo) {
      lds_put16(s_g2 + tok * FLD + f0, hi);
      lds_put16(s_g2l + tok * FLD + f0, lo);
    };
    // Message i of the six that carry the other CUs' G2: two for a wave that finishes Out, one for a wave that has its own to form.
    auto take_g2 = [&](auto& x, int first, auto meanwhile) {
      constexpr int N = sizeof(x) / sizeof(x[0]);
      take([&](int i) { return g_slot(slot, other((first + i) >> 1), (first + i) & 1); }, x, meanwhile);
#pragma unroll
      for (int i = 0; i < N; i++) {
        u32x4 v[2];
#pragma unroll
        for (int k = 0; k < 4; k++) {
          v[k >> 1][2 * (k & 1)] = static_cast<uint32_t>(x[i][k]);
          v[k >> 1][2 * (k & 1) + 1] = static_cast<uint32_t>(x[i][k] >> 32);
        }
        put_g2(16 * other((first + i) >> 1) + 8 * ((first + i) & 1) + q8, v[0], v[1]);
      }
    };
    bf16* const xk_next = reinterpret_cast<bf16*>(smem + QD_XK + ((mb + 1) & 1) * SM_TILE);   // (last read a mini-batch ago)
    if (owns) {
      uint64_t x[QD_CUS - 1][4];
      auto from = [&](int o) { return p_slot(mb & 1, part, other(o), half); };
      take(from, x, [&]() { put2(xk_next, xk_n); });
      TTT_STAGE(FQH_TAKE);
      float z[8], gx[8], own[8];
#pragma unroll
      for (int e = 0; e < 8; e++) { z[e] = b2v[e]; own[e] = own_blk == 0 ? m[0][e] : m[1][e]; }
      add_shares(z, own, x);
      const float scale = ln_loss_gradient(z, target, bf2f(eta), gam, bet, gx);
      f32x16 g2;
#pragma unroll
      for (int e = 0; e < 8; e++) { g2[e] = gx[e] * scale; g2[8 + e] = 0.f; }
      bf16x8 o, ol;
      split8_plain(g2, 0, o, ol);
      u32x4 hi = __builtin_bit_cast(u32x4, o), lo = __builtin_bit_cast(u32x4, ol);
#pragma unroll
      for (int k = 0; k < 4; k++) { hi[k] = min(hi[k], WD_EMPTY - 1); lo[k] = min(lo[k], WD_EMPTY - 1); }   // (a NaN stays one)
      const uint64_t y[4] = {hi[0] | (uint64_t)hi[1] << 32, hi[2] | (uint64_t)hi[3] << 32, lo[0] | (uint64_t)lo[1] << 32, lo[2] | (uint64_t)lo[3] << 32};
      put4(g_slot(slot, part, half), y);
      put_g2(own_tok, hi, lo);
      TTT_STAGE(FQH_LN);
      uint64_t y1[1][4];
      take_g2(y1, 4 + half, [&]() {
        // this wave's share of the step of b2
        float* const share = s_b2p + (2 * part + half) * FD;
        ln_token_sum_store_product(share, gx, scale, lane, f0);
        TTT_WAVE_SYNC();
        wd_put(b_slot(slot, part, half), min(__builtin_bit_cast(uint32_t, share[lane]), WD_EMPTY - 1), near);
      });
      // the marks: what was received; what was sent for mini-batch mb - 1, which everyone has read now that their next sums are here
#pragma unroll
      for (int o = 0; o < QD_CUS - 1; o++) mark(from(o));
      mark(g_slot(before, part, half));
      wd_put(b_slot(before, part, half), ~0ull, near);
    } else {
      put2(xk_next, xk_n);
      if (mb > 1) finish_output(mb - 2, slot == 2 ? 0 : slot + 1, mo);
      load_b2();
      TTT_STAGE(FQH_OUTPUT);
      uint64_t y[2][4];
      take_g2(y, 2 * half, nothing);
    }
    if (gave_up && lane == 0) *s_flag = 1;
    TTT_STAGE(FQH_TAKE2);
    __syncthreads();   // B2
    TTT_STAGE(FQH_B2);
    __builtin_amdgcn_s_setprio(0);
    if (flag() != 0) {
      if (lane == 0) report_status(w_status);
      return;
    }
    // (gathered: Out's sums of mini-batch mb - 1; nothing there yet in the first one, and not sent)
    if (owns || half == 1) gather_output();
    else {   // b2 after this mini-batch: + the sum over the tokens of G2, eight shares in a fixed order
      uint64_t x[6][1];
      take([&](int i) { return b_slot(slot, other(i >> 1), i & 1); }, x, gather_output);
      float mine[2] = {s_b2p[2 * part * FD + lane], s_b2p[(2 * part + 1) * FD + lane]};
#pragma unroll
      for (int o = 0; o < QD_CUS; o++) {
        if (o == part) { b2L += mine[0]; b2L += mine[1]; }
        if (o < QD_CUS - 1) { b2L += wd_lo(x[2 * o][0]); b2L += wd_lo(x[2 * o + 1][0]); }
      }
      s_b2[lane] = b2L;
    }
    TTT_STAGE(FQH_GIVE);
    __syncthreads();   // B3
    TTT_STAGE(FQH_B3);
    if (mb > 0) give_output(before);
    put2(s_xq, xq);
    // the next mini-batch's inputs, under way until its sums are here
    const int next = min(mb + 1, last);
    xk_n = load2(gXK, min(mb + 2, last));
    xq = load2(gXQ, next);
    load_own(next);
    TTT_STAGE(FQH_NEXT);
    __syncthreads();   // B4
    TTT_STAGE(FQH_B4);
  }
  if (part < 2) TTT_STAGES_END(bh, STAGE_ROLE_HALF + part);
  // Out of the last two mini-batches
  const int slot1 = slot == 0 ? 2 : slot - 1, slot2 = slot1 == 0 ? 2 : slot1 - 1;
  if (!owns) {
    if (p.NC > 1) {
      kv[0] = g_ld8h(gXQ, own_off, (p.NC - 2) * TILE_BYTES);
      finish_output(p.NC - 2, slot2, mo);
    }
    kv[0] = g_ld8h(gXQ, own_off, last * TILE_BYTES);
    load_b2();
  }
  __syncthreads();
  __syncthreads();
  gather_output();
  give_output(slot1);
  if (!owns) finish_output(last, slot1, mo);
  if (gave_up && lane == 0) report_status(w_status);
}

}  // namespace ttt
