// Forward scan with the recurrence of one (batch, head) spread over two CUs, where four each (ttt_mlp_fwd_quad.hpp) do not fit:
// 65 to 80 pairs on 256 CUs.
//
// The recurrence of a pair is sequential and one CU spends 19.4 k clocks on a mini-batch of it, close to the sum of
// what the two waves of each SIMD issue.  Here two workgroups of the same XCD hold 128 hidden columns each, and inside a
// workgroup the eight waves are of two kinds:
//   waves 0-3 (one per SIMD)  32 hidden columns each: every matrix product and the state, as in ttt_mlp_fwd.hip
//   waves 4-7                 the sums over the hidden dimension, their exchange with the other CU and the LayerNorm lanes
// A mini-batch is taken in two blocks of 32 tokens, so that block 0's sums travel to the other CU and through the
// LayerNorm while the compute waves form block 1, and block 1's while they apply block 0's share of the weight step.
// What crosses the CUs is one or two fp32 tiles per mini-batch and direction (16 / 32 KiB; both CUs form the LayerNorm of
// all tokens, from the same sums in the same order).  No flags: a word is sent as it is and its slot holds an impossible
// value (a NaN that is never sent) before and after; the receiver polls the data itself and puts the mark back.
// One more workgroup per pair computes Out from the states left in a ring, as in the two-workgroup launch.
// Every sum has the order of the one-workgroup kernel: results are the same to the bit.
//
// What bounds it: the chain, 14.2 k clocks per mini-batch (with a second workgroup for Out beside it): block 0's Z1, GELU and partial sums
// 2.7 k; block 1's 3.5 k while block 0's sums cross (gather and send 1.3 k, 1.0 k under way, LayerNorm 1.7 k) and 0.7 k of waiting for them;
// block 0's weight step 1.9 k while block 1's sums cross and 2.5 k of waiting for those; block 1's weight step and the
// split of the new state 2.65 k.  80 pairs x 512 mini-batches 3.72 ms; the recurrence on one CU 4.4.
#include "ttt_mlp_exchange.hpp"
#include "ttt_mlp_fwd_common.hpp"
#include "ttt_mlp_fwd_quad.hpp"

namespace ttt {

constexpr int WD_NCOMP = 4;                              // compute waves per workgroup
// LDS carve-up of a recurrence workgroup (bytes)
constexpr int WD_XK = 0;                                 // two buffers, alternating per mini-batch
constexpr int WD_G2 = WD_XK + 2 * SM_TILE;
constexpr int WD_G2L = WD_G2 + SM_TILE;
constexpr int WD_P0 = WD_G2L + SM_TILE;                  // per compute wave: its partial sum of token block 0, [32 tok][F] fp32
constexpr int WD_PTILE = 32 * LDP * 4;
constexpr int WD_P1 = WD_P0 + WD_NCOMP * WD_PTILE;       // the same for block 1; before that sum is formed, the two terms of
constexpr int WD_LDT = 36;                               // W2[shard, :] as [F][hid] (row stride in elements)
constexpr int WD_WTILE = FD * WD_LDT * 2;
constexpr int WD_P1TILE = 2 * WD_WTILE;
static_assert(WD_PTILE <= WD_P1TILE, "block 1's sums take the place of the W2 tiles");
constexpr int WD_X2T = WD_P1 + WD_NCOMP * WD_P1TILE;     // per compute wave: X2 shard, [hid][tok]
constexpr int WD_B2 = WD_X2T + WD_NCOMP * SM_X2T_TILE;
constexpr int WD_GAM = WD_B2 + FD * 4;
constexpr int WD_BET = WD_GAM + FD * 4;
constexpr int WD_B2P = WD_BET + FD * 4;                  // [8 groups of 8 tokens][F]: shares of the step of b2
constexpr int WD_FLAG = WD_B2P + 8 * FD * 4;             // [0] non-zero: a wait gave up; [1] helper waves that have left their shares of b2
constexpr int WD_BYTES = WD_FLAG + 16;
static_assert(WD_BYTES <= SM_FWD_BYTES, "the launch asks for SM_FWD_BYTES (the output branch's carve-up)");

// Synchronisation words of a pair: 0 / 8 mini-batches handed over by the two halves, 16 mini-batches finished by the
// output workgroup, 24 .. the XCD each workgroup of the pair runs on (+ 1).
constexpr int WDW_GIVEN = 0, WDW_TAKEN = 16, WDW_XCD = 24;

TTT_DEV void fwd_wide_recurrence(const FwdParams& p, unsigned char* smem, const int bh, const int half) {
  bf16* const s_g2 = reinterpret_cast<bf16*>(smem + WD_G2);
  bf16* const s_g2l = reinterpret_cast<bf16*>(smem + WD_G2L);
  float* const s_b2 = reinterpret_cast<float*>(smem + WD_B2);
  float* const s_gam = reinterpret_cast<float*>(smem + WD_GAM);
  float* const s_bet = reinterpret_cast<float*>(smem + WD_BET);
  float* const s_b2p = reinterpret_cast<float*>(smem + WD_B2P);
  typedef __attribute__((address_space(3))) int* lint_t;
  const lint_t s_flag = (lint_t)reinterpret_cast<int*>(smem + WD_FLAG);
  auto flag = [&]() { return __hip_atomic_load(s_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, c = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave of the workgroup
  const bool compute = w < WD_NCOMP;
  const int u = w & 3;                                      // number among its kind
  // hidden block of compute wave u: the halves hold whole wave pairs (v, v + 4) of the one-workgroup kernel
  const int v = 2 * half + (u & 1) + 4 * (u >> 1);
  const int head = bh % p.NH;
  const int hid0 = FW_NS * v;

  int* const words = p.sync + (size_t)bh * BWD_SYNC_STRIDE;
  int* const w_status = p.status;
  if (tid == 0) say_xcd(words + WDW_XCD + half);
  if (tid < FD) {
    s_b2[tid] = p.b2[(size_t)bh * FD + tid];
    s_gam[tid] = p.ttt_norm_weight[head * FD + tid];
    s_bet[tid] = p.ttt_norm_bias[head * FD + tid];
  }
  if (tid < 2) s_flag[tid] = 0;
  const size_t x_base = uni64((size_t)bh * p.NC * (CS * FD));

  if (compute) {
    const gptr_t gW1ck = gbuf(p.W1_ck + uni64((size_t)bh * p.K * FD * HID)), gW2ck = gbuf(p.W2_ck + uni64((size_t)bh * p.K * HID * FD));
    AccT<2, 1> W1s;
    AccT<1, 2> W2s;
    {
      const gptr_t W1 = gbuf(p.W1 + (size_t)bh * FD * HID), W2 = gbuf(p.W2 + (size_t)bh * HID * FD);
#pragma unroll
      for (int b = 0; b < 2; b++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int row = 8 * (i >> 2) + (i & 3);   // + 4h in the lane offset
          W1s.b[b][0][i] = g_ldf(W1, (4 * h * HID + c) * 4, ((32 * b + row) * HID + hid0) * 4);
          W2s.b[0][b][i] = g_ldf(W2, (4 * h * FD + c) * 4, ((hid0 + row) * FD + 32 * b) * 4);
        }
    }
    float b1L = p.b1[(size_t)bh * HID + hid0 + c];
    float* const s_P0 = reinterpret_cast<float*>(smem + WD_P0 + u * WD_PTILE);
    float* const s_P1 = reinterpret_cast<float*>(smem + WD_P1 + u * WD_P1TILE);
    bf16* const s_x2t = reinterpret_cast<bf16*>(smem + WD_X2T + u * SM_X2T_TILE);
    bf16* const t_hi = reinterpret_cast<bf16*>(s_P1);
    bf16* const t_lo = t_hi + WD_WTILE / 2;
    // the two bf16 terms of the state, formed once per mini-batch: operands of Z1 and Z2, the transposition, and (the
    // high-order ones) what the output branch is given
    OpdT<1, 4> w1h, w1l;
    OpdT<2, 2> w2h, w2l;
    cvt_chain_split(W1s, w1h, w1l);
    cvt_chain_split(W2s, w2h, w2l);
    __syncthreads();   // the flag is clear
    __syncthreads();   // XK of mini-batch 0, b2, norm parameters; the helpers know where the other workgroups are
    if (flag() != 0) return;

    int lane_v = lane;
#define WD_LANE                                             \
  asm volatile("" : "+v"(lane_v));                          \
  const int lane = lane_v, h = lane >> 5, c = lane & 31;    \
  (void)h; (void)c
    // Chunk k of the state after mini-batch m for the output branch (W1: k < 4, W2; the biases with the first).  Eight stores of
    // 1 KiB in a row from every wave stall it for 1.5 k clocks, so they are spread over the next mini-batch's block 1, which
    // has time: its sums wait for the other CU.
    auto store_image = [&](int m, int k) {
      WD_LANE;
      // (m = -1: the initial state, to a slot that is not in use yet)
      const size_t slot = (size_t)bh * FWD_WIDE_RING + (m + FWD_WIDE_RING) % FWD_WIDE_RING;
      const gptr_t gImg = gbuf(p.state_img + slot * (FWD_IMG_BYTES / 2));
      g_st_stream<bf16x8>(gImg, 16 * ((v << 6) | lane), k * 8192, k < 4 ? w1h.v[0][k] : w2h.v[(k - 4) >> 1][k & 1]);
      if (k == 0) p.bias_img[slot * FWD_BIAS_FLOATS + hid0 + c] = b1L;   // both halves of the wave hold it
    };
    bf16x8 xk[4];
#pragma unroll
    for (int s = 0; s < 4; s++) xk[s] = xpiece_rows(reinterpret_cast<const bf16*>(smem + WD_XK), 0, s, c, h);
    TTT_STAGES_BEGIN();
    for (int mb = 0; mb < p.NC; mb++) {
      const bf16* const s_xk = reinterpret_cast<const bf16*>(smem + WD_XK + (mb & 1) * SM_TILE);
      if (mb % p.cgs == 0) {   // checkpoint: the state before this mini-batch
        WD_LANE;
        const int ck_slot = mb / p.cgs;
        const unsigned ck = static_cast<unsigned>(ck_slot) * (FD * HID * 4u);
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
          for (int i = 0; i < 16; i++) {
            const int row = 8 * (i >> 2) + (i & 3);
            g_stf(gW1ck, (4 * h * HID + c) * 4, ck + ((32 * b + row) * HID + hid0) * 4, W1s.b[b][0][i]);
            g_stf(gW2ck, (4 * h * FD + c) * 4, ck + ((hid0 + row) * FD + 32 * b) * 4, W2s.b[0][b][i]);
          }
        if (h == 0) p.b1_ck[((size_t)bh * p.K + ck_slot) * HID + hid0 + c] = b1L;
      }
      f32x16 d1[2];
      OpdT<1, 4> x2lo;
      // XK of token block rb of mini-batch m (lane = tok): read a stage ahead of its products
      auto load_xk = [&](int m, int rb) {
        WD_LANE;
        const bf16* const x = reinterpret_cast<const bf16*>(smem + WD_XK + (m & 1) * SM_TILE);
#pragma unroll
        for (int s = 0; s < 4; s++) xk[s] = xpiece_rows(x, rb, s, c, h);
      };
      // X2 = gelu(Z1), gelu'(Z1) of token block rb; X2's high-order term to LDS
      auto z1_block = [&](int rb, bool images) {
        WD_LANE;
        f32x16 x2;   // Z1 = XK W1 + b1
#pragma unroll
        for (int i = 0; i < 16; i++) x2[i] = b1L;
#pragma unroll
        for (int s = 0; s < 4; s++) x2 = MFMA(xk[s], w1l.v[0][s], x2);
#pragma unroll
        for (int s = 0; s < 4; s++) x2 = MFMA(xk[s], w1h.v[0][s], x2);
#pragma unroll
        for (int q = 0; q < 4; q++) {
          if (images) {
            __builtin_amdgcn_sched_barrier(0);
            store_image(mb - 1, q);
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int i = 4 * q; i < 4 * q + 4; i++) {
            float g, d;
            gelu_fd(x2[i], g, d);
            x2[i] = g;
            d1[rb][i] = d;
          }
        }
#pragma unroll
        for (int t = 0; t < 2; t++) {
          bf16x8 xh;
          split8_plain(x2, t, xh, x2lo.v[0][2 * rb + t]);
          store_piece_rows<FLD>(s_x2t, 0, 2 * rb + t, c, h, xh);
        }
        TTT_WAVE_SYNC();
      };
      // Z2^T partial of token block rb (rows F, lane = tok), left in this wave's tile as [tok][F]
      auto z2_block = [&](int rb, float* s_Pw) {
        WD_LANE;
        bf16x8 xb[2];
#pragma unroll
        for (int s = 0; s < 2; s++) xb[s] = piece_tr<FLD>(s_x2t, rb, s, lane);
#pragma unroll
        for (int fb = 0; fb < 2; fb++) {
          f32x16 z;
#pragma unroll
          for (int i = 0; i < 16; i++) z[i] = 0.f;
#pragma unroll
          for (int s = 0; s < 2; s++) {
            z = MFMA(w2l.v[fb][s], xb[s], z);
            z = MFMA(w2h.v[fb][s], xb[s], z);
          }
#pragma unroll
          for (int g = 0; g < 4; g++) {
            f32x4 q = {z[4 * g], z[4 * g + 1], z[4 * g + 2], z[4 * g + 3]};
            *reinterpret_cast<f32x4*>(s_Pw + c * LDP + 32 * fb + 8 * g + 4 * h) = q;
          }
        }
      };
      z1_block(0, false);
      load_xk(mb, 1);
      z2_block(0, s_P0);
      __builtin_amdgcn_sched_barrier(0);
      TTT_STAGE(FWC_BLOCK0);
      __syncthreads();                                    // B1: block 0's partial sums
      TTT_STAGE(FWC_B1);
      __builtin_amdgcn_sched_barrier(0);
      z1_block(1, true);
      bf16x8 wh[4], wl[4];   // W2[shard, :] with F contracted: its terms as rows [F][hid], read back transposed
      {
        WD_LANE;
#pragma unroll
        for (int fb = 0; fb < 2; fb++)
#pragma unroll
          for (int s = 0; s < 2; s++) {
            store_piece_rows<WD_LDT>(t_hi, fb, s, c, h, w2h.v[fb][s]);
            store_piece_rows<WD_LDT>(t_lo, fb, s, c, h, w2l.v[fb][s]);
            __builtin_amdgcn_sched_barrier(0);
            store_image(mb - 1, 4 + 2 * fb + s);
            __builtin_amdgcn_sched_barrier(0);
          }
        TTT_WAVE_SYNC();
#pragma unroll
        for (int s = 0; s < 4; s++) {
          wh[s] = piece_tr<WD_LDT>(t_hi, 0, s, lane);
          wl[s] = piece_tr<WD_LDT>(t_lo, 0, s, lane);
        }
        TTT_WAVE_SYNC();
      }
      z2_block(1, s_P1);
      // the operands of the weight step that do not wait for G2
      bf16x8 xkt[2][2], xh[2];
      auto step_operands = [&](int rb) {
        WD_LANE;
#pragma unroll
        for (int t = 0; t < 2; t++) {
#pragma unroll
          for (int fb = 0; fb < 2; fb++) xkt[t][fb] = xpiece_tr(s_xk, fb, 2 * rb + t, lane);
          xh[t] = piece_rows<FLD>(s_x2t, 0, 2 * rb + t, c, h);
        }
      };
      step_operands(0);
      float colsum = 0.f;
      // G1 = (G2 W2^T) * gelu'(Z1) of token block rb and its share of the weight step.  One wave per SIMD: what hides the LDS
      // latency and the vector instructions is their order - operands are asked for a product ahead, and W2's step, which
      // does not need G1, keeps the matrix pipe busy while G1 is finished and split.
      auto update_block = [&](int rb) {
        WD_LANE;
        f32x16 g1;
#pragma unroll
        for (int i = 0; i < 16; i++) g1[i] = 0.f;
        bf16x8 ah[2], al[2], gh[2][2], gl[2][2];
        auto step_g2 = [&](int t) {   // G2 with tokens contracted (lane = F), for W2's step
#pragma unroll
          for (int fb = 0; fb < 2; fb++) {
            gh[t][fb] = piece_tr<FLD>(s_g2, fb, 2 * rb + t, lane);
            gl[t][fb] = piece_tr<FLD>(s_g2l, fb, 2 * rb + t, lane);
          }
        };
        ah[0] = piece_rows<FLD>(s_g2, rb, 0, c, h);
        al[0] = piece_rows<FLD>(s_g2l, rb, 0, c, h);
#pragma unroll
        for (int s = 0; s < 4; s++) {
          if (s < 3) {
            ah[(s + 1) & 1] = piece_rows<FLD>(s_g2, rb, s + 1, c, h);
            al[(s + 1) & 1] = piece_rows<FLD>(s_g2l, rb, s + 1, c, h);
          }
          if (s == 3) step_g2(0);
          __builtin_amdgcn_sched_barrier(0);
          g1 = MFMA(al[s & 1], wh[s], g1);
          g1 = MFMA(ah[s & 1], wl[s], g1);
          g1 = MFMA(ah[s & 1], wh[s], g1);
          __builtin_amdgcn_sched_barrier(0);
        }
        step_g2(1);
        bf16x8 g1h[2], g1l[2];
#pragma unroll
        for (int k = 0; k < 12; k++) {   // W2[shard, :] += X2^T G2; with each of the first eight products two values of G1
          const int t = k / 6, fb = (k / 3) % 2, o = k % 3;
          W2s.b[0][fb] = MFMA(o == 0 ? x2lo.v[0][2 * rb + t] : xh[t], o == 1 ? gl[t][fb] : gh[t][fb], W2s.b[0][fb]);
          __builtin_amdgcn_sched_barrier(0);
          if (k < 8) {
            bf16x2 h2, l2;
            split2_product(g1[2 * k], d1[rb][2 * k], g1[2 * k + 1], d1[rb][2 * k + 1], h2, l2);
            colsum = __builtin_fmaf(g1[2 * k + 1], d1[rb][2 * k + 1], __builtin_fmaf(g1[2 * k], d1[rb][2 * k], colsum));
            const int j = (2 * k) % 8;
            g1h[k / 4][j] = h2[0]; g1h[k / 4][j + 1] = h2[1];
            g1l[k / 4][j] = l2[0]; g1l[k / 4][j + 1] = l2[1];
            __builtin_amdgcn_sched_barrier(0);
          }
        }
#pragma unroll
        for (int t = 0; t < 2; t++)     // W1[:, shard] += XK^T G1
#pragma unroll
          for (int fb = 0; fb < 2; fb++) {
            W1s.b[fb][0] = MFMA(xkt[t][fb], g1l[t], W1s.b[fb][0]);
            W1s.b[fb][0] = MFMA(xkt[t][fb], g1h[t], W1s.b[fb][0]);
          }
      };
      __builtin_amdgcn_sched_barrier(0);
      TTT_STAGE(FWC_BLOCK1);
      __syncthreads();                                    // B2: block 1's partial sums; G2 of block 0
      TTT_STAGE(FWC_B2);
      __builtin_amdgcn_sched_barrier(0);
      update_block(0);
      step_operands(1);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the last mini-batch's images, issued a block ago, are out
      __builtin_amdgcn_sched_barrier(0);
      TTT_STAGE(FWC_STEP0);
      __syncthreads();                                    // B3: G2 of block 1
      TTT_STAGE(FWC_B3);
      __builtin_amdgcn_sched_barrier(0);
      const int gave_up = flag();
      update_block(1);
      b1L += half_sum_valu(colsum);
      load_xk(mb + 1, 0);   // (put there before B2)
      cvt_chain_split(W2s, w2h, w2l);
      cvt_chain_split(W1s, w1h, w1l);
      TTT_STAGE(FWC_STEP1);
      if (gave_up != 0) return;
    }
    TTT_STAGES_END(bh, STAGE_ROLE_HALF + half);
#pragma unroll
    for (int k = 0; k < 8; k++) store_image(p.NC - 1, k);
#undef WD_LANE
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();   // the last mini-batch's state is out
    return;
  }

  // ------------------------------------------------------------------ helper waves
  const int q8 = lane >> 3, f0 = 8 * (lane & 7);
  const int t_in = 8 * u + q8;                        // this lane's token inside a block
  const gptr_t gXK = gbuf(p.XK + x_base), gXV = gbuf(p.XV + x_base);
  const gptr_t gEta = gbuf(p.last_eta + uni64((size_t)bh * p.NC * CS));
  const unsigned voff = (t_in * FD + f0) * 2;         // its 8 features of token t_in in an input tile
  // XK of mini-batch m reaches LDS through these lanes, which need their part of it for the LayerNorm as well
  bf16x8 xk_n[2];
  auto load_xk = [&](int m) {
#pragma unroll
    for (int k = 0; k < 2; k++) xk_n[k] = g_ld8h(gXK, voff, m * TILE_BYTES + k * (TILE_BYTES / 2));
  };
  auto put_xk = [&](int m) {
    bf16* const d = reinterpret_cast<bf16*>(smem + WD_XK + (m & 1) * SM_TILE);
#pragma unroll
    for (int k = 0; k < 2; k++) lds_put16(d + xrow(32 * k + t_in) + f0, __builtin_bit_cast(u32x4, xk_n[k]));
  };
  load_xk(0);
  put_xk(0);
  __syncthreads();   // the flag is clear
  bool alive = true;
  const bool near = on_one_xcd(words + WDW_XCD, 3, lane, w_status, p.wait_limit, alive);
  if (!alive && lane == 0) *s_flag = 1;
  __syncthreads();
  if (flag() != 0) {
    if (lane == 0) report_status(w_status);
    return;
  }
  const gword64_t xch = (gword64_t)(p.xchg + (size_t)bh * FWD_XCHG_WORDS);
  const float* const s_row0 = reinterpret_cast<const float*>(smem + WD_P0) + t_in * LDP + f0;
  const float* const s_row1 = reinterpret_cast<const float*>(smem + WD_P1) + t_in * LDP + f0;
  float b2v[8], b2L = s_b2[lane];                     // b2 of this lane's features, and of feature `lane` (wave 4 stores that one)
#pragma unroll
  for (int e = 0; e < 8; e++) b2v[e] = s_b2[f0 + e];
  float gx[2][8], scale[2] = {0.f, 0.f};               // G2 of the two blocks (gx * scale), whose token sums wait until the compute waves have what they wait for
  __builtin_amdgcn_s_setprio(2);                      // these waves' few instructions are what the other four wait for
  int seen = 0;                                       // mini-batches the output workgroup is known to have finished
  bool gave_up = false;
  TTT_STAGES_BEGIN();

  // The sum has the order of the one-workgroup kernel, (((b2 + P0) + P1) + P2) + P3 over the wave pairs: half 0 holds P0 and P1 and
  // sends b2 + P0 + P1, half 1 sends P2 and P3.
  float m0[8], m1[8];
  auto gather_send = [&](int mb, int blk) {
#pragma unroll
    for (int q = 0; q < 2; q++) {
      f32x4 a[4];
#pragma unroll
      for (int k = 0; k < 4; k++)
        a[k] = *reinterpret_cast<const f32x4*>((blk == 0 ? s_row0 + k * (WD_PTILE / 4) : s_row1 + k * (WD_P1TILE / 4)) + 4 * q);
      const f32x4 pa = a[0] + a[2], pb = a[1] + a[3];
#pragma unroll
      for (int e = 0; e < 4; e++) { m0[4 * q + e] = pa[e]; m1[4 * q + e] = pb[e]; }
    }
    const gword64_t dst = xch + ((((mb & 1) * 2 + half) * 2 + blk) * 4 + u) * 512 + lane;
    if (half == 0) {
#pragma unroll
      for (int e = 0; e < 8; e++) m0[e] = (b2v[e] + m0[e]) + m1[e];
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++) wd_put(dst + 256 + 64 * k, wd_pack(m1[2 * k], m1[2 * k + 1]), near);
    }
#pragma unroll
    for (int k = 0; k < 4; k++) wd_put(dst + 64 * k, wd_pack(m0[2 * k], m0[2 * k + 1]), near);
  };
  auto finish_block = [&](int mb, int blk, bf16x8 xk, bf16x8 xv, bf16 eta) {
    const int tok = 32 * blk + t_in;
    const gword64_t src = xch + ((((mb & 1) * 2 + 1 - half) * 2 + blk) * 4 + u) * 512 + lane;
    float z[8];
    if (half == 0) {
      uint64_t wv[8];
      if (!wd_take(src, wv, w_status, p.wait_limit)) gave_up = true;
      TTT_STAGE(blk == 0 ? FWH_TAKE0 : FWH_TAKE1);
#pragma unroll
      for (int k = 0; k < 8; k++) wd_put(src + 64 * k, ~0ull, near);
#pragma unroll
      for (int k = 0; k < 4; k++) {
        z[2 * k] = (m0[2 * k] + wd_lo(wv[k])) + wd_lo(wv[4 + k]);
        z[2 * k + 1] = (m0[2 * k + 1] + wd_hi(wv[k])) + wd_hi(wv[4 + k]);
      }
    } else {
      uint64_t wv[4];
      if (!wd_take(src, wv, w_status, p.wait_limit)) gave_up = true;
      TTT_STAGE(blk == 0 ? FWH_TAKE0 : FWH_TAKE1);
#pragma unroll
      for (int k = 0; k < 4; k++) wd_put(src + 64 * k, ~0ull, near);
#pragma unroll
      for (int k = 0; k < 4; k++) {
        z[2 * k] = (wd_lo(wv[k]) + m0[2 * k]) + m1[2 * k];
        z[2 * k + 1] = (wd_hi(wv[k]) + m0[2 * k + 1]) + m1[2 * k + 1];
      }
    }
    scale[blk] = ln_loss_gradient(z, xk, xv, bf2f(eta), s_gam + f0, s_bet + f0, gx[blk]);
    f32x16 g2;
#pragma unroll
    for (int e = 0; e < 8; e++) { g2[e] = gx[blk][e] * scale[blk]; g2[8 + e] = 0.f; }
    bf16x8 o, ol;
    split8_plain(g2, 0, o, ol);
    lds_put16(s_g2 + tok * FLD + f0, __builtin_bit_cast(u32x4, o));
    lds_put16(s_g2l + tok * FLD + f0, __builtin_bit_cast(u32x4, ol));
  };
  // b2 after mini-batch m: + the sum over the tokens of G2, eight shares in a fixed order.  Every lane keeps its own features.
  auto step_b2 = [&](int m) {
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const float* const q = s_b2p + k * FD;
      const f32x4 lo = *reinterpret_cast<const f32x4*>(q + f0), hi = *reinterpret_cast<const f32x4*>(q + f0 + 4);
#pragma unroll
      for (int e = 0; e < 4; e++) { b2v[e] += lo[e]; b2v[4 + e] += hi[e]; }
      b2L += q[lane];
    }
    if (u == 0 && half == 0) p.bias_img[((size_t)bh * FWD_WIDE_RING + m % FWD_WIDE_RING) * FWD_BIAS_FLOATS + HID + lane] = b2L;
  };
  // The slot that mini-batch mb's state goes to is free once the output branch, which only just keeps up, is done with mini-batch mb - RING:
  // waited for behind block 0's sums (72 pairs x 256 1.78 ms so, 1.86 ms ahead of them).
  auto ring_slot = [&](int mb) {
    if (u == 3 && mb >= FWD_WIDE_RING) {
      const int need = mb - FWD_WIDE_RING + 1;
      if (seen < need) {
        const uint64_t t0 = wall_clock64();
        while ((seen = __builtin_amdgcn_readfirstlane(__hip_atomic_load(words + WDW_TAKEN, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) < need) {
          if (__hip_atomic_load(w_status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 || wall_clock64() - t0 > p.wait_limit) {
            raise_status(w_status);
            gave_up = true;
            break;
          }
          __builtin_amdgcn_s_sleep(4);
        }
      }
    }
  };
  // this half's states of mini-batches 0 .. n - 1 are out
  auto give = [&](int n) {
    if (!near) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __hip_atomic_store(words + WDW_GIVEN + 8 * half, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };

  for (int mb = 0; mb < p.NC; mb++) {
    if (u == 0 && half == 0 && mb % p.cgs == 0) p.b2_ck[((size_t)bh * p.K + mb / p.cgs) * FD + lane] = b2L;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the marks put back in the last mini-batch are in place, its b2 is out
    // this mini-batch's XV and eta and the next one's XK: under way while the compute waves form block 0
    const bf16x8 xk[2] = {xk_n[0], xk_n[1]};
    bf16x8 xv[2];
    bf16 eta[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
      xv[k] = g_ld8h(gXV, voff, mb * TILE_BYTES + k * (TILE_BYTES / 2));
      eta[k] = g_ldh(gEta, 2 * t_in, mb * (CS * 2) + k * CS);
    }
    load_xk(mb + 1 < p.NC ? mb + 1 : mb);
    TTT_STAGE(FWH_ASK);
    __syncthreads();   // B1
    TTT_STAGE(FWH_B1);
    gather_send(mb, 0);
    put_xk(mb + 1);   // the buffer was last read a mini-batch ago
    TTT_STAGE(FWH_SEND0);
    finish_block(mb, 0, xk[0], xv[0], eta[0]);
    ring_slot(mb);
    TTT_STAGE(FWH_LN0);
    __syncthreads();   // B2
    TTT_STAGE(FWH_B2);
    gather_send(mb, 1);
    TTT_STAGE(FWH_SEND1);
    finish_block(mb, 1, xk[1], xv[1], eta[1]);
    if (gave_up && lane == 0) *s_flag = 1;
    TTT_STAGE(FWH_LN1);
    __syncthreads();   // B3
    TTT_STAGE(FWH_B3);
    if (flag() != 0) {
      if (lane == 0) report_status(w_status);
      return;
    }
    if (u == 0 && lane == 0 && mb > 0) give(mb);   // the stores of the last mini-batch's state were acknowledged before B3
    // b2's step, while the compute waves are busy: the four helper waves wait for each other's shares (all of them come here)
    ln_token_sum_store_product(s_b2p + u * FD, gx[0], scale[0], lane, f0);
    ln_token_sum_store_product(s_b2p + (4 + u) * FD, gx[1], scale[1], lane, f0);
    if (lane == 0) __hip_atomic_fetch_add(s_flag + 1, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    while (__hip_atomic_load(s_flag + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < 4 * (mb + 1)) __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    step_b2(mb);
    TTT_STAGE(FWH_B2STEP);
  }
  TTT_STAGES_END(bh, STAGE_ROLE_HALF + half);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (u == 0 && lane == 0) give(p.NC);
}

// Four workgroups per (batch, head) that share its recurrence and compute Out, or three: the two halves of the recurrence and one that
// computes Out.  Workgroups are dealt to the 8 XCDs in turn, so the grid is laid out for a multiple of 8 pairs
// (workgroups of pairs that do not exist leave at once) and the workgroups of a pair are 8 apart: same XCD, same L2.
template <bool QUAD>
TTT_DEV void fwd_wide(const FwdParams& p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const bool quad = QUAD || p.quad != 0;
  const int b = blockIdx.x, per = quad ? QD_CUS : 3;
  int bh = p.scatter ? b / per : (b / (8 * per)) * 8 + (b & 7);
  const int role = (p.scatter ? b : b >> 3) % per;
  if (bh >= p.nbh) return;
  bh += p.bh0;
  if (quad) {
    fwd_quad_recurrence(p, smem, bh, role);
    return;
  }
  if (role < 2) {
    fwd_wide_recurrence(p, smem, bh, role);
    return;
  }
  int* const words = p.sync + (size_t)bh * BWD_SYNC_STRIDE;
  if (threadIdx.x == 0) say_xcd(words + WDW_XCD + role);
  fwd_output_branch<1, true>(p, smem, bh);
}
__global__ __launch_bounds__(FW_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void ttt_mlp_fwd_wide_kernel(const FwdParams p) { fwd_wide<false>(p); }
// Four workgroups per pair and nothing else: 1 % shorter than the kernel that holds both launches in calls of a few hundred mini-batches (12 pairs x 32
// 163.3 -> 161.5 us, 24 x 256 1.228 -> 1.213 ms, 64 x 96 0.492 -> 0.486).
__global__ __launch_bounds__(FW_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void ttt_mlp_fwd_wide_early_kernel(const FwdParams p) {
  fwd_wide<true>(p);
}

// Clears the synchronisation words and marks every word of the exchange empty.
__global__ void ttt_mlp_fwd_wide_clear(int* w, int n, const int* report, uint4* x, int nx) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  clear_word(w, n, i, report);
  for (int k = i; k < nx; k += gridDim.x * blockDim.x) x[k] = make_uint4(~0u, ~0u, ~0u, ~0u);
}

}  // namespace ttt

hipError_t ttt_mlp_fwd_wide_enqueue(const ttt::FwdParams& p, TttKernel kernel, int grid, hipStream_t stream) {
  auto launch = [&](auto k) -> hipError_t {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, ttt::SM_FWD_BYTES);
    if (e != hipSuccess) return e;
    const int n = static_cast<int>(ttt::bwd_sync_ints(p.nbh));
    int* const words = p.status - (size_t)p.nbh * ttt::BWD_SYNC_STRIDE;   // p.sync and p.xchg are moved back by bh0 entries
    const int per = p.quad ? ttt::FWD_QUAD_XCHG_WORDS : ttt::FWD_XCHG_WORDS, nx = p.nbh * (per / 2);
    const int need = nx > n ? nx : n;
    hipLaunchKernelGGL(ttt::ttt_mlp_fwd_wide_clear, dim3((need + 255) / 256), dim3(256), 0, stream, words, n, p.report,
                       reinterpret_cast<uint4*>(p.xchg + (size_t)p.bh0 * per), nx);
    hipLaunchKernelGGL(k, dim3(grid), dim3(ttt::FW_THREADS), ttt::SM_FWD_BYTES, stream, p);
    return hipGetLastError();
  };
  switch (kernel) {
    TTT_FWD_WIDE_KERNELS(TTT_KERNEL_LAUNCH)
    default: return hipErrorInvalidValue;
  }
}
