// Reverse walk of one (batch, head) spread over four CUs, which form grad_L_XK, grad_L_XV and the norm gradients as well (up to 40
// pairs on 256 CUs: the walk's chain is the bound there).
//
// CU `part` of a pair holds the hidden columns part and part + 4 of the eight of 32 (a wave of the one-workgroup kernel each), so its
// sums over the hidden dimension, z_part + z_{part+4}, are the shares P_part that the other launch shapes add up as ((P0 + P1) + P2) + P3:
// same results to the bit.
//   waves 0-3 (one per SIMD)  two per shard: a token block of everything that has tokens, half of the features of the running
//                             gradients (16 + 16 registers, on two CUs 64); what the two need of each other crosses in LDS
//   waves 4-7                 sums over the CU's columns, their exchange, the LayerNorm of the CU's 16 tokens (two of the waves), its rows of
//                             grad_L_XK (the other two, a mini-batch later), the gradient wrt b2, the tiles
// Per mini-batch two exchanges are waited for: the shares of the gradient wrt dl/dZ2, each to the CU that takes those tokens through the
// LayerNorm, and its dZ2 to all; the shares of grad_L_XK cross while the next mini-batch's weight step runs.
//   BX  both halves of the running gradients in LDS       B1  shares in LDS         B2  dZ2 in LDS
//   B3  dZ1 in LDS                                        BE  shares of grad_L_XK, the next mini-batch's output-branch operands
//
// Messages carry no flag.  A word is empty when all its bits are set, and no message has such a word (a NaN keeps another pattern).  Sums have one
// reader, which marks the words empty again once it has them: two slots.  dZ2 has three, so its writer marks them, knowing from
// the next mini-batch's sums that they are past it: three slots.  Marks are put behind BX of the next mini-batch and are in
// place (vmcnt) before its B1, hence before this CU sends anything from which another could conclude that it may use the slot again.
//
// What bounds it: per-CU memory latency and issue, and then the chain.  A CU gets some 16 bytes per clock out of HBM (its requests in flight over the
// latency), a wave that asks for more waits to issue, and the words an exchange waits for queue behind what was asked for before them.  A mini-batch
// takes 74 KiB, so little is asked for between B1 and B2, where sums and dZ2 cross: W1 (needed behind B2) and the next Z1, whose GELU family the
// compute waves evaluate in that wait (as images from the replays it was 16 KiB more, and 11 k clocks more of each replay); images go
// straight to LDS where two waves need them (read twice by registers: 24 KiB more), and each stage's operands are asked for one or two
// stages ahead.  24 pairs x 512, clocks per mini-batch with the stage clocks in: all operands asked for in a row behind B1 18.5 k, that
// with tiles straight to LDS as well 20.9 k (4 bytes per lane and request; and behind such a request the compiler waits for all
// of them before it reads LDS), spread as here 17.4 k, the helper waves' own sums out of scratch memory 16.2 k: what the output branch
// adds 1.7 k, weight step backwards 2.8 k, sums out 0.9 k, their wait 2.7 k, LayerNorm 1.5 k, dZ2 crossing 1.3 k, inner MLP backwards 1.3 k, update
// 1.4 k, the rest barriers.  Times of launches are at the rule that chooses it (ttt_mlp_c_abi.hip).
#pragma once
#include "ttt_mlp_exchange.hpp"

namespace ttt {

constexpr int BWQ_CUS = 4;
// LDS carve-up of a workgroup of the walk (bytes)
constexpr int BWQ_XQ = 0;
constexpr int BWQ_GZB = BWQ_XQ + SB_TILE;                 // gZ2_bar
constexpr int BWQ_XK = BWQ_GZB + SB_TILE;
constexpr int BWQ_GZ2 = BWQ_XK + SB_TILE;             // dl/dZ2
constexpr int BWQ_DZ2 = BWQ_GZ2 + SB_TILE;
constexpr int BWQ_LTILE = 32 * LDF * 2;                   // per shard: W2 before the step and gW1 as rows [hid][F]
constexpr int BWQ_W2 = BWQ_DZ2 + SB_TILE;
constexpr int BWQ_GW1 = BWQ_W2 + 2 * BWQ_LTILE;
constexpr int BWQ_GW2 = BWQ_GW1 + 2 * BWQ_LTILE;          // per shard: gW2 as rows [F][hid], X2 and -eta u (later dZ1) as rows [tok][hid]
constexpr int BWQ_X2 = BWQ_GW2 + 2 * SB_WTILE;
constexpr int BWQ_U = BWQ_X2 + 2 * SB_WTILE;
constexpr int BWQ_IMG = BWQ_U + 2 * SB_WTILE;             // per shard: images of X2_bar, gZ1_bar and W1 before the step, four pieces each
constexpr int BWQ_P = BWQ_IMG + 2 * 3 * 4 * 1024;              // per compute wave: its share of a sum, [32 tok][F] fp32
constexpr int BWQ_PTILE = 32 * LDR * 4;
constexpr int BWQ_GY = BWQ_P + 4 * BWQ_PTILE;             // g_y of this CU's 16 tokens, fp32, two buffers
constexpr int BWQ_GB1 = BWQ_GY + 2 * 16 * FD * 4;         // gradient wrt b1, [shard][32]
constexpr int BWQ_GB2 = BWQ_GB1 + 2 * BW_NS * 4;
constexpr int BWQ_GAM = BWQ_GB2 + FD * 4;
constexpr int BWQ_DETA = BWQ_GAM + FD * 4;                // [shard][64 tokens]
constexpr int BWQ_ETA = BWQ_DETA + 2 * CS * 4;            // bf16
constexpr int BWQ_RED = BWQ_ETA + CS * 2;             // norm-gradient accumulators of this CU's two halves of 8 tokens, [half][2][64]
constexpr int BWQ_FLAG = BWQ_RED + 2 * 2 * FD * 4;        // [0] a wait gave up, [1] this CU is the last one of the walk
constexpr int BWQ_BYTES = BWQ_FLAG + 16;
static_assert(BWQ_BYTES <= SM_BWD_BYTES, "the launch asks for SM_BWD_BYTES (the replay's carve-up)");
// Words of the exchange (BWQ_XCHG_WORDS): sums as [2 slots][to CU][from another][2 halves of its 16 tokens][4 words and one for d eta][lane],
// the same for grad_L_XK without that word, dZ2 as [3 slots][CU][2 halves][2 words][lane]; then the norm-gradient sums at the end,
// [8 "waves" of 8 tokens][4][64] fp32.
constexpr int BWQ_XDK = 2 * BWQ_CUS * (BWQ_CUS - 1) * 2 * 5 * 64;
constexpr int BWQ_XDZ = BWQ_XDK + 2 * BWQ_CUS * (BWQ_CUS - 1) * 2 * 4 * 64;
constexpr int BWQ_XSUM = BWQ_XDZ + 3 * BWQ_CUS * 2 * 2 * 64;
static_assert(BWQ_XSUM + BW_NWAVE * 4 * FD / 2 == BWQ_XCHG_WORDS, "exchange of four CUs");
// Synchronisation words of a pair: BWW_WALKED, + 4 and 24 the groups done, 16 .. the XCD each workgroup runs on (+ 1), 25 the workgroups
// that are through.
constexpr int BWQW_XCD = 16, BWQW_JOIN = 25;

// A piece of an image (1 KiB, 16 bytes per lane) straight to LDS.  In assembly, since behind the builtin the compiler waits for the data before
// the wave's next read of LDS, whatever it reads; the wave waits (vmcnt) and meets the others at a barrier where the data is due.
TTT_DEV void image_to_lds(gptr_t img, unsigned off, int s, unsigned t16, bf16x8* dst) {
  const gptr_t g = img + static_cast<uint64_t>(uni(off + s * CHUNK_BYTES));
  const unsigned to = uni(static_cast<unsigned>(reinterpret_cast<uintptr_t>((lword_t)(dst + 64 * s))));
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(t16), "s"(g) : "memory", "m0");
}

TTT_DEV void bwd_quad_walk(const BwdParams& p, unsigned char* smem, const int bh, const int part) {
  typedef __attribute__((address_space(3))) int* lint_t;
  const lint_t s_flag = (lint_t)reinterpret_cast<int*>(smem + BWQ_FLAG);
  auto flag = [&](int i) { return __hip_atomic_load(s_flag + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, c = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int head = bh % p.NH;
  const int cgs = p.cgs, n_sets = p.n_sets;
  bf16* const s_xq = reinterpret_cast<bf16*>(smem + BWQ_XQ);
  bf16* const s_gzb = reinterpret_cast<bf16*>(smem + BWQ_GZB);
  bf16* const s_dz2 = reinterpret_cast<bf16*>(smem + BWQ_DZ2);
  float* const s_gb1 = reinterpret_cast<float*>(smem + BWQ_GB1);
  float* const s_gb2 = reinterpret_cast<float*>(smem + BWQ_GB2);
  float* const s_gam = reinterpret_cast<float*>(smem + BWQ_GAM);
  float* const s_deta = reinterpret_cast<float*>(smem + BWQ_DETA);
  float* const s_red = reinterpret_cast<float*>(smem + BWQ_RED);
  int* const words = p.sync + (size_t)bh * BWD_SYNC_STRIDE;
  bf16x8 ones;
#pragma unroll
  for (int j = 0; j < 8; j++) ones[j] = (bf16)1.0f;
  if (tid == 0) say_xcd(words + BWQW_XCD + part);
  if (tid < 2) s_flag[tid] = 0;
  if (tid < FD) {
    s_gam[tid] = p.ttt_norm_weight[head * FD + tid];
    s_gb2[tid] = p.grad_L_b2_last[(size_t)bh * FD + tid];
    s_gb1[tid] = p.grad_L_b1_last[(size_t)bh * HID + BW_NS * (part + 4 * (tid >> 5)) + (tid & 31)];
  }
  if (tid < 4 * FD) s_red[tid] = 0.f;
  // this (batch, head)'s part of each class of tensor (elements), and the per-group tensors of set `set`
  const size_t ox = uni64((size_t)bh * p.NC * (CS * FD)), oe = uni64((size_t)bh * p.NC * CS);
  const size_t of = uni64((size_t)bh * cgs * (CS * FD)), oh = uni64((size_t)bh * cgs * (CS * HID));
  const size_t ot = uni64((size_t)bh * cgs * CS), ock = uni64((size_t)bh * p.K * (FD * HID));
  // The pointers are read from the kernel-argument segment where they are used (see bwd_body).
  typedef const __attribute__((address_space(4))) BwdParams* KernArgs;
  KernArgs ka = (KernArgs)__builtin_amdgcn_kernarg_segment_ptr();
#define QGRP(name) (set ? ka->alt_##name[set - 1] : ka->name)
#define QSCHED() __builtin_amdgcn_sched_barrier(0)

  if (w < 4) {
    // ================================================================ compute waves
    const int sh = w & 1, tb = w >> 1;                     // shard of this CU's two; token block, and half of the features
    const int v = part + 4 * sh;                           // hidden block, = wave of the one-workgroup kernel
    const int hid0 = BW_NS * v;
    bf16* const s_w2 = reinterpret_cast<bf16*>(smem + BWQ_W2 + sh * BWQ_LTILE);
    bf16* const s_gw1 = reinterpret_cast<bf16*>(smem + BWQ_GW1 + sh * BWQ_LTILE);
    bf16* const s_gw2 = reinterpret_cast<bf16*>(smem + BWQ_GW2 + sh * SB_WTILE);
    bf16* const s_x2 = reinterpret_cast<bf16*>(smem + BWQ_X2 + sh * SB_WTILE);
    bf16* const s_u = reinterpret_cast<bf16*>(smem + BWQ_U + sh * SB_WTILE);
    float* const s_Pw = reinterpret_cast<float*>(smem + BWQ_P + w * BWQ_PTILE);
    bf16x8* const s_x2b = reinterpret_cast<bf16x8*>(smem + BWQ_IMG + sh * 3 * 4 * 1024);   // what the output branch adds (lane = hid, contraction = tok)
    bf16x8* const s_g1b = s_x2b + 4 * 64;
    bf16x8* const s_w1 = s_g1b + 4 * 64;             // (lane = F, contraction = hid)
    float* const s_gb1w = s_gb1 + BW_NS * sh;
    int lane_v = lane;
#define WQ_LANE                                                        \
  asm volatile("" : "+v"(lane_v));                                     \
  const int lane = lane_v & 63, h = lane >> 5, c = lane & 31;          \
  const unsigned t16 = 16 * ((v << 6) | lane);                         \
  (void)h; (void)c; (void)t16
    f32x16 gW1, gW2;   // of the running gradients: gW1[32 tb .., hid0 ..] (rows F), gW2[hid0 .., 32 tb ..] (rows hid)
    {
      const gptr_t g1 = gbuf(p.grad_L_W1_last + (size_t)bh * FD * HID), g2 = gbuf(p.grad_L_W2_last + (size_t)bh * HID * FD);
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int row = 8 * (i >> 2) + (i & 3);   // + 4h in the lane offset
        gW1[i] = g_ldf(g1, (4 * h * HID + c) * 4, ((32 * tb + row) * HID + hid0) * 4);
        gW2[i] = g_ldf(g2, (4 * h * FD + c) * 4, ((hid0 + row) * FD + 32 * tb) * 4);
      }
    }
    __syncthreads();   // flags
    __syncthreads();   // placement known, the first group is there, its last mini-batch's tiles too
    if (flag(0) != 0) return;
    // Operands of a mini-batch, asked for during the one before it (its state is half of a wave's registers elsewhere).
    bf16x8 w2bf[2];                   // this wave's half of W2 before the step (lane = hid, contraction = F)
    bf16x8 gq[2], aq[2], bq[2];       // gelu, gelu', gelu'' of Z1 of this wave's tokens, evaluated a mini-batch ahead (gq: Z1 until then)
    gptr_t gX2B, gGZ1B, gI1, gI2, gZ;
    auto group_images = [&](int set) {
      gX2B = gbuf(QGRP(X2_bar_group) + oh);
      gGZ1B = gbuf(QGRP(Z1_bar_group) + oh);
      gI1 = gbuf(QGRP(X2_group) + oh);
      gI2 = gbuf(QGRP(grad_l_wrt_Z1_group) + oh);
      gZ = gbuf(QGRP(Z1_group) + oh);
    };
    const gptr_t gCk1 = gbuf(ka->W1_ck + ock), gCk2 = gbuf(ka->W2_ck + ock);
    auto ask_bar = [&](int j) {
      WQ_LANE;
#pragma unroll
      for (int t = 0; t < 2; t++) {
        image_to_lds(gX2B, j * IMG_BYTES, 2 * tb + t, t16, s_x2b);
        image_to_lds(gGZ1B, j * IMG_BYTES, 2 * tb + t, t16, s_g1b);
      }
    };
    auto ask_step = [&](int k, int j) {
      WQ_LANE;
      if (j > 0) {
#pragma unroll
        for (int t = 0; t < 2; t++) w2bf[t] = chunk_load(gI2, (j - 1) * IMG_BYTES, 2 * tb + t, t16);
      } else {
#pragma unroll
        for (int t = 0; t < 2; t++) w2bf[t] = piece_from_f32(gCk2, static_cast<unsigned>(k) * (FD * HID * 4u), FD, hid0, 0, 2 * tb + t, c, h);
      }
    };
    auto ask_z = [&](int j) {
      WQ_LANE;
#pragma unroll
      for (int t = 0; t < 2; t++) gq[t] = image_load(gZ, j * IMG_BYTES, 2 * tb + t, t16);
    };
    auto gelu = [&]() {
#pragma unroll
      for (int t = 0; t < 2; t++) {
        const bf16x8 z = gq[t];
        gelu_images<false>(z, gq[t], aq[t], bq[t]);
        asm volatile("" : "+v"(gq[t]), "+v"(aq[t]), "+v"(bq[t]));   // finished here
      }
    };
    // gb1 += row sums of a 32-row operand of four pieces, formed on the matrix cores (as lds_rowsum_add_jit)
    auto rowsum = [&](const bf16x8 (&a)[4]) {
      f32x16 t;
#pragma unroll
      for (int i = 0; i < 16; i++) t[i] = 0.f;
#pragma unroll
      for (int s = 0; s < 4; s++) t = MFMA(a[s], ones, t);
      return t;
    };
    auto add_gb1 = [&](const f32x16& t) {
      WQ_LANE;
      if (c == 0) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
          f32x4 old = *reinterpret_cast<const f32x4*>(s_gb1w + 8 * g + 4 * h);
#pragma unroll
          for (int e = 0; e < 4; e++) old[e] += t[4 * g + e];
          *reinterpret_cast<f32x4*>(s_gb1w + 8 * g + 4 * h) = old;
        }
      }
      WAVE_SYNC();
    };
    auto store_share = [&](const f32x16 (&z)[2]) {   // [32 tok][F]
      WQ_LANE;
#pragma unroll
      for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          f32x4 q = {z[rb][4 * g], z[rb][4 * g + 1], z[rb][4 * g + 2], z[rb][4 * g + 3]};
          *reinterpret_cast<f32x4*>(s_Pw + c * LDR + 32 * rb + 8 * g + 4 * h) = q;
        }
    };
    int n = 0;   // mini-batches walked
    TTT_STAGES_BEGIN();
    group_images(0);
    {
      const int j0 = min(cgs, p.NC - (p.K - 1) * cgs) - 1;
      ask_bar(j0);
      ask_step(p.K - 1, j0);
      ask_z(j0);
      gelu();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();   // the first tiles
    __builtin_amdgcn_s_setprio(1);
    for (int k = p.K - 1; k >= 0; k--) {
      const int n_mb = min(cgs, p.NC - k * cgs);
      const int done = p.K - 1 - k;
      for (int j = n_mb - 1; j >= 0; j--, n++) {
        const bf16* const s_xk = reinterpret_cast<const bf16*>(smem + BWQ_XK);
        const bf16* const s_gz2 = reinterpret_cast<const bf16*>(smem + BWQ_GZ2);
        const bf16* const s_eta = reinterpret_cast<const bf16*>(smem + BWQ_ETA);
        // ---- what the output branch adds to the running gradients
        {
          WQ_LANE;
          bf16x8 x2b[4], g1b[4], zb[4], xq[4];
#pragma unroll
          for (int s = 0; s < 4; s++) {
            x2b[s] = s_x2b[64 * s + lane];
            g1b[s] = s_g1b[64 * s + lane];
          }
#pragma unroll
          for (int s = 0; s < 4; s++) zb[s] = xpiece_tr(s_gzb, tb, s, lane);
#pragma unroll
          for (int s = 0; s < 4; s++) xq[s] = xpiece_tr(s_xq, tb, s, lane);
          QSCHED();
#pragma unroll
          for (int s = 0; s < 4; s++) {
            gW2 = MFMA(x2b[s], zb[s], gW2);
            gW1 = MFMA(xq[s], g1b[s], gW1);
          }
          if (tb == 0) add_gb1(rowsum(g1b));
#pragma unroll
          for (int t = 0; t < 2; t++) {
            store_piece_rows<LDH>(s_gw2, tb, t, c, h, pack8(gW2, t));
            store_piece_rows<LDF>(s_gw1, 0, 2 * tb + t, c, h, pack8(gW1, t));
          }
#pragma unroll
          for (int t = 0; t < 2; t++) store_piece_rows<LDF>(s_w2, 0, 2 * tb + t, c, h, w2bf[t]);
        }
        QSCHED();
        TTT_STAGE(BQC_BAR);
        __syncthreads();                                    // BX: both halves of the running gradients
        TTT_STAGE(BQC_BX);
        QSCHED();
        // ---- the weight step, backwards (state BEFORE this mini-batch)
        bf16x8 t2p[2], d1p[2], g1[2];   // d1p: gelu'(Z1)
        bf16x8 gz[4];
        float neg_eta;
        {
          WQ_LANE;
          neg_eta = -bf2f(s_eta[32 * tb + c]);
          AccT<1, 1> R, S;   // R = gZ2 W2^T, S = XK gW1 + gb1   (rows hid, lane = tok)
          acc_zero(R);
          acc_init_rows_lds(S, s_gb1w, h);
          bf16x8 w2r[4], w1r[4], xk[4];
#pragma unroll
          for (int s = 0; s < 4; s++) {
            gz[s] = xpiece_rows(s_gz2, tb, s, c, h);
            w2r[s] = piece_rows<LDF>(s_w2, 0, s, c, h);
            w1r[s] = piece_rows<LDF>(s_gw1, 0, s, c, h);
            xk[s] = xpiece_rows(s_xk, tb, s, c, h);
          }
          QSCHED();
          bf16x8 gw2[2][2], w2t[2][2];
#pragma unroll
          for (int s = 0; s < 4; s++) {
            R.b[0][0] = MFMA(w2r[s], gz[s], R.b[0][0]);
            S.b[0][0] = MFMA(w1r[s], xk[s], S.b[0][0]);
            if (s == 1) {
              QSCHED();
#pragma unroll
              for (int t = 0; t < 2; t++)
#pragma unroll
                for (int rb = 0; rb < 2; rb++) gw2[rb][t] = piece_rows<LDH>(s_gw2, rb, t, c, h);   // lane = F, contraction = hid
              QSCHED();
            }
          }
          f32x16 pz[2];
#pragma unroll
          for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int e = 0; e < 16; e++) pz[rb][e] = 0.f;
#pragma unroll
          for (int t = 0; t < 2; t++)
#pragma unroll
            for (int rb = 0; rb < 2; rb++) pz[rb] = MFMA(gw2[rb][t], gq[t], pz[rb]);   // gW2^T X2^T
          float de = 0.f;
          bf16x8 uc[2], uh[2];
#pragma unroll
          for (int t = 0; t < 2; t++) {
#pragma unroll
            for (int jj = 0; jj < 8; jj++) {
              const float a = (float)aq[t][jj], b = (float)bq[t][jj];
              const float r0 = R.b[0][0][8 * t + jj], sv = S.b[0][0][8 * t + jj];
              const float gz1 = r0 * a;                                   // dl/dZ1
              de = __builtin_fmaf(gz1, sv, de);
              uc[t][jj] = (bf16)(sv * a);
              uh[t][jj] = (bf16)(neg_eta * sv * a);
              t2p[t][jj] = (bf16)(neg_eta * r0 * sv * b);
              g1[t][jj] = (bf16)(neg_eta * gz1);
            }
            d1p[t] = aq[t];
            store_piece_rows<LDH>(s_x2, tb, t, c, h, gq[t]);              // X2 rows [tok][hid]
            store_piece_rows<LDH>(s_u, tb, t, c, h, uh[t]);               // -eta u rows [tok][hid]
          }
          QSCHED();
#pragma unroll
          for (int t = 0; t < 2; t++)
#pragma unroll
            for (int rb = 0; rb < 2; rb++) w2t[rb][t] = piece_tr<LDF>(s_w2, rb, t, lane);
          QSCHED();
#pragma unroll
          for (int s = 0; s < 4; s++)
#pragma unroll
            for (int jj = 0; jj < 8; jj++) de = __builtin_fmaf((float)gz[s][jj], pz[s >> 1][8 * (s & 1) + jj], de);
#pragma unroll
          for (int t = 0; t < 2; t++)
#pragma unroll
            for (int rb = 0; rb < 2; rb++) pz[rb] = MFMA(w2t[rb][t], uc[t], pz[rb]);   // + W2^T u^T
          const float a = half_sum_valu(de);
          if (h == 0) s_deta[sh * CS + 32 * tb + c] = a;
          store_share(pz);
        }
        QSCHED();
        TTT_STAGE(BQC_STEP);
        __syncthreads();                                    // B1: the sums
        TTT_STAGE(BQC_B1);
        QSCHED();
        if (j > 0) {   // (a group's first mini-batch takes it from the checkpoint, below)
          WQ_LANE;
#pragma unroll
          for (int t = 0; t < 2; t++)
            image_to_lds(gI1, (j - 1) * IMG_BYTES, 2 * tb + t, t16, s_w1);
        }
        QSCHED();
        if (j == 0) group_images((done + 1) % n_sets);   // (the helpers made sure of it before B1)
        const int kn = j > 0 || k == 0 ? k : k - 1, jn = j > 0 ? j - 1 : k == 0 ? 0 : cgs - 1;   // (behind the last mini-batch: dropped)
        ask_z(jn);
        // ---- while they cross: the products that do not need them, and the next mini-batch's GELU family
        f32x16 q, dk[2];
        {
          WQ_LANE;
          bf16x8 gw[4], ut[4], gt[4];
#pragma unroll
          for (int s = 0; s < 4; s++) {
            gw[s] = piece_tr<LDH>(s_gw2, 0, s, lane);
            ut[s] = piece_tr<LDH>(s_u, 0, s, lane);
            gt[s] = xpiece_tr(s_gz2, tb, s, lane);
          }
#pragma unroll
          for (int e = 0; e < 16; e++) q[e] = dk[0][e] = dk[1][e] = 0.f;
#pragma unroll
          for (int s = 0; s < 4; s++) {
            q = MFMA(gw[s], gz[s], q);                       // gZ2 gW2^T
            gW2 = MFMA(ut[s], gt[s], gW2);                   // (-eta u)^T gZ2
          }
#pragma unroll
          for (int t = 0; t < 2; t++)
#pragma unroll
            for (int rb = 0; rb < 2; rb++) dk[rb] = MFMA(piece_tr<LDF>(s_gw1, rb, t, lane), g1[t], dk[rb]);   // gW1 G1^T
#pragma unroll
          for (int e = 0; e < 16; e++) q[e] *= neg_eta;
          QSCHED();
          if (j == 0) {
#pragma unroll
            for (int t = 0; t < 2; t++) s_w1[64 * (2 * tb + t) + lane] = piece_from_f32(gCk1, static_cast<unsigned>(k) * (FD * HID * 4u), HID, 32 * tb, hid0, t, c, h);
          }
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // W1 is there
          gelu();
        }
        QSCHED();
        TTT_STAGE(BQC_PRODUCTS);
        __syncthreads();                                    // B2: dZ2
        TTT_STAGE(BQC_B2);
        QSCHED();
        const int gone = flag(0);   // (asked for here, looked at behind the products)
        {
          WQ_LANE;
          bf16x8 w2r[4], dr[4], x2[4], dt[4];
#pragma unroll
          for (int s = 0; s < 4; s++) {
            w2r[s] = piece_rows<LDF>(s_w2, 0, s, c, h);
            dr[s] = piece_rows<LDX>(s_dz2, tb, s, c, h);
          }
          QSCHED();
          ask_bar(jn);
          QSCHED();
#pragma unroll
          for (int s = 0; s < 4; s++) q = MFMA(w2r[s], dr[s], q);                              // + dZ2 W2^T
          QSCHED();
#pragma unroll
          for (int s = 0; s < 4; s++) {
            x2[s] = piece_tr<LDH>(s_x2, 0, s, lane);
            dt[s] = piece_tr<LDX>(s_dz2, tb, s, lane);
          }
          QSCHED();
          bf16x8 dz[2];
#pragma unroll
          for (int t = 0; t < 2; t++) {
#pragma unroll
            for (int jj = 0; jj < 8; jj++) dz[t][jj] = (bf16)__builtin_fmaf(q[8 * t + jj], (float)d1p[t][jj], (float)t2p[t][jj]);   // dZ1
            store_piece_rows<LDH>(s_u, tb, t, c, h, dz[t]);                                    // rows [tok][hid]
          }
          if (gone != 0) return;
          QSCHED();
#pragma unroll
          for (int s = 0; s < 4; s++) gW2 = MFMA(x2[s], dt[s], gW2);                           // + X2^T dZ2
#pragma unroll
          for (int t = 0; t < 2; t++)
#pragma unroll
            for (int rb = 0; rb < 2; rb++) dk[rb] = MFMA(s_w1[64 * (2 * rb + t) + lane], dz[t], dk[rb]);          // + W1 dZ1^T
        }
        QSCHED();
        TTT_STAGE(BQC_MLP);
        __syncthreads();                                    // B3: dZ1
        TTT_STAGE(BQC_B3);
        QSCHED();
        {
          WQ_LANE;
          bf16x8 dz1[4], xkt[4];
#pragma unroll
          for (int s = 0; s < 4; s++) {
            dz1[s] = piece_tr<LDH>(s_u, 0, s, lane);
            xkt[s] = xpiece_tr(s_xk, tb, s, lane);
          }
          QSCHED();
          ask_step(kn, jn);
          QSCHED();
#pragma unroll
          for (int s = 0; s < 4; s++) gW1 = MFMA(xkt[s], dz1[s], gW1);                         // + XK^T dZ1
          if (tb == 1) add_gb1(rowsum(dz1));
          store_share(dk);
        }
        asm volatile("s_waitcnt vmcnt(2)" ::: "memory");   // the next mini-batch's images are there (what ask_step asked for is two loads at least)
        QSCHED();
        TTT_STAGE(BQC_UPDATE);
        __syncthreads();                                    // BE: grad_L_XK's shares; the next mini-batch's tiles
        TTT_STAGE(BQC_BE);
        QSCHED();
      }
    }
    if (part < 2) TTT_STAGES_END(bh, STAGE_ROLE_WALK_HALF + part);
    {
      const gptr_t g1 = gbuf(p.grad_L_W1_init + (size_t)bh * FD * HID), g2 = gbuf(p.grad_L_W2_init + (size_t)bh * HID * FD);
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int row = 8 * (i >> 2) + (i & 3);
        g_stf(g1, (4 * h * HID + c) * 4, ((32 * tb + row) * HID + hid0) * 4, gW1[i]);
        g_stf(g2, (4 * h * FD + c) * 4, ((hid0 + row) * FD + 32 * tb) * 4, gW2[i]);
      }
      if (tb == 0 && lane < BW_NS) p.grad_L_b1_init[(size_t)bh * HID + hid0 + lane] = s_gb1w[lane];
    }
    __syncthreads();
    return;
  }

  // ================================================================== helper waves
  const int u = w - 4;                                   // number among them
  const int q8 = lane >> 3, f0 = 8 * (lane & 7);
  const int t_in = 8 * u + q8;                           // the rows that this lane sums, sends and brings in: token t_in of both blocks
  // This CU's 16 tokens (half u & 1 of them, as rows of 8 lanes each): two waves, whose rows they are anyway, take their sums through the
  // LayerNorm and give dZ2, grad_L_XV and d eta; the other two finish grad_L_XK of them a mini-batch later.
  const bool owns = (u >> 1) == (part & 1);
  const int half = u & 1, own_blk = part >> 1, own_tok = 16 * part + 8 * half + q8;
  const unsigned voff = (t_in * FD + f0) * 2, own_off = (own_tok * FD + f0) * 2;
  int* const w_status = p.status;
  bool gave_up = false;   // (kept to itself until the stage whose closing barrier precedes the reads of s_flag[0])
  __syncthreads();   // flags
  auto wait_group = [&](int done) {   // group number `done` (from the end) has been replayed
    if (!__all(lane != 0 || wait_word(words + done % n_sets, parts_until(p, done), w_status, p.wait_limit))) gave_up = true;
  };
  // What these waves themselves take for their token.
  struct Own {
    bf16x8 xh, go, old;   // old: what grad_L_XV (waves that own) or grad_L_XK held
    float sd;
    bf16 eta, deta;
  } nw;
  // Where all that comes from (the group's at the last group_tiles): read from the kernel arguments once, not where it is used, since a read
  // of those waits for the wave's reads of LDS as well.
  const bool ow = p.overwrite != 0;
  const gptr_t bXQ = gbuf(p.XQ + ox), bXK = gbuf(p.XK + ox), bETA = gbuf(p.last_eta + oe);
  const gptr_t bOLD = ow ? gbuf(zero_tile) : owns ? gbuf(p.grad_L_XV + ox) : gbuf(p.grad_L_XK + ox);
  const gptr_t bOLDE = ow ? gbuf(zero_tile) : gbuf(p.grad_L_last_eta + oe);
  gptr_t bZB, bGZ, bXH, bGO, bSD;
  auto group_tiles = [&](int set) {
    asm volatile("" : "+s"(ka));
    bZB = gbuf(QGRP(grad_x_hat_fused_group) + of);
    bGZ = gbuf(QGRP(grad_l_wrt_Z2_group) + of);
    bXH = gbuf(QGRP(x_hat_fused_group) + of);
    bGO = gbuf(QGRP(grad_output_fused_group) + of);
    bSD = gbuf(QGRP(std_fused_group) + ot);
  };
  auto ask = [&](int k, int j) {
    const int mb = k * cgs + j;
    if (owns) {
      nw.xh = g_ld_stream<bf16x8>(bXH, own_off, j * TILE_BYTES);
      nw.go = g_ld_stream<bf16x8>(bGO, own_off, j * TILE_BYTES);
      nw.sd = g_ldf(bSD, 4 * own_tok, j * (CS * 4));
      nw.eta = g_ldh(bETA, 2 * own_tok, mb * (CS * 2));
      nw.deta = g_ldh(bOLDE, 2 * own_tok, ow ? 0u : mb * (CS * 2));
    }
    nw.old = g_ld_stream<bf16x8>(bOLD, own_off, ow ? 0u : mb * TILE_BYTES);
  };
  // The tiles of a mini-batch, token row t_in of both blocks: what the output branch needs, and the other two.
  struct Tiles {
    bf16x8 xq[2], zb[2], xk[2], gz[2];
    bf16 eta;
  } nx;
  auto ask_out = [&](int k, int j) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      nx.xq[i] = g_ld8h(bXQ, voff, (k * cgs + j) * TILE_BYTES + i * (TILE_BYTES / 2));
      nx.zb[i] = g_ld_stream<bf16x8>(bZB, voff, j * TILE_BYTES + i * (TILE_BYTES / 2));
    }
  };
  auto ask_step = [&](int k, int j) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      nx.xk[i] = g_ld8h(bXK, voff, (k * cgs + j) * TILE_BYTES + i * (TILE_BYTES / 2));
      nx.gz[i] = g_ld_stream<bf16x8>(bGZ, voff, j * TILE_BYTES + i * (TILE_BYTES / 2));
    }
    if (u == 0) nx.eta = g_ldh(bETA, 2 * lane, (k * cgs + j) * (CS * 2));
  };
  auto put_out = [&]() {
    bf16* const q = reinterpret_cast<bf16*>(smem) + xrow(t_in) + f0;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      ln_store_h(q + BWQ_XQ / 2 + i * (16 * XPAIR), nx.xq[i]);
      ln_store_h(q + BWQ_GZB / 2 + i * (16 * XPAIR), nx.zb[i]);
    }
  };
  auto put_step = [&]() {
    bf16* const q = reinterpret_cast<bf16*>(smem) + xrow(t_in) + f0;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      ln_store_h(q + BWQ_XK / 2 + i * (16 * XPAIR), nx.xk[i]);
      ln_store_h(q + BWQ_GZ2 / 2 + i * (16 * XPAIR), nx.gz[i]);
    }
    if (u == 0) reinterpret_cast<bf16*>(smem + BWQ_ETA)[lane] = nx.eta;
  };
  bool alive = true;
  const bool near = on_one_xcd(words + BWQW_XCD, BWQ_CUS, lane, w_status, p.wait_limit, alive);
  if (!alive) gave_up = true;
  wait_group(0);   // (every helper wave itself)
  if (!gave_up) {
    const int j0 = min(cgs, p.NC - (p.K - 1) * cgs) - 1;
    group_tiles(0);
    ask_out(p.K - 1, j0);
    ask_step(p.K - 1, j0);
    put_out();
  }
  if (gave_up && lane == 0) s_flag[0] = 1;
  __syncthreads();
  if (flag(0) != 0) {
    if (lane == 0) report_status(w_status);
    return;
  }
  __syncthreads();   // the first tiles
  const gptr_t xch = gbuf(p.xchg + (size_t)bh * BWQ_XCHG_WORDS);
  auto words_at = [&](unsigned first) {   // (a scalar base and the lane's offset, as in g_ld)
    gptr_t q = xch + static_cast<uint64_t>(uni(8 * first));
    unsigned o = 8 * lane;
    asm("" : "+s"(q), "+v"(o));
    return (gword64_t)(q + static_cast<uint64_t>(o));
  };
  auto message = [&](int n, int to, int from) { return (((n & 1) * BWQ_CUS + to) * (BWQ_CUS - 1) + from - (from > to ? 1 : 0)) * 2 + half; };
  auto p_slot = [&](int n, int to, int from) { return words_at(message(n, to, from) * (5 * 64)); };
  auto k_slot = [&](int n, int to, int from) { return words_at(BWQ_XDK + message(n, to, from) * (4 * 64)); };
  auto z_slot = [&](int slot, int cu, int half) { return words_at(BWQ_XDZ + ((slot * BWQ_CUS + cu) * 2 + half) * (2 * 64)); };
  auto put_words = [&](gword64_t dst, const auto& x) {   // (one branch for all of them)
    constexpr int N = sizeof(x) / sizeof(uint64_t);
    if (near) {
#pragma unroll
      for (int k = 0; k < N; k++) wd_put(dst + 64 * k, x[k], true);
    } else {
#pragma unroll
      for (int k = 0; k < N; k++) wd_put(dst + 64 * k, x[k], false);
    }
  };
  auto other = [&](int o) { return o + (o >= part ? 1 : 0); };   // the CUs but this one
  // Waits for N messages of W words per lane, number i at at(i); `meanwhile` once, between the first request and its answer.
  auto take = [&](auto at, auto& x, auto meanwhile) __attribute__((always_inline)) {
    constexpr int N = sizeof(x) / sizeof(x[0]), W = sizeof(x[0]) / sizeof(uint64_t);
    uint64_t t0 = 0;
    for (unsigned i_try = 0;; i_try++) {
#pragma unroll
      for (int i = 0; i < N; i++) {
        const gword64_t src = at(i);
#pragma unroll
        for (int k = 0; k < W; k++) x[i][k] = __hip_atomic_load(src + 64 * k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      if (i_try == 0) meanwhile();
      uint32_t most = 0;   // (the mark is the largest of all words)
#pragma unroll
      for (int i = 0; i < N; i++)
#pragma unroll
        for (int k = 0; k < W; k++) most = max(most, max(static_cast<uint32_t>(x[i][k]), static_cast<uint32_t>(x[i][k] >> 32)));
      if (__all(most != WD_EMPTY)) return;
      if (i_try == 1 || (i_try & 7) == 0) {   // (the clock is not asked every time: its answer takes as long as the words')
        const uint64_t now = wall_clock64();
        if (i_try == 0) t0 = now;
        else if (now - t0 > p.wait_limit || ((i_try & 63) == 0 && __hip_atomic_load(w_status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
          raise_status(w_status);
          gave_up = true;
          return;
        }
      }
    }
  };
  auto nothing = []() {};
  // Sum over this CU's hidden columns for token row t of block blk.
  auto gather = [&](int blk, int t, float (&m)[8]) {
    const float* const row = reinterpret_cast<const float*>(smem + BWQ_P + 2 * blk * BWQ_PTILE) + t * LDR + f0;
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const f32x4 s = *reinterpret_cast<const f32x4*>(row + 4 * q) + *reinterpret_cast<const f32x4*>(row + BWQ_PTILE / 4 + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; e++) m[4 * q + e] = s[e];
    }
  };
  // The four CUs' shares in their order, ((P0 + P1) + P2) + P3: this CU's own and what came from the others.
  auto sum_shares = [&](float (&z)[8], const float (&own)[8], const auto& x) {
    auto add_other = [&](int o) {
#pragma unroll
      for (int k = 0; k < 4; k++) { z[2 * k] += wd_lo(x[o][k]); z[2 * k + 1] += wd_hi(x[o][k]); }
    };
    auto add_own = [&]() {
#pragma unroll
      for (int e = 0; e < 8; e++) z[e] += own[e];
    };
    if (part == 0) {
#pragma unroll
      for (int e = 0; e < 8; e++) z[e] = own[e];
      add_other(0);
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++) { z[2 * k] = wd_lo(x[0][k]); z[2 * k + 1] = wd_hi(x[0][k]); }
      if (part == 1) add_own();
    }
    add_other(1);
    if (part == 2) add_own();
    add_other(2);
    if (part == 3) add_own();
  };
  const gptr_t bDETA = gbuf(p.grad_L_last_eta + oe), bDXV = gbuf(p.grad_L_XV + ox), bDXK = gbuf(p.grad_L_XK + ox);
  float* const s_dgw = s_red + half * 2 * FD;
  float* const s_dbw = s_dgw + FD;
  float nr0 = 0.f, nr1 = 0.f;   // the replays' share of the norm gradients, of "wave" 2 part + half
  float gam[8];
  ln_load_f32(gam, s_gam + f0);
  // grad_L_XK's sums of the mini-batch before, gathered ahead of BX and sent behind it (own tokens': mo)
  float so[2][8], mo[8];
  bf16x8 dxk_old;               // what grad_L_XK held in that mini-batch
#pragma unroll
  for (int e = 0; e < 8; e++) { mo[e] = 0.f; dxk_old[e] = (bf16)0.f; }
  auto gather_dk = [&]() {
    gather(0, t_in, so[0]);
    gather(1, t_in, so[1]);
    if (!owns) gather(own_blk, own_tok & 31, mo);
  };
  auto give_dk = [&](int n) {
#pragma unroll
    for (int blk = 0; blk < 2; blk++) {
      const int to = 2 * blk + (u >> 1);
      if (to != part) {
        const float (&m)[8] = so[blk];
        const uint64_t x[4] = {wd_pack(m[0], m[1]), wd_pack(m[2], m[3]), wd_pack(m[4], m[5]), wd_pack(m[6], m[7])};
        put_words(k_slot(n, to, part), x);
      }
    }
  };
  auto finish_dk = [&](int n, int mb) {
    uint64_t x[BWQ_CUS - 1][4];
    auto from = [&](int o) { return k_slot(n, part, other(o)); };
    take(from, x, nothing);
    const uint64_t marks[4] = {~0ull, ~0ull, ~0ull, ~0ull};
#pragma unroll
    for (int o = 0; o < BWQ_CUS - 1; o++) put_words(from(o), marks);
    float z[8];
    sum_shares(z, mo, x);
    const float* const y = reinterpret_cast<const float*>(smem + BWQ_GY) + (n & 1) * (16 * FD) + (8 * half + q8) * FD + f0;
#pragma unroll
    for (int e = 0; e < 8; e++) z[e] = (float)dxk_old[e] + (z[e] + y[e]);
    g_st_stream<bf16x8>(bDXK, own_off, mb * TILE_BYTES, cvt8(z));
  };

  int n = 0, slot = 0, mb_before = 0;   // slot = n % 3
  TTT_STAGES_BEGIN();
  for (int k = p.K - 1; k >= 0; k--) {
    const int n_mb = min(cgs, p.NC - k * cgs);
    const int done = p.K - 1 - k, set = done % n_sets;
    for (int j = n_mb - 1; j >= 0; j--, n++, slot = slot == 2 ? 0 : slot + 1) {
      const int mb = k * cgs + j;
      gather_dk();       // (of the mini-batch before; nothing there yet in the first one, and not sent)
      put_step();        // (XK is read up to BE)
      TTT_STAGE(BQH_GATHER);
      __syncthreads();   // BX
      TTT_STAGE(BQH_BX);
      ask(k, j);
      if (n > 0) {
        give_dk(n - 1);
        if (owns) {   // read by now, in all four CUs: the sums of the mini-batch before, and dZ2 of the one before that
          const uint64_t marks[5] = {~0ull, ~0ull, ~0ull, ~0ull, ~0ull}, marks2[2] = {~0ull, ~0ull};
#pragma unroll
          for (int o = 0; o < BWQ_CUS - 1; o++) put_words(p_slot(n - 1, part, other(o)), marks);
          put_words(z_slot(slot == 2 ? 0 : slot + 1, part, half), marks2);
        }
      }
      // gradient wrt b2: what the output branch adds
      if (u < 2) lds_rowsum_add_jit(s_gb2 + 32 * u, [&](int s) { return xpiece_tr(s_gzb, u, s, lane); }, ones, c, h);
      const bool more = n + 1 < p.NC;
      if (j == 0 && k > 0) wait_group(done + 1);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the marks are in place, and nothing is in the way of the sums
      TTT_STAGE(BQH_ASK);
      __builtin_amdgcn_s_setprio(2);   // from here to B2 these waves' instructions are what the other four wait for
      __syncthreads();   // B1
      TTT_STAGE(BQH_B1);
      {
        f32x4 z[2][2][2];
        float e[2][2];
#pragma unroll
        for (int blk = 0; blk < 2; blk++) {
#pragma unroll
          for (int q = 0; q < 2; q++)
#pragma unroll
            for (int i = 0; i < 2; i++)
              z[blk][q][i] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(smem + BWQ_P + (2 * blk + i) * BWQ_PTILE) + t_in * LDR + f0 + 4 * q);
          e[blk][0] = s_deta[32 * blk + t_in];
          e[blk][1] = s_deta[CS + 32 * blk + t_in];
        }
        QSCHED();   // (all of them asked for before the first is used)
#pragma unroll
        for (int blk = 0; blk < 2; blk++) {
          const int to = 2 * blk + (u >> 1);
          if (to != part) {
            const f32x4 a = z[blk][0][0] + z[blk][0][1], b = z[blk][1][0] + z[blk][1][1];
            const uint64_t x[5] = {wd_pack(a[0], a[1]), wd_pack(a[2], a[3]), wd_pack(b[0], b[1]), wd_pack(b[2], b[3]), wd_pack(e[blk][0] + e[blk][1], 0.f)};
            put_words(p_slot(n, to, part), x);
          }
        }
      }
      TTT_STAGE(BQH_SEND);
      // Message i of the six that carry the other CUs' dZ2: two for a wave that finishes grad_L_XK, one for a wave that has its own to form.
      auto take_dz = [&](auto& x, int first, auto meanwhile) {
        constexpr int N = sizeof(x) / sizeof(x[0]);
        take([&](int i) { return z_slot(slot, other((first + i) >> 1), (first + i) & 1); }, x, meanwhile);
#pragma unroll
        for (int i = 0; i < N; i++) {
          const u32x4 y = {static_cast<uint32_t>(x[i][0]), static_cast<uint32_t>(x[i][0] >> 32), static_cast<uint32_t>(x[i][1]), static_cast<uint32_t>(x[i][1] >> 32)};
          const int tok = 16 * other((first + i) >> 1) + 8 * ((first + i) & 1) + q8;
          ln_store_h(s_dz2 + tok * LDX + f0, __builtin_bit_cast(bf16x8, y));
        }
      };
      bf16x8 out;   // grad_L_XV (waves that own)
      bf16 deta;
      if (owns) {
        uint64_t x[BWQ_CUS - 1][5];
        auto from = [&](int o) { return p_slot(n, part, other(o)); };
        float gb[8], xh[8], go[8], gz[8], own[8], d_own;
        take(from, x, [&]() {
          gather(own_blk, own_tok & 31, own);
          d_own = s_deta[own_tok] + s_deta[CS + own_tok];
          ln_load_f32(gb, s_gb2 + f0);
          ln_cvt8(xh, nw.xh);
          ln_cvt8(go, nw.go);
          ln_load(gz, reinterpret_cast<const bf16*>(smem + BWQ_GZ2) + xrow(own_tok) + f0);
        });
        TTT_STAGE(BQH_TAKE);
        float gg[8], gy[8], dg[8], dz[8];
        sum_shares(gg, own, x);
        const float d0 = wd_lo(x[0][4]), d1 = wd_lo(x[1][4]), d2 = wd_lo(x[2][4]);
        const float d_sum = ((part == 0 ? d_own : d0) + (part == 0 ? d0 : part == 1 ? d_own : d1)) + ((part < 2 ? d1 : part == 2 ? d_own : d2) + (part < 3 ? d2 : d_own));
        const float tot = walk_layernorm(gg, gb, -bf2f(nw.eta), xh, go, gz, gam, nw.sd, gy, dg, dz) + d_sum;
        const bf16x8 z = cvt8(dz);
        u32x4 zw = __builtin_bit_cast(u32x4, z);
#pragma unroll
        for (int e = 0; e < 4; e++) zw[e] = min(zw[e], WD_EMPTY - 1);   // (a NaN stays one)
        const uint64_t y[2] = {zw[0] | (uint64_t)zw[1] << 32, zw[2] | (uint64_t)zw[3] << 32};
        put_words(z_slot(slot, part, half), y);
        ln_store_h(s_dz2 + own_tok * LDX + f0, __builtin_bit_cast(bf16x8, zw));
        TTT_STAGE(BQH_LN);
        uint64_t x1[1][2];
        take_dz(x1, 4 + half, [&]() {
          float dxv[8];
#pragma unroll
          for (int e = 0; e < 8; e++) dxv[e] = (float)nw.old[e] - gy[e];                        // dXV accumulates -g_y
          out = cvt8(dxv);
          deta = (bf16)((float)nw.deta - tot);
          float* const yy = reinterpret_cast<float*>(smem + BWQ_GY) + (n & 1) * (16 * FD) + (8 * half + q8) * FD + f0;
          const f32x4 y0 = {gy[0], gy[1], gy[2], gy[3]}, y1 = {gy[4], gy[5], gy[6], gy[7]};
          *reinterpret_cast<f32x4*>(yy) = y0;
          *reinterpret_cast<f32x4*>(yy + 4) = y1;
          ln_token_sum_add(s_dgw, dg, lane, f0);
          ln_token_sum_add(s_dbw, gy, lane, f0);
        });
      } else {
        if (n > 0) finish_dk(n - 1, mb_before);
        TTT_STAGE(BQH_DXK);
        uint64_t y[2][2];
        take_dz(y, 2 * half, nothing);
      }
      if (gave_up && lane == 0) s_flag[0] = 1;
      TTT_STAGE(BQH_TAKE2);
      __syncthreads();   // B2
      TTT_STAGE(BQH_B2);
      __builtin_amdgcn_s_setprio(0);
      if (flag(0) != 0) {
        if (lane == 0) report_status(w_status);
        return;
      }
      const int kn = j > 0 ? k : k - 1, jn = j > 0 ? j - 1 : cgs - 1;
      if (more) {
        if (j == 0) group_tiles((done + 1) % n_sets);
        ask_out(kn, jn);
        ask_step(kn, jn);
      }
      if (u < 2) lds_rowsum_add_jit(s_gb2 + 32 * u, [&](int s) { return piece_tr<LDX>(s_dz2, u, s, lane); }, ones, c, h);
      TTT_STAGE(BQH_PUT);
      __syncthreads();   // B3
      TTT_STAGE(BQH_B3);
      if (owns && j == n_mb - 1) {   // the group's norm-gradient sums, by eighths: published with it
        const float* np = p.norm_partial + ((size_t)bh * BWD_MAX_SETS + set) * (8 * BW_NWAVE * 2 * FD) + (2 * part + half) * 2 * FD + lane;
        const int eighth = (cgs + 7) / 8;
        float a0 = np[0], a1 = np[FD];
        for (int e = 1; e * eighth < n_mb; e++) {
          a0 += np[e * (BW_NWAVE * 2 * FD)];
          a1 += np[e * (BW_NWAVE * 2 * FD) + FD];
        }
        nr0 += a0;
        nr1 += a1;
      }
      if (more) {
        put_out();   // (read up to B1)
      }
      dxk_old = nw.old;
      if (owns) {
        if ((lane & 7) == 0) g_sth(bDETA, 2 * own_tok, mb * (CS * 2), deta);
        g_st_stream<bf16x8>(bDXV, own_off, mb * TILE_BYTES, out);
        // All four CUs are past the mini-batch before: the replays may have its group's set.
        if (part == 0 && half == 0 && lane == 0 && n > 0 && j == n_mb - 1) {
          __hip_atomic_store(words + BWW_WALKED, done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(words + BWW_WALKED + 4, done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(words + 24, done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      mb_before = mb;
      TTT_STAGE(BQH_NORM);
      __syncthreads();   // BE
      TTT_STAGE(BQH_BE);
    }
  }
  if (part < 2) TTT_STAGES_END(bh, STAGE_ROLE_WALK_HALF + part);
  // grad_L_XK of the last mini-batch
  gather_dk();
  give_dk(p.NC - 1);
  if (!owns) finish_dk(p.NC - 1, mb_before);
  // The norm gradients: every "wave" of 8 tokens leaves its two pairs of sums, and the CU that is through last adds them up, the replays'
  // sum + the walk's, in the order of the other launch shapes.
  float* const sums = reinterpret_cast<float*>(p.xchg + (size_t)bh * BWQ_XCHG_WORDS + BWQ_XSUM);
  if (owns) {
    float* const q = sums + (2 * part + half) * 4 * FD + lane;
    q[0] = s_dgw[lane]; q[FD] = s_dbw[lane]; q[2 * FD] = nr0; q[3 * FD] = nr1;
  }
  if (u < 2 && part == 0 && lane < 32) p.grad_L_b2_init[(size_t)bh * FD + 32 * u + lane] = s_gb2[32 * u + lane];
  if (gave_up && lane == 0) report_status(w_status);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // (the helper waves alone from here on: each counts itself, the last of all sixteen finishes)
  int last = 0;
  if (lane == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    last = __hip_atomic_fetch_add(words + BWQW_JOIN, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 4 * BWQ_CUS - 1;
  }
  if (__any(last != 0)) {
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#pragma unroll
    for (int which = 0; which < 2; which++) {
      float s = 0.f, sr = 0.f;
#pragma unroll
      for (int x = 0; x < BW_NWAVE; x++) {
        s += sums[(x * 4 + which) * FD + lane];
        sr += sums[(x * 4 + 2 + which) * FD + lane];
      }
      (which == 0 ? p.grad_L_ttt_norm_weight : p.grad_L_ttt_norm_bias)[(size_t)bh * FD + lane] = sr + s;
    }
  }
  __syncthreads();
#undef QGRP
#undef WQ_LANE
#undef QSCHED
}

}  // namespace ttt
