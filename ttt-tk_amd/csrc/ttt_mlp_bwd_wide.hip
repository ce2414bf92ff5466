// Remat backward with the reverse walk of one (batch, head) spread over several CUs (few pairs: the walk's chain is the bound).
//
// The walk on one CU spends 28 k clocks on a mini-batch.  In bwd_wide_walk two workgroups of one XCD hold 128 hidden columns each
// (two of the four wave pairs of ttt_mlp_bwd.hip), with two kinds of waves as in ttt_mlp_fwd_wide.hip:
//   waves 0-3 (one per SIMD)  32 hidden columns each: every matrix product and the running gradients
//   waves 4-7                 sums over the hidden dimension, their exchange with the other CU, the LayerNorm lanes, the
//                             gradient wrt b2, and the next mini-batch's tiles through their registers into LDS
// The sum that crosses (the gradient wrt dl/dZ2, one fp32 tile per mini-batch and direction) is taken in two blocks of 32
// tokens: block 0's travels while block 1 is computed, block 1's while the products that do not wait for it run.
// Further workgroups replay checkpoint groups in turn (bwd_body<1>) or form grad_L_XK / grad_L_XV and the norm gradients
// (bwd_finish_dxk), whole ones for each pair or shared by the pairs of an XCD; that launch also runs with the walk on one CU
// (ttt_mlp_bwd_gang_kernel).  Every sum has the order of the one-workgroup kernel: same results to the bit.
//
// 48 pairs x 256 mini-batches 3.60 ms with the walk on one CU, 3.03 ms here; 48 x 4,096 49.8 -> 41.2 ms.
// With the stage clocks in, 21.8 k clocks per mini-batch at 48 pairs, where the two replaying workgroups bound it (42.9 k clocks
// per mini-batch each, hardly any of it waiting).  Up to 40 pairs, where this chain would be the bound (19.2 k), the walk has
// four CUs (ttt_mlp_bwd_quad.hpp).
#define TTT_BWD_ROLES_ONLY
#include "ttt_mlp_bwd.hip"
#include "ttt_mlp_exchange.hpp"

namespace ttt {

// LDS carve-up of a workgroup of the walk (bytes)
constexpr int BWW_XQ = 0;
constexpr int BWW_GZB = BWW_XQ + SB_TILE;                 // gZ2_bar
constexpr int BWW_XK = BWW_GZB + SB_TILE;                 // two buffers, alternating per mini-batch
constexpr int BWW_GZ2 = BWW_XK + 2 * SB_TILE;             // dl/dZ2, two buffers
constexpr int BWW_DZ2 = BWW_GZ2 + 2 * SB_TILE;
constexpr int BWW_T12 = BWW_DZ2 + SB_TILE;                // per compute wave: T1, T2
constexpr int BWW_T0 = BWW_T12 + 4 * SB_REGION;           // per compute wave: X2 rows
constexpr int BWW_P = BWW_T0 + 4 * SB_WTILE;              // per compute wave: its partial sum of one token block, [32 tok][F] fp32
constexpr int BWW_PTILE = 32 * LDR * 4;
constexpr int BWW_GB1 = BWW_P + 4 * BWW_PTILE;            // gradient wrt b1, 32 per compute wave
constexpr int BWW_GB2 = BWW_GB1 + 4 * BW_NS * 4;
constexpr int BWW_GAM = BWW_GB2 + FD * 4;
constexpr int BWW_DETA = BWW_GAM + FD * 4;                // [4 compute waves][64 tokens]
constexpr int BWW_ETA = BWW_DETA + 4 * CS * 4;            // fp32, two buffers
constexpr int BWW_FLAG = BWW_ETA + 2 * CS * 4;            // [0] a wait gave up, [1] gathers of block 0 done
constexpr int BWW_BYTES = BWW_FLAG + 16;
static_assert(BWW_BYTES <= SM_BWD_BYTES, "the launch asks for SM_BWD_BYTES (the replay's carve-up)");

// Second-order pass through the fused LayerNorm loss for the 8 features of this lane's token.  gg: the sum over the hidden
// dimension of what the weight step backwards gives (gradient wrt dl/dZ2 before the bias term and -eta); gb: gradient
// wrt b2; xh, go, gz: x_hat, grad_output and dl/dZ2 of the loss.  Out: gy (gradient wrt y), dg (norm-weight gradient
// terms), dz = dZ2; returns sum_F gz * gb, the bias part of d eta.
TTT_DEV float walk_layernorm(float (&gg)[8], const float (&gb)[8], float neg_eta, const float (&xh)[8], const float (&go)[8],
                             const float (&gz)[8], const float (&gam)[8], float sdf, float (&gy)[8], float (&dg)[8], float (&dz)[8]) {
#pragma clang fp contract(off)   // which product of a sum of two is fused is written out: every launch shape gives the same bits
  float gs[8];
#pragma unroll
  for (int e = 0; e < 8; e++) gs[e] = gg[e] + gb[e];
#pragma unroll
  for (int e = 0; e < 8; e++) gg[e] = gs[e] * neg_eta;             // grad wrt dl/dZ2
  const float rsd = 1.f / sdf;
  const float eta_bias = oct_sum(dot8(gz, gb));
  float s0 = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) s0 = __builtin_fmaf(gs[e], neg_eta, s0);
  s0 = oct_sum(s0);
  const float a = oct_sum(dot8(gg, xh));
  float bb = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) bb = __builtin_fmaf(go[e] * gam[e], xh[e], bb);
  bb = oct_sum(bb);
  const float inv = rsd * (1.f / FD);
  float sg = 0.f, sx = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const float ggx = __builtin_fmaf(-__builtin_fmaf(xh[e], a, s0), 1.f / FD, gg[e]) * rsd;
    gy[e] = gam[e] * ggx;
    dg[e] = __builtin_fmaf(go[e], ggx, gy[e] * xh[e]);
    dz[e] = __builtin_fmaf(gy[e], gam[e], -(__builtin_fmaf(go[e] * gam[e], a, gg[e] * bb) * inv));
    sg = __builtin_fmaf(-__builtin_fmaf(dz[e], xh[e], gg[e] * gz[e]), rsd, sg);
    sx += dz[e];
  }
  sg = oct_sum(sg);
  sx = oct_sum(sx);
#pragma unroll
  for (int e = 0; e < 8; e++) dz[e] = __builtin_fmaf(dz[e], rsd, __builtin_fmaf(sg, xh[e], -(sx * rsd)) * (1.f / FD));
  return eta_bias;
}

TTT_DEV void bwd_wide_walk(const BwdParams& p, unsigned char* smem, const int bh, const int half) {
  typedef __attribute__((address_space(3))) int* lint_t;
  const lint_t s_flag = (lint_t)reinterpret_cast<int*>(smem + BWW_FLAG);
  auto flag = [&](int i) { return __hip_atomic_load(s_flag + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, c = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int u = w & 3;                                   // number among its kind
  const int v = 2 * half + (u & 1) + 4 * (u >> 1);       // compute wave u: hidden block, = wave of the one-workgroup kernel
  const int head = bh % p.NH, hid0 = BW_NS * v;
  const int cgs = p.cgs, n_sets = p.n_sets;
  bf16* const s_xq = reinterpret_cast<bf16*>(smem + BWW_XQ);
  bf16* const s_gzb = reinterpret_cast<bf16*>(smem + BWW_GZB);
  bf16* const s_dz2 = reinterpret_cast<bf16*>(smem + BWW_DZ2);
  float* const s_gb2 = reinterpret_cast<float*>(smem + BWW_GB2);
  float* const s_gam = reinterpret_cast<float*>(smem + BWW_GAM);
  float* const s_deta = reinterpret_cast<float*>(smem + BWW_DETA);
  int* const words = p.sync + (size_t)bh * BWD_SYNC_STRIDE;
  bf16x8 ones;
#pragma unroll
  for (int j = 0; j < 8; j++) ones[j] = (bf16)1.0f;
  if (tid == 0) say_xcd(words + BWW_XCD + half);
  if (tid < 2) s_flag[tid] = 0;
  if (tid < FD) {
    s_gam[tid] = p.ttt_norm_weight[head * FD + tid];
    s_gb2[tid] = p.grad_L_b2_last[(size_t)bh * FD + tid];
  }
  // this (batch, head)'s part of each class of tensor (elements), and the per-group tensors of set `set`
  const size_t ox = uni64((size_t)bh * p.NC * (CS * FD)), oe = uni64((size_t)bh * p.NC * CS);
  const size_t of = uni64((size_t)bh * cgs * (CS * FD)), oh = uni64((size_t)bh * cgs * (CS * HID));
  const size_t ot = uni64((size_t)bh * cgs * CS), ock = uni64((size_t)bh * p.K * (FD * HID));
  // The pointers are read from the kernel-argument segment where they are used (see bwd_body).
  typedef const __attribute__((address_space(4))) BwdParams* KernArgs;
  KernArgs ka = (KernArgs)__builtin_amdgcn_kernarg_segment_ptr();
#define WGRP(name) (set ? ka->alt_##name[set - 1] : ka->name)
  int lane_v = lane;
#define WW_LANE                                                        \
  asm volatile("" : "+v"(lane_v));                                     \
  const int lane = lane_v, h = lane >> 5, c = lane & 31;               \
  const unsigned t16 = 16 * ((v << 6) | lane);                         \
  (void)h; (void)c; (void)t16

  if (w < 4) {
    // ================================================================ compute waves
    bf16* const T1 = reinterpret_cast<bf16*>(smem + BWW_T12 + u * SB_REGION);
    bf16* const T2 = T1 + 64 * LDH;
    bf16* const T0 = reinterpret_cast<bf16*>(smem + BWW_T0 + u * SB_WTILE);
    float* const s_Pw = reinterpret_cast<float*>(smem + BWW_P + u * BWW_PTILE);
    float* const s_gb1w = reinterpret_cast<float*>(smem + BWW_GB1) + u * BW_NS;
    AccT<2, 1> gW1s;
    AccT<1, 2> gW2s;
    acc_load_rows(gW1s, gbuf(p.grad_L_W1_last + (size_t)bh * FD * HID), 0, HID, 0, hid0, c, h);
    acc_load_rows(gW2s, gbuf(p.grad_L_W2_last + (size_t)bh * HID * FD), 0, FD, hid0, 0, c, h);
    if (lane < BW_NS) s_gb1w[lane] = p.grad_L_b1_last[(size_t)bh * HID + hid0 + lane];
    __syncthreads();   // flags
    __syncthreads();   // placement known, the first group is there, its last mini-batch's tiles too
    if (flag(0) != 0) return;
    bf16x8 x2b[4], g1b[4];   // what the output branch adds (lane = hid, contraction = tok), asked for a mini-batch ahead
    bf16x8 w2bf[4];          // W2 before the step, and gelu, gelu', gelu'' of Z1 by token block
    bf16x8 gq[2][2], aq[2][2], bq[2][2];
    gptr_t gX2B, gGZ1B, gI2, gZ;
    auto group_images = [&](int set) {
      gX2B = gbuf(WGRP(X2_bar_group) + oh);
      gGZ1B = gbuf(WGRP(Z1_bar_group) + oh);
      gI2 = gbuf(WGRP(grad_l_wrt_Z1_group) + oh);
      gZ = gbuf(WGRP(Z1_group) + oh);
    };
    const gptr_t gCk = gbuf(ka->W2_ck + ock);
    auto ask_gelu = [&](int i, int j) {
      WW_LANE;
#pragma unroll
      for (int t = 0; t < 2; t++) {
        gq[i][t] = chunk_load(gZ, j * IMG_BYTES, 2 * i + t, t16);
      }
    };
    // Operands are asked for one to two stages ahead (one CU cannot keep enough requests in flight to hide the way to HBM: 80 KiB
    // asked for in a row take 9 k clocks to issue); what the grad_L_XK workgroup reads next is left in the L2.
    auto ask_bar = [&](int j) {
      WW_LANE;
#pragma unroll
      for (int s = 0; s < 4; s++) {
        x2b[s] = image_load(gX2B, j * IMG_BYTES, s, t16);
        g1b[s] = chunk_load(gGZ1B, j * IMG_BYTES, s, t16);
      }
    };
    auto ask_step = [&](int k, int j) {
      WW_LANE;
      if (j > 0) {
#pragma unroll
        for (int s = 0; s < 4; s++) w2bf[s] = chunk_load(gI2, (j - 1) * IMG_BYTES, s, t16);
      } else {
#pragma unroll
        for (int s = 0; s < 4; s++) w2bf[s] = piece_from_f32(gCk, static_cast<unsigned>(k) * (FD * HID * 4u), FD, hid0, 0, s, c, h);
      }
      ask_gelu(0, j);
    };
    // One wave per SIMD: the latency of an LDS read is hidden only by what is put between it and its use, so operands are read a
    // product or more ahead, and the fences keep the scheduler from sinking the reads again.
#define SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)
    // row sums of a 32-row operand of four pieces on the matrix cores (as lds_rowsum_add_jit), and their addition to gb1
    auto rowsum4 = [&](bf16x8 a, bf16x8 b, bf16x8 c4, bf16x8 d) {
      f32x16 t;
#pragma unroll
      for (int i = 0; i < 16; i++) t[i] = 0.f;
      t = MFMA(a, ones, t);
      t = MFMA(b, ones, t);
      t = MFMA(c4, ones, t);
      return MFMA(d, ones, t);
    };
    auto add_gb1 = [&](const f32x16& t) {
      WW_LANE;
      f32x4 old[4];
#pragma unroll
      for (int g = 0; g < 4; g++) old[g] = *reinterpret_cast<const f32x4*>(s_gb1w + 8 * g + 4 * h);
      if (c == 0) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
#pragma unroll
          for (int e = 0; e < 4; e++) old[g][e] += t[4 * g + e];
          *reinterpret_cast<f32x4*>(s_gb1w + 8 * g + 4 * h) = old[g];
        }
      }
      WAVE_SYNC();
    };
    int n = 0;   // mini-batches walked
    TTT_STAGES_BEGIN();
    group_images(0);
    ask_bar(min(cgs, p.NC - (p.K - 1) * cgs) - 1);
    ask_step(p.K - 1, min(cgs, p.NC - (p.K - 1) * cgs) - 1);
    for (int k = p.K - 1; k >= 0; k--) {
      const int n_mb = min(cgs, p.NC - k * cgs);
      const int done = p.K - 1 - k;
      const gptr_t gDZ = gbuf(ka->fin_dz + uni64(((size_t)bh * 2 + (done & 1)) * cgs) * (CS * HID));
      for (int j = n_mb - 1; j >= 0; j--, n++) {
        const unsigned ho = j * IMG_BYTES;
        const bf16* const s_xk = reinterpret_cast<const bf16*>(smem + BWW_XK + (n & 1) * SB_TILE);
        const bf16* const s_gz2 = reinterpret_cast<const bf16*>(smem + BWW_GZ2 + (n & 1) * SB_TILE);
        const float* const s_eta = reinterpret_cast<const float*>(smem + BWW_ETA) + (n & 1) * CS;
        // ---- what the output branch adds to the running gradients
        {
          WW_LANE;
          bf16x8 zb[4][2], xq[4][2];
#pragma unroll
          for (int s = 0; s < 4; s++)
#pragma unroll
            for (int fb = 0; fb < 2; fb++) zb[s][fb] = piece_tr<LDX>(s_gzb, fb, s, lane);
          SCHED_FENCE();
          f32x16 t = rowsum4(g1b[0], g1b[1], g1b[2], g1b[3]);
#pragma unroll
          for (int s = 0; s < 4; s++) {
#pragma unroll
            for (int fb = 0; fb < 2; fb++) gW2s.b[0][fb] = MFMA(x2b[s], zb[s][fb], gW2s.b[0][fb]);
#pragma unroll
            for (int fb = 0; fb < 2; fb++) xq[s][fb] = xpiece_tr(s_xq, fb, s, lane);
            SCHED_FENCE();
          }
#pragma unroll
          for (int s = 0; s < 4; s++)
#pragma unroll
            for (int fb = 0; fb < 2; fb++) gW1s.b[fb][0] = MFMA(xq[s][fb], g1b[s], gW1s.b[fb][0]);
          add_gb1(t);
        }
        ask_gelu(1, j);
        TTT_STAGE(BWC_BAR_TERMS);
        // ---- the weight step, backwards (state BEFORE this mini-batch), one token block at a time
        bf16x8 t2p[2][2], uhp[2][2], d1p[2][2];   // d1p: gelu'(Z1)
        float eta_i[2];
        {
          WW_LANE;
#pragma unroll
          for (int s = 0; s < 4; s++) store_piece_rows<LDF>(T1, 0, s, c, h, w2bf[s]);   // W2 before the step, rows [hid][F]
          store_state_rows<LDF>(T2, gW1s, c, h);                                         // gW1 rows [hid][F]
          WAVE_SYNC();
        }
        auto step_back = [&](int i) {
          WW_LANE;
          eta_i[i] = s_eta[32 * i + c];
          AccT<1, 1> R, S;   // R = gZ2 W2^T, S = XK gW1 + gb1   (rows hid, lane = tok)
          acc_zero(R);
          acc_init_rows_lds(S, s_gb1w, h);
          bf16x8 w2r[4], w1r[4], gz[4], xk[4];
#pragma unroll
          for (int s = 0; s < 4; s++) {
            w2r[s] = piece_rows<LDF>(T1, 0, s, c, h);
            gz[s] = piece_rows<LDX>(s_gz2, i, s, c, h);
            w1r[s] = piece_rows<LDF>(T2, 0, s, c, h);
            xk[s] = xpiece_rows(s_xk, i, s, c, h);
          }
          SCHED_FENCE();
#pragma unroll
          for (int s = 0; s < 4; s++) {
            R.b[0][0] = MFMA(w2r[s], gz[s], R.b[0][0]);
            S.b[0][0] = MFMA(w1r[s], xk[s], S.b[0][0]);
          }
          AccT<2, 1> pz;
          acc_zero(pz);
          float de = 0.f;
          bf16x8 x2c[2], uc[2];
#pragma unroll
          for (int t = 0; t < 2; t++) {
            const bf16x8 zc = gq[i][t];
#pragma unroll
            for (int jj = 0; jj < 8; jj++) {
              float g, a, b;
              gelu_fdd((float)zc[jj], g, a, b);
              x2c[t][jj] = (bf16)g;
              aq[i][t][jj] = (bf16)a;
              bq[i][t][jj] = (bf16)b;
            }
            asm volatile("" : "+v"(x2c[t]), "+v"(aq[i][t]), "+v"(bq[i][t]));   // finished here (see the replay's gelu')
#pragma unroll
            for (int jj = 0; jj < 8; jj++) {
              const float a = (float)aq[i][t][jj], b = (float)bq[i][t][jj];
              const float r0 = R.b[0][0][8 * t + jj], sv = S.b[0][0][8 * t + jj];
              const float gz1 = r0 * a;                                   // dl/dZ1
              de = __builtin_fmaf(gz1, sv, de);
              uc[t][jj] = (bf16)(sv * a);
              uhp[i][t][jj] = (bf16)(-eta_i[i] * sv * a);
              t2p[i][t][jj] = (bf16)(-eta_i[i] * r0 * sv * b);
            }
            d1p[i][t] = aq[i][t];
            store_piece_rows<LDH>(T0, i, t, c, h, x2c[t]);                // X2 rows [tok][hid]
          }
          bf16x8 gzv[4], w2t[2][2];
#pragma unroll
          for (int s = 0; s < 2; s++) gzv[s] = piece_rows<LDX>(s_gz2, i, s, c, h);
          SCHED_FENCE();
          // pz = gW2^T X2^T ; d eta partial ; + W2^T u^T
#pragma unroll
          for (int t = 0; t < 2; t++)
#pragma unroll
            for (int rb = 0; rb < 2; rb++) pz.b[rb][0] = MFMA(piece_state(gW2s, rb, t), x2c[t], pz.b[rb][0]);
#pragma unroll
          for (int s = 0; s < 4; s++) {
#pragma unroll
            for (int jj = 0; jj < 8; jj++) de = __builtin_fmaf((float)gzv[s][jj],  pz.b[s >> 1][0][8 * (s & 1) + jj], de);
            if (s == 1) {
              SCHED_FENCE();
              gzv[2] = piece_rows<LDX>(s_gz2, i, 2, c, h);
              gzv[3] = piece_rows<LDX>(s_gz2, i, 3, c, h);
#pragma unroll
              for (int q = 0; q < 4; q++) w2t[q >> 1][q & 1] = piece_tr<LDF>(T1, q & 1, q >> 1, lane);
              SCHED_FENCE();
            }
          }
#pragma unroll
          for (int t = 0; t < 2; t++)
#pragma unroll
            for (int rb = 0; rb < 2; rb++) pz.b[rb][0] = MFMA(w2t[t][rb], uc[t], pz.b[rb][0]);
          const float a = half_sum_valu(de);
          if (i == 1) {   // block 0's sums have been gathered (long since)
            while (flag(1) < 4 * (n + 1)) __builtin_amdgcn_s_sleep(1);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
          }
          if (h == 0) s_deta[u * CS + 32 * i + c] = a;
#pragma unroll
          for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
              const f32x16& x = pz.b[rb][0];
              f32x4 q = {x[4 * g], x[4 * g + 1], x[4 * g + 2], x[4 * g + 3]};
              *reinterpret_cast<f32x4*>(s_Pw + c * LDR + 32 * rb + 8 * g + 4 * h) = q;
            }
        };
        step_back(0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // dZ1 of the last mini-batch is out (and everything asked for is here)
        __builtin_amdgcn_sched_barrier(0);
        TTT_STAGE(BWC_STEP0);
        __syncthreads();                                    // B1: block 0's sums
        TTT_STAGE(BWC_B1);
        __builtin_amdgcn_sched_barrier(0);
        step_back(1);
        // ---- inner MLP backwards and the updates of the running gradients, token block i
        f32x16 dx2[2], gb1_t;                               // gradient wrt X2; row sums of dZ1
        auto mlp_back = [&](int i) {
          WW_LANE;
          bf16x8 w2r[4], dr[4], dt[2][2], x2[2], xkt[2][2], dz1[2];
#pragma unroll
          for (int s = 0; s < 4; s++) {
            w2r[s] = piece_rows<LDF>(T1, 0, s, c, h);
            dr[s] = piece_rows<LDX>(s_dz2, i, s, c, h);
          }
          SCHED_FENCE();
          f32x16 q = dx2[i];
#pragma unroll
          for (int s = 0; s < 4; s++) q = MFMA(w2r[s], dr[s], q);                              // + dZ2 W2^T
          SCHED_FENCE();
#pragma unroll
          for (int t = 0; t < 2; t++) {
            x2[t] = piece_tr<LDH>(T0, 0, 2 * i + t, lane);
#pragma unroll
            for (int fb = 0; fb < 2; fb++) dt[t][fb] = piece_tr<LDX>(s_dz2, fb, 2 * i + t, lane);
          }
          SCHED_FENCE();
#pragma unroll
          for (int t = 0; t < 2; t++)
#pragma unroll
            for (int fb = 0; fb < 2; fb++) gW2s.b[0][fb] = MFMA(x2[t], dt[t][fb], gW2s.b[0][fb]);   // + X2^T dZ2
#pragma unroll
          for (int t = 0; t < 2; t++) {
            bf16x8 dz;
#pragma unroll
            for (int jj = 0; jj < 8; jj++) dz[jj] = (bf16)__builtin_fmaf(q[8 * t + jj], (float)d1p[i][t][jj], (float)t2p[i][t][jj]);   // dZ1
            image_store(gDZ, ho, 2 * i + t, t16, dz);                                    // for the grad_L_XK workgroup
            store_piece_rows<LDH>(T2, i, t, c, h, dz);                                         // rows [tok][hid]
          }
#pragma unroll
          for (int t = 0; t < 2; t++)
#pragma unroll
            for (int fb = 0; fb < 2; fb++) xkt[t][fb] = xpiece_tr(s_xk, fb, 2 * i + t, lane);
          WAVE_SYNC();
#pragma unroll
          for (int t = 0; t < 2; t++) dz1[t] = piece_tr<LDH>(T2, 0, 2 * i + t, lane);
          if (i == 0) {
#pragma unroll
            for (int e = 0; e < 16; e++) gb1_t[e] = 0.f;
          }
#pragma unroll
          for (int t = 0; t < 2; t++) {
#pragma unroll
            for (int fb = 0; fb < 2; fb++) gW1s.b[fb][0] = MFMA(xkt[t][fb], dz1[t], gW1s.b[fb][0]);   // + XK^T dZ1
            gb1_t = MFMA(dz1[t], ones, gb1_t);
          }
        };
        __builtin_amdgcn_sched_barrier(0);
        TTT_STAGE(BWC_STEP1);
        __syncthreads();                                    // B2: block 1's sums; dZ2 of block 0
        TTT_STAGE(BWC_B2);
        __builtin_amdgcn_sched_barrier(0);
        if (j == 0) group_images((done + 1) % n_sets);
        const int kn = j > 0 || k == 0 ? k : k - 1, jn = j > 0 ? j - 1 : cgs - 1;   // (behind the last mini-batch: dropped)
        // ---- while block 1's sums cross: the products of the inner MLP backwards that do not need them
        {
          WW_LANE;
          store_state_rows<LDH>(T2, gW2s, c, h);            // gW2 rows [F][hid] (transposed read gives lane = hid)
          bf16x8 gz[2][4], gw[4];
#pragma unroll
          for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < 2; i++) gz[i][s] = piece_rows<LDX>(s_gz2, i, s, c, h);
          WAVE_SYNC();
#pragma unroll
          for (int s = 0; s < 4; s++) gw[s] = piece_tr<LDH>(T2, 0, s, lane);
          SCHED_FENCE();
          f32x16 q[2];
#pragma unroll
          for (int i = 0; i < 2; i++)
#pragma unroll
            for (int e = 0; e < 16; e++) q[i][e] = 0.f;
#pragma unroll
          for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < 2; i++) q[i] = MFMA(gw[s], gz[i][s], q[i]);                  // P2 = gZ2 gW2^T
          WAVE_SYNC();
#pragma unroll
          for (int i = 0; i < 2; i++)
#pragma unroll
            for (int t = 0; t < 2; t++) store_piece_rows<LDH>(T2, i, t, c, h, uhp[i][t]);   // -eta u rows [tok][hid]
          ask_bar(jn);   // the next mini-batch's output-branch images (the helpers made sure of its group before B1)
          bf16x8 ut[4], gt[4][2];
#pragma unroll
          for (int s = 0; s < 4; s++)
#pragma unroll
            for (int fb = 0; fb < 2; fb++) gt[s][fb] = piece_tr<LDX>(s_gz2, fb, s, lane);
          WAVE_SYNC();
#pragma unroll
          for (int s = 0; s < 4; s++) ut[s] = piece_tr<LDH>(T2, 0, s, lane);
          SCHED_FENCE();
#pragma unroll
          for (int s = 0; s < 4; s++)
#pragma unroll
            for (int fb = 0; fb < 2; fb++) gW2s.b[0][fb] = MFMA(ut[s], gt[s][fb], gW2s.b[0][fb]);   // (-eta u)^T gZ2
#pragma unroll
          for (int i = 0; i < 2; i++)
#pragma unroll
            for (int e = 0; e < 16; e++) dx2[i][e] = q[i][e] * -eta_i[i];
          WAVE_SYNC();
        }
        TTT_STAGE(BWC_PRODUCTS);
        mlp_back(0);
        __builtin_amdgcn_sched_barrier(0);
        TTT_STAGE(BWC_MLP0);
        __syncthreads();                                    // B3: dZ2 of block 1; the next mini-batch's tiles
        TTT_STAGE(BWC_B3);
        __builtin_amdgcn_sched_barrier(0);
        const int gave_up = flag(0);
        mlp_back(1);
        ask_step(kn, jn);
        add_gb1(gb1_t);
        TTT_STAGE(BWC_MLP1);
        if (gave_up != 0) return;
      }
    }
    TTT_STAGES_END(bh, STAGE_ROLE_WALK_HALF + half);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();   // the last dZ1 is out
    acc_store_rows(gW1s, gbuf(p.grad_L_W1_init + (size_t)bh * FD * HID), 0, HID, 0, hid0, c, h);
    acc_store_rows(gW2s, gbuf(p.grad_L_W2_init + (size_t)bh * HID * FD), 0, FD, hid0, 0, c, h);
    if (lane < BW_NS) p.grad_L_b1_init[(size_t)bh * HID + hid0 + lane] = s_gb1w[lane];
    return;
  }

  // ================================================================== helper waves
  const int q8 = lane >> 3, f0 = 8 * (lane & 7), t_in = 8 * u + q8;   // LayerNorm lanes: token t_in of a block, features f0 ..
  const unsigned voff = (t_in * FD + f0) * 2;
  constexpr unsigned HALF_TILE = TILE_BYTES / 2;                        // 32 tokens
  int* const w_status = p.status;
  // A wave that gives up keeps that to itself until the stage whose closing barrier precedes the reads of s_flag[0] (B3, or the
  // barrier that opens the walk): all eight waves then read the same value and leave together, or none does.  Raised at the
  // top of a mini-batch it could be seen by one wave and missed by another, which then waited for the first without a limit.
  bool gave_up = false;
  __syncthreads();   // flags
  auto wait_for = [&](int* word, int target) {
    if (!__all(lane != 0 || wait_word(word, target, w_status, p.wait_limit))) gave_up = true;
  };
  // group number `done` (from the end) has been replayed
  auto wait_group = [&](int done) { wait_for(words + done % n_sets, parts_until(p, done)); };
  // What one mini-batch needs from HBM besides the operand images: a chunk of 16 bytes per lane and token block of each
  // tile - the lanes that hold a chunk are the LayerNorm lanes of that token and those features.
  struct Ahead {
    bf16x8 xq[2], xk[2], gz[2], gzb[2], xh[2], go[2];
    float sd[2];
    bf16 eta[2], deta[2];
  } nx;
  auto ask = [&](int k, int j) {
    const int set = (p.K - 1 - k) % n_sets, mb = k * cgs + j;
    asm volatile("" : "+s"(ka));
    const gptr_t gq = gbuf(ka->XQ + ox), gk = gbuf(ka->XK + ox), gz = gbuf(WGRP(grad_l_wrt_Z2_group) + of);
    const gptr_t gb = gbuf(WGRP(grad_x_hat_fused_group) + of), gx = gbuf(WGRP(x_hat_fused_group) + of);
    const gptr_t gg = gbuf(WGRP(grad_output_fused_group) + of), gs = gbuf(WGRP(std_fused_group) + ot);
    const gptr_t ge = gbuf(ka->last_eta + oe), gd = gbuf(ka->grad_L_last_eta + oe), zero = gbuf(zero_tile);
    const bool ow = ka->overwrite != 0;
#pragma unroll
    for (int b = 0; b < 2; b++) {
      const unsigned xo = mb * TILE_BYTES + b * HALF_TILE, so = j * TILE_BYTES + b * HALF_TILE;
      nx.gz[b] = g_ld8h(gz, voff, so);
      nx.gzb[b] = g_ld_stream<bf16x8>(gb, voff, so);
      nx.xq[b] = g_ld8h(gq, voff, xo);
      nx.xk[b] = g_ld8h(gk, voff, xo);
      nx.xh[b] = g_ld_stream<bf16x8>(gx, voff, so);
      nx.go[b] = g_ld_stream<bf16x8>(gg, voff, so);
      nx.sd[b] = g_ldf(gs, 4 * t_in, (j * CS + 32 * b) * 4);
      nx.eta[b] = g_ldh(ge, 2 * t_in, (mb * CS + 32 * b) * 2);
      nx.deta[b] = g_ldh(ow ? zero : gd, 2 * t_in, ow ? 0u : (mb * CS + 32 * b) * 2);
    }
  };
  auto put = [&](int n) {   // tiles of the mini-batch that is walked as number n
    bf16* const s_xk = reinterpret_cast<bf16*>(smem + BWW_XK + (n & 1) * SB_TILE);
    bf16* const s_gz2 = reinterpret_cast<bf16*>(smem + BWW_GZ2 + (n & 1) * SB_TILE);
    float* const s_eta = reinterpret_cast<float*>(smem + BWW_ETA) + (n & 1) * CS;
#pragma unroll
    for (int b = 0; b < 2; b++) {
      const int row = 32 * b + t_in;
      ln_store_h(s_xq + xrow(row) + f0, nx.xq[b]);
      ln_store_h(s_xk + xrow(row) + f0, nx.xk[b]);
      ln_store_h(s_gz2 + row * LDX + f0, nx.gz[b]);
      ln_store_h(s_gzb + row * LDX + f0, nx.gzb[b]);
      if ((lane & 7) == 0) s_eta[row] = bf2f(nx.eta[b]);
    }
  };
  const bool near = [&]() {
    bool alive = true;
    bool one = on_one_xcd(words + BWW_XCD, 2, lane, w_status, p.wait_limit, alive);
    one = workers_here(words + BWW_WORKERS, p.n_finish + p.n_replay, w_status, p.wait_limit, alive) && one;
    if (!alive) gave_up = true;
    return one;
  }();
  wait_group(0);   // (every helper wave itself)
  {
    const int j0 = min(cgs, p.NC - (p.K - 1) * cgs) - 1;
    if (!gave_up) {
      ask(p.K - 1, j0);
      put(0);
    }
  }
  if (gave_up && lane == 0) s_flag[0] = 1;
  __syncthreads();
  if (flag(0) != 0) {
    if (lane == 0) report_status(w_status);
    return;
  }
  const gword64_t xch = (gword64_t)(p.xchg + (size_t)bh * BWW_XCHG_WORDS);
  const float* const s_row = reinterpret_cast<const float*>(smem + BWW_P) + t_in * LDR + f0;
  float gam[8];
  ln_load_f32(gam, s_gam + f0);
  const gptr_t bDETA = gbuf(p.grad_L_last_eta + oe);
  __builtin_amdgcn_s_setprio(2);

  int n = 0;
  TTT_STAGES_BEGIN();
  for (int k = p.K - 1; k >= 0; k--) {
    const int n_mb = min(cgs, p.NC - k * cgs);
    const int done = p.K - 1 - k;
    const size_t ofin = uni64(((size_t)bh * 2 + (done & 1)) * cgs);
    const gptr_t bFGY = gbuf(p.fin_gy + ofin * (2 * CS * FD));
    for (int j = n_mb - 1; j >= 0; j--, n++) {
      const int mb = k * cgs + j;
      const bf16* const s_gz2 = reinterpret_cast<const bf16*>(smem + BWW_GZ2 + (n & 1) * SB_TILE);
      const Ahead cur = nx;
      // ---- ahead of time, while the compute waves are busy: the next mini-batch
      const bool more = n + 1 < p.NC;
      if (j == 0 && k > 0) wait_group(done + 1);
      const int kn = j > 0 ? k : k - 1, jn = j > 0 ? j - 1 : cgs - 1;
      // gradient wrt b2: what the output branch adds
      if (u < 2) lds_rowsum_add_jit(s_gb2 + 32 * u, [&](int s) { return piece_tr<LDX>(s_gzb, u, s, lane); }, ones, c, h);
      // (everybody is still here, so the flag reads 0; read at this place it holds these loads back until the sums above are
      // through, 0.729 instead of 0.732 ms for 24 pairs x 64 mini-batches)
      if (more && flag(0) == 0) ask(kn, jn);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // g_y of the last mini-batch and the marks put back are in place
      TTT_STAGE(BWH_ASK);
      __syncthreads();   // B1
      TTT_STAGE(BWH_B1);
      if (u == 0 && lane == 0 && n > 0) {
        // all waves' stores of the last mini-batch were acknowledged before the barrier, all its reads are done
        if (!near) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __hip_atomic_store(words + BWW_GIVEN + 4 * half, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (j == n_mb - 1) __hip_atomic_store(words + BWW_WALKED + 4 * half, done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      // the order of the one-workgroup kernel, ((P0 + P1) + P2) + P3 over the wave pairs: half 0 sends P0 + P1, half 1 P2 and P3
      float m0[8], m1[8], d_mine, gy[8], dg[8], tot;
      auto gather_send = [&](int blk) {   // this CU's sums over its 128 hidden columns; sent to the other CU
#pragma unroll
        for (int q = 0; q < 2; q++) {
          f32x4 a[4];
#pragma unroll
          for (int i = 0; i < 4; i++) a[i] = *reinterpret_cast<const f32x4*>(s_row + i * (BWW_PTILE / 4) + 4 * q);
          const f32x4 pa = a[0] + a[2], pb = a[1] + a[3];
#pragma unroll
          for (int e = 0; e < 4; e++) { m0[4 * q + e] = pa[e]; m1[4 * q + e] = pb[e]; }
        }
        const float* const d = s_deta + 32 * blk + t_in;
        d_mine = (d[0] + d[2 * CS]) + (d[CS] + d[3 * CS]);
        const gword64_t dst = xch + ((((n & 1) * 2 + half) * 2 + blk) * 4 + u) * (64 * BWW_WORDS) + lane;
        if (half == 0) {
#pragma unroll
          for (int e = 0; e < 8; e++) m0[e] += m1[e];
        } else {   // (d eta is half 0's to write)
          wd_put(dst + 256, wd_pack(d_mine, 0.f), near);
#pragma unroll
          for (int i = 0; i < 4; i++) wd_put(dst + 64 * (5 + i), wd_pack(m1[2 * i], m1[2 * i + 1]), near);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) wd_put(dst + 64 * i, wd_pack(m0[2 * i], m0[2 * i + 1]), near);
      };
      auto finish_block = [&](int blk) {
        const int tok = 32 * blk + t_in;
        const gword64_t src = xch + ((((n & 1) * 2 + 1 - half) * 2 + blk) * 4 + u) * (64 * BWW_WORDS) + lane;
        float gg[8], gb[8], xh[8], go[8], gz[8], dz[8], d_sum = 0.f;
        if (half == 0) {
          uint64_t wv[9];
          if (!wd_take(src, wv, w_status, p.wait_limit)) gave_up = true;
          TTT_STAGE(blk == 0 ? BWH_TAKE0 : BWH_TAKE1);
#pragma unroll
          for (int i = 0; i < 9; i++) wd_put(src + 64 * i, ~0ull, near);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            gg[2 * i] = (m0[2 * i] + wd_lo(wv[i])) + wd_lo(wv[5 + i]);
            gg[2 * i + 1] = (m0[2 * i + 1] + wd_hi(wv[i])) + wd_hi(wv[5 + i]);
          }
          d_sum = d_mine + wd_lo(wv[4]);
        } else {
          uint64_t wv[4];
          if (!wd_take(src, wv, w_status, p.wait_limit)) gave_up = true;
          TTT_STAGE(blk == 0 ? BWH_TAKE0 : BWH_TAKE1);
#pragma unroll
          for (int i = 0; i < 4; i++) wd_put(src + 64 * i, ~0ull, near);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            gg[2 * i] = (wd_lo(wv[i]) + m0[2 * i]) + m1[2 * i];
            gg[2 * i + 1] = (wd_hi(wv[i]) + m0[2 * i + 1]) + m1[2 * i + 1];
          }
        }
        ln_load_f32(gb, s_gb2 + f0);
        ln_cvt8(xh, cur.xh[blk]);
        ln_cvt8(go, cur.go[blk]);
        ln_cvt8(gz, cur.gz[blk]);
        tot = walk_layernorm(gg, gb, -bf2f(cur.eta[blk]), xh, go, gz, gam, cur.sd[blk], gy, dg, dz) + d_sum;
        ln_store(s_dz2 + tok * LDX + f0, dz);
      };
      // what the block gives to the caller and to the grad_L_XK workgroup, once the other waves have what they wait for
      auto store_block = [&](int blk) {
        if (half == 0) {   // both halves hold these; one writes them
          if ((lane & 7) == 0) g_sth(bDETA, 2 * t_in, (mb * CS + 32 * blk) * 2, (bf16)((float)cur.deta[blk] - tot));
          const unsigned o = 2 * j * 4 * HALF_TILE + 2 * blk * HALF_TILE;   // g_y and the norm-weight terms: two fp32 tiles per mini-batch
          const f32x4 y0 = {gy[0], gy[1], gy[2], gy[3]}, y1 = {gy[4], gy[5], gy[6], gy[7]};
          const f32x4 d0 = {dg[0], dg[1], dg[2], dg[3]}, d1 = {dg[4], dg[5], dg[6], dg[7]};
          g_st_stream<f32x4>(bFGY, 2 * voff, o, y0);
          g_st_stream<f32x4>(bFGY, 2 * voff + 16, o, y1);
          g_st_stream<f32x4>(bFGY, 2 * voff, o + 2 * TILE_BYTES, d0);
          g_st_stream<f32x4>(bFGY, 2 * voff + 16, o + 2 * TILE_BYTES, d1);
        }
      };
      gather_send(0);
      // (a release of LDS only: one of everything would also wait for the words just sent)
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      if (lane == 0) __hip_atomic_fetch_add(s_flag + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      // the group's hand-over set to the grad_L_XK workgroup is free (written from here on)
      if (j == n_mb - 1 && done >= 2) wait_for(words + 24, done - 1);
      TTT_STAGE(BWH_SEND0);
      finish_block(0);
      TTT_STAGE(BWH_LN0);
      __syncthreads();   // B2
      TTT_STAGE(BWH_B2);
      gather_send(1);
      store_block(0);
      if (more) put(n + 1);   // XQ and gZ2_bar are read before B1 only, XK and gZ2 alternate
      TTT_STAGE(BWH_SEND1);
      finish_block(1);
      if (gave_up && lane == 0) s_flag[0] = 1;
      TTT_STAGE(BWH_LN1);
      __syncthreads();   // B3
      TTT_STAGE(BWH_B3);
      if (flag(0) != 0) {
        if (lane == 0) report_status(w_status);
        return;
      }
      store_block(1);
      if (u < 2) lds_rowsum_add_jit(s_gb2 + 32 * u, [&](int s) { return piece_tr<LDX>(s_dz2, u, s, lane); }, ones, c, h);
      TTT_STAGE(BWH_STORE1);
    }
  }
  TTT_STAGES_END(bh, STAGE_ROLE_WALK_HALF + half);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (u == 0 && lane == 0) {
    if (!near) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __hip_atomic_store(words + BWW_GIVEN + 4 * half, p.NC, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(words + BWW_WALKED + 4 * half, p.K, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (u < 2 && half == 0 && lane < 32) p.grad_L_b2_init[(size_t)bh * FD + 32 * u + lane] = s_gb2[32 * u + lane];
#undef WGRP
#undef WW_LANE
}

}  // namespace ttt
#include "ttt_mlp_bwd_quad.hpp"
namespace ttt {

// The workgroups of a gang: gang g has pairs g, g + 8, .. and, as workgroups are dealt to the 8 XCDs in turn, one XCD.  WALKERS of
// them walk each pair, the others work for all of its pairs: n_replay take the replays in turn, ordered by group, then by pair (all
// walks go at one pace) and then by part of the group, n_finish the finishing of the groups (grad_L_XK and the norm gradients) in the same
// order.  With a finishing workgroup for each pair it stays with that
// pair; with none (QUAD) the walkers finish what they walk; with fewer, the last group of each pair is finished by a replaying workgroup, all of them together.
// Nobody waits for a later job than his own: a replay waits for the set of n_sets groups ago to be walked and finished, the
// finishing of a group for its walk and the group before, a walk for its replay and the finishing of two groups ago; so of
// the jobs not yet done the first can always go on.
// WIDE: the walk on several CUs, two, or with PARTS (groups replayed in parts) four.  IMG: the replays evaluate the GELU family for a walk on one CU
// (on two or four its waves have the time).  EVEN: a walk on four, and as many replaying workgroups for every pair.  OWN: a
// finishing workgroup, if any, for every pair.
template <bool WIDE, bool IMG, bool EVEN, bool OWN, bool PARTS>
__global__ __launch_bounds__(BW_THREADS) void ttt_mlp_bwd_gang_kernel(const BwdParams p) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  // (57 to 64 pairs wait for their walks: the stores of the eighths cost them nothing, registers for the sum do: 64 x 128 2.231 ms so, 2.245 with them)
  constexpr bool EIGHTHS = PARTS || (!WIDE && OWN);
  constexpr bool QUAD = WIDE && PARTS, IMAGES = IMG && !WIDE;
  constexpr int WALKERS = QUAD ? BWQ_CUS : WIDE ? 2 : 1;   // per pair
  const int b = blockIdx.x, walkers = WALKERS * p.gang_pairs;
  const int slots = walkers + p.n_finish + p.n_replay;
  const int gang = uni(p.scatter ? b / slots : b & 7);   // (a division leaves its result in a vector register)
  int slot = uni(p.scatter ? b % slots : b >> 3);
  const int pairs = (p.nbh - gang + 7) / 8;   // of this gang
  // Where every pair has as many replaying workgroups, what belongs to a pair is placed side by side (24 pairs x 512 4.66 ms, 4.70 by
  // kind; the CUs that share an instruction cache are a few workgroups apart).
  if (QUAD ? EVEN : OWN && slots % p.gang_pairs == 0) {
    const int per = uni(slots / p.gang_pairs), i = uni(slot / per), role = slot - i * per;
    slot = role < WALKERS ? WALKERS * i + role : walkers + (role - WALKERS) * p.gang_pairs + i;
  }
  if (pairs <= 0) return;
  const int bh0 = p.bh0 + gang;
  if (slot < walkers) {
    const int i = slot / WALKERS;
    if (i >= pairs) return;
    if constexpr (QUAD) bwd_quad_walk(p, smem, bh0 + 8 * i, slot & 3);
    else if constexpr (WIDE) bwd_wide_walk(p, smem, bh0 + 8 * i, slot & 1);
    else bwd_body<2, IMAGES, true>(p, smem, bh0 + 8 * i, p.K - 1, 0);
    return;
  }
  slot -= walkers;
  if (WIDE && threadIdx.x < pairs) say_worker(p.sync + (size_t)(bh0 + 8 * (int)threadIdx.x) * BWD_SYNC_STRIDE + BWW_WORKERS);
  const bool replays = slot >= p.n_finish;
  const int r = slot - p.n_finish;
  if (replays) {
    const int shared = PARTS ? min(p.n_shared, p.K) : 0, shared_jobs = shared * pairs * p.n_parts, jobs = shared_jobs + (p.K - shared) * pairs;
    for (int job = r; job < jobs; job += p.n_replay) {
      int n = job, part = 0, before = 0;   // job -> number of the group and pair, ordered by group and then by pair
      if (PARTS && job < shared_jobs) {
        n = uni(job / p.n_parts);
        part = job - n * p.n_parts;
      } else {
        n = job - shared_jobs;
        before = shared;
      }
      const int q = uni(n / pairs), k = uni(p.K - 1 - (before + q));
      if (!bwd_body<1, IMAGES, true, WIDE, PARTS, false, EIGHTHS>(p, smem, uni(bh0 + 8 * (n - q * pairs)), k, k, uni(part))) return;
    }
  }
  if constexpr (QUAD) return;
  if constexpr (OWN) {
    if (!replays && slot < pairs) bwd_finish_dxk<IMAGES, WIDE, true, EIGHTHS>(p, smem, bh0 + 8 * slot, p.K - 1);
  } else {
    // (n_replay >= pairs: one of the last groups each)
    const int last = (p.K - 1) * pairs, end = replays ? last + pairs : last;
    for (int job = replays ? last + r : slot; job < end; job += replays ? p.n_replay : p.n_finish) {
      const int done = uni(job / pairs);
      if (!bwd_finish_dxk<IMAGES, WIDE, false, EIGHTHS>(p, smem, bh0 + 8 * (job - done * pairs), p.K - 1 - done)) return;
    }
  }
}

// Clears the synchronisation words and marks every word of the exchange empty.
__global__ void ttt_mlp_bwd_wide_clear(int* w, int n, const int* report, uint4* x, int nx) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  clear_word(w, n, i, report);
  if (i < nx) x[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
}

}  // namespace ttt

hipError_t ttt_mlp_bwd_gang_enqueue(const ttt::BwdParams& p, TttKernel kernel, int grid, hipStream_t stream) {
  auto launch = [&](auto k) -> hipError_t {
    const int n = static_cast<int>(ttt::bwd_sync_ints(p.nbh));
    int* const words = p.status - (size_t)p.nbh * ttt::BWD_SYNC_STRIDE;   // p.sync and p.xchg are moved back by bh0 entries
    const int per = kernel == BWD_GANG_AHEAD || kernel == BWD_GANG_PARTS ? ttt::BWQ_XCHG_WORDS : ttt::BWW_XCHG_WORDS, nx = p.wide ? p.nbh * (per / 2) : 0;
    hipLaunchKernelGGL(ttt::ttt_mlp_bwd_wide_clear, dim3(((nx > n ? nx : n) + 255) / 256), dim3(256), 0, stream, words, n, p.report,
                       reinterpret_cast<uint4*>(p.xchg + (size_t)p.bh0 * per), nx);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, ttt::SM_BWD_BYTES);   // (while that runs)
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k, dim3(grid), dim3(ttt::BW_THREADS), ttt::SM_BWD_BYTES, stream, p);
    return hipGetLastError();
  };
  switch (kernel) {
    TTT_BWD_GANG_KERNELS(TTT_KERNEL_LAUNCH)
    default: return hipErrorInvalidValue;
  }
}
