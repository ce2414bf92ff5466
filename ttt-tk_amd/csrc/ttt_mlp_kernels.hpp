// Internal interface between the C ABI and the kernel translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ttt {

struct FwdParams {
  const __bf16 *XQ, *XK, *XV, *last_eta;
  const float *ttt_norm_weight, *ttt_norm_bias;
  const float *W1, *b1, *W2, *b2;
  float *W1_ck, *b1_ck, *W2_ck, *b2_ck;
  __bf16* Out;
  int B, NH, NC, K, cgs;
  // Two-workgroup mode only (sync != nullptr): per (batch, head) a ring of 2 * FWD_RING_MAX mini-batch slots
  // (2 << ring_log2 of them in use: 1 << ring_log2 mini-batches per hand-over, chosen by the launcher from NC)
  // with the bf16 operand images (64 KiB) and the bias vectors (256 + 64 floats) of the state after a
  // mini-batch, and the words the two workgroups signal with (layout as in the backward).
  // The workspace pointers are indexed by the global (batch, head) number like everything else: the
  // launcher passes them moved back by bh0 entries.
  __bf16* state_img;
  float* bias_img;
  int ring_log2;
  int* sync;
  int* status;    // the status word behind the synchronisation words
  int* report;    // one more int, in host memory, that a wait that gives up is told to (or nullptr)
  unsigned long long wait_limit;   // ticks of the 100 MHz clock a workgroup waits for another before it gives up
  // Recurrence on two workgroups (ttt_mlp_fwd_wide.hip): what they exchange, [B*NH][2 parities][2 halves][2 token blocks][2 x 2048 fp32];
  // the ring then has FWD_WIDE_RING slots.  On four (quad != 0, ttt_mlp_fwd_quad.hpp): FWD_QUAD_XCHG_WORDS per pair, and no ring.
  // scatter: the workgroups of a pair on consecutive XCDs instead of on one, for tests.
  unsigned long long* xchg;
  int quad, scatter;
  int bh0, nbh;   // this launch covers (batch, head) pairs bh0 .. bh0 + nbh - 1
  // One workgroup per pair, sequence cut into segments (seg_len > 0, a multiple of cgs): workgroup i of the launch
  // runs job job0 + i, job q = segment q / (B*NH) of pair q % (B*NH); a segment starts from the checkpoint that the
  // segment before it left (an earlier launch on the same stream) and leaves the one the next starts from.
  int seg_len, job0;
#ifdef TTT_STAGE_CLOCKS
  unsigned* stage_clocks;   // [B*NH][STAGE_ROLES][8 waves][STAGE_SLOTS] or nullptr (see below)
#endif
};
constexpr int FWD_RING_MAX = 32;               // most mini-batches per hand-over (8 or 32 are compiled)
constexpr int FWD_WIDE_RING = 8;               // ring slots with the recurrence on two workgroups
constexpr int FWD_XCHG_WORDS = 2 * 2 * 2 * 2048;  // 8-byte words of a pair's exchange: 128 KiB
constexpr int FWD_QUAD_XCHG_WORDS = 48640;      // with the recurrence on four workgroups (ttt_mlp_fwd_quad.hpp): 380 KiB
constexpr int FWD_IMG_BYTES = 64 * 256 * 2 * 2;  // W1 and W2 as bf16 operands
constexpr int FWD_BIAS_FLOATS = 256 + 64;

constexpr int BWD_MAX_PARTS = 4;
constexpr int BWD_MAX_SETS = 6;   // sets of per-group tensors in use at once, at most

// A set of the per-group tensors that carry a replayed group to the walk.
struct BwdSet {
  __bf16 *X2_group, *Z1_group, *Z1_bar_group, *X2_bar_group, *grad_l_wrt_Z2_group, *grad_l_wrt_Z1_group;
  __bf16 *x_hat_fused_group, *grad_x_hat_fused_group, *grad_output_fused_group;
  float *std_fused_group, *W1_init_group;
};
constexpr int BWD_HELP_SETS = 3;
struct BwdParams {
  const __bf16 *XQ, *XK, *XV, *last_eta;
  const float *ttt_norm_weight, *ttt_norm_bias;
  const float *W1_ck, *b1_ck, *W2_ck, *b2_ck;
  float *W1_init_group, *b1_init_group, *W2_init_group, *b2_init_group;
  __bf16* x_hat_ln_group;
  float* std_ln_group;
  __bf16 *X2_group, *Z1_group, *Z1_bar_group, *X2_bar_group;
  __bf16 *grad_l_wrt_Z2_group, *grad_l_wrt_Z1_group;
  __bf16 *x_hat_fused_group, *grad_x_hat_fused_group, *grad_output_fused_group;
  float* std_fused_group;
  const float *grad_L_W1_last, *grad_L_b1_last, *grad_L_W2_last, *grad_L_b2_last;
  const __bf16* grad_L_XQW;
  float *grad_L_ttt_norm_weight, *grad_L_ttt_norm_bias;
  float *grad_L_W1_init, *grad_L_b1_init, *grad_L_W2_init, *grad_L_b2_init;
  __bf16 *grad_L_last_eta, *grad_L_XQ, *grad_L_XK, *grad_L_XV;
  int B, NH, NC, K, cgs;
  // Several workgroups per (batch, head) only (sync != nullptr): replays, the walk and, in a gang, the finishing of the groups
  // on workgroups of their own.  Group number g (0 = the last group of the sequence) is replayed into set g % n_sets of the
  // per-group tensors that carry it to the walk: set 0 = the caller's tensors, sets 1.. = alt_*[set - 1] from the workspace.
  __bf16 *alt_X2_group[BWD_MAX_SETS - 1], *alt_Z1_group[BWD_MAX_SETS - 1], *alt_Z1_bar_group[BWD_MAX_SETS - 1], *alt_X2_bar_group[BWD_MAX_SETS - 1];
  __bf16 *alt_grad_l_wrt_Z2_group[BWD_MAX_SETS - 1], *alt_grad_l_wrt_Z1_group[BWD_MAX_SETS - 1];
  __bf16 *alt_x_hat_fused_group[BWD_MAX_SETS - 1], *alt_grad_x_hat_fused_group[BWD_MAX_SETS - 1], *alt_grad_output_fused_group[BWD_MAX_SETS - 1];
  float* alt_std_fused_group[BWD_MAX_SETS - 1];
  float* alt_W1_init_group[BWD_MAX_SETS - 1];
  // [B*NH][BWD_MAX_SETS][8][8 waves][2][64]: the replay's share of the norm-weight / norm-bias gradients of the group in a set, by eighths
  // of it (bwd_body's EIGHTHS), else their sum in the place of the first
  float* norm_partial;
  float* norm_park;      // [B*NH][8 waves][2][64]: their sum over the groups walked so far (without a grad_L_XK workgroup)
  __bf16* walk_park;     // [B*NH][64][256]: one register image the walking workgroup parks across its LayerNorm stage
  // Gang (gang_pairs > 0: pairs per XCD, gang g = pairs g, g + 8, ..; ttt_mlp_bwd_wide.hip): n_replay workgroups replay for all of
  // its pairs, n_finish form grad_L_XK, grad_L_XV and the walk's share of the norm gradients from what the walk hands over per
  // mini-batch - one register image (dZ1: [B*NH][2 sets][cgs][64][256] bf16) and two fp32 tiles (g_y and the norm-weight
  // gradient terms: [B*NH][2][cgs][2][64][64]); the two sets alternate by group.  They keep their own copy of the running
  // gradient wrt W1 and form G1 = -eta * dl/dZ1 themselves; fin_park: [B*NH][FIN_PARK_FLOATS], that copy and the norm-gradient
  // sums between two groups of a pair (n_finish < gang_pairs only).
  int gang_pairs, n_replay, n_finish;
  // One workgroup per pair and CUs to spare (n_helpers > 0): these replay groups ahead of the pairs, into sets 1 .. n_sets - 1 of
  // help_sets (0: the caller's tensors).
  int n_helpers;
  BwdSet help_sets[BWD_HELP_SETS];
  // The first n_shared groups (at most n_sets) are replayed in n_parts stretches, by as many workgroups at once: part i its eighths
  // part_start[i] .. part_start[i + 1] - 1.
  int n_shared, n_parts, part_start[BWD_MAX_PARTS + 1];
  __bf16* fin_dz;
  float* fin_gy;
  float* fin_park;
  // wide: the walk on two workgroups, which exchange through xchg, [B*NH][2 parities][2 halves][2 token blocks][BWW_WORDS *
  // 256 8-byte words]; or on four, which form grad_L_XK, grad_L_XV and the norm gradients as well (n_finish = 0), and exchange through
  // [B*NH][BWQ_XCHG_WORDS], which reaches into what fin_dz and fin_gy are otherwise.
  // scatter: the workgroups of a gang on consecutive XCDs instead of on one, for tests.
  int wide;
  unsigned long long* xchg;
  int n_sets;
  int scatter;
  int* sync;
  int* status;    // the status word behind the synchronisation words
  int* report;    // one more int, in host memory, that a wait that gives up is told to (or nullptr)
  unsigned long long wait_limit;   // ticks of the 100 MHz clock a workgroup waits for another before it gives up
  int overwrite;  // non-zero: grad_L_XQ / XK / XV / last_eta are stored, not added to (every element is written exactly once)
  int bh0, nbh;   // this launch covers (batch, head) pairs bh0 .. bh0 + nbh - 1 (workspace pointers moved back by bh0 entries)
  // One workgroup per pair, sequence cut into segments of seg_groups checkpoint groups (> 0): workgroup i of the launch
  // runs job job0 + i, job q = segment q / (B*NH) of pair q % (B*NH), segment 0 being the sequence's last groups.  A
  // segment takes the running gradients from grad_L_*_init, where the segment before it (an earlier launch on the same
  // stream) left them, and the norm-gradient sums from the pair's slots of x_hat_ln_group.
  int seg_groups, job0;
#ifdef TTT_STAGE_CLOCKS
  unsigned* stage_clocks;   // [B*NH][STAGE_ROLES][8 waves][STAGE_SLOTS] or nullptr (see below)
#endif
};

// Layout of `sync` (ints): 32 per (batch, head).  Words 0 .. 5: the parts of groups replayed into each set
// so far (norm_partial is written with them).  Walk on one workgroup: word 16 the groups it has finished, word 12 the
// mini-batches of the last group it walks that it has handed on (that group is handed over in chunks).  Word 24 the groups
// whose finishing is done - then one status word behind all of them (non-zero: a wait gave up).
constexpr int BWD_SYNC_STRIDE = 32;
// One workgroup per pair with helpers: words 1, 2 the group last replayed into that set, + 1; words BWD_HELP, + 1 (one 8-byte word)
// where the pair is and what is taken: bits 0-23 two times the number of the group it is at, + 1 from its walk on; bits 24-43
// and 44-63 the number, + 1, of the group taken into set 1 and 2 (0: the set is free).  A sequence has fewer than 2^18 groups
// (its tensors stay below 2 GiB per pair).
constexpr int BWD_HELP = 16;
// With the walk on two workgroups: BWW_WALKED + 0 / 4 groups and BWW_GIVEN + 0 / 4 mini-batches done by its two halves,
// BWW_XCD .. their XCDs, BWW_WORKERS (two words) the gang's other workgroups by XCD.
constexpr int BWW_WORDS = 9;                                // per lane: two times 8 fp32 sums and the token's share of d eta
constexpr int BWW_XCHG_WORDS = 2 * 2 * 2 * BWW_WORDS * 256;  // 8-byte words of a pair's exchange: 144 KiB
// With the walk on four (ttt_mlp_bwd_quad.hpp, which names its own words): those that count groups done, words 8, 12 and 24, alike.
constexpr int BWQ_XCHG_WORDS = 31744;                       // 248 KiB
constexpr int BWW_WALKED = 8, BWW_GIVEN = 16, BWW_XCD = 26, BWW_WORKERS = 28;
constexpr int FIN_PARK_FLOATS = 64 * 256 + 8 * 4 * 64;
inline size_t bwd_sync_ints(long long BH) { return (size_t)BH * BWD_SYNC_STRIDE + 32; }   // 32: STATUS_WORDS (ttt_mlp_common.hpp)

// ---- optional stage clocks.  A library built with -DTTT_STAGE_CLOCKS (stage_clocks.py builds one beside the product
// library) reads the shader clock at the boundaries of the stages named here and adds up, per wave, the clocks
// spent in each; every wave stores its sums when the kernel ends.  The product library
// is built without the macro and contains none of this.  Reading the clock is a scalar-memory operation: every
// boundary also waits for the wave's outstanding LDS reads, which makes an instrumented kernel some 10 % slower.
// Role of a workgroup in the buffer: forward 0 = the recurrence (or the one workgroup), 1 / 2 = the output branch, 3 / 4 = the halves
// of a recurrence on two workgroups; backward 0 = the replaying workgroups together, 4 = the reverse walk (or the one
// workgroup), 5 = the grad_L_XK workgroup, 6 / 7 = the halves of a walk on two workgroups.
constexpr int STAGE_SLOTS = 24;
constexpr int STAGE_ROLES = 8;
constexpr int STAGE_ROLE_OUT = 1, STAGE_ROLE_HALF = 3, STAGE_ROLE_WALK = 4, STAGE_ROLE_DXK = 5, STAGE_ROLE_WALK_HALF = 6;
enum FwdStage {
  FS_TOP,            // barrier that opens the mini-batch, checkpoint store, wait for the other workgroup
  FS_F1_GELU,        // Z1 = XK W1 + b1, GELU and its derivative
  FS_X2_SPLIT,       // X2 in two terms, high-order term to LDS
  FS_F2_PAIRSUM,     // Z2 = X2 W2 and its sum over the wave pairs (two barriers)
  FS_LN,             // LayerNorm + loss gradient of 8 tokens per wave, G2 to LDS
  FS_LN_BARRIER,     // barrier after it
  FS_F3,             // G1 = (G2 W2^T) * GELU'(Z1), including the transposition of W2's terms through LDS
  FS_F4,             // W1 step
  FS_F5,             // W2 step and b2
  FS_HANDOVER,       // recurrence workgroup: state images for the output branch
  FS_PUBLISH,        // recurrence workgroup: counter for the output branch
  FS_OUT_FORWARD,    // output branch: Z1_bar, GELU, Z2_bar and its pair sum
  FS_OUT_LN,         // output branch: LayerNorm, residual, store; next inputs
  FS_COUNT
};
enum BwdStage {
  BS_GROUP,          // per checkpoint group: waits for the other workgroups, parking / loading of state and gradients
  BS_R_TOP,          // replay: barrier that opens the mini-batch
  BS_R_F1_GELU,      // replay: Z1, GELU family, images of Z1
  BS_R_F2_PAIRSUM,   // replay: Z2 and its pair sum
  BS_R_LN,           // replay: fused LayerNorm + loss gradient, saved tiles, barrier
  BS_R_F3,           // replay: G1
  BS_R_WSTEP,        // replay: W1 and W2 steps
  BS_R_IMAGES,       // replay: operand images of the state after the step
  BS_R_OUT_FORWARD,  // replay: output branch forward with its pair sum
  BS_R_OUT_LN,       // replay: output LayerNorm forward and backward, next inputs, barrier
  BS_R_OUT_BACKWARD, // replay: gZ1_bar, grad_L_XQ with its pair sum, images for the walk
  BS_W_TOP,          // walk: tiles of the mini-batch into LDS (two barriers)
  BS_W_BAR_TERMS,    // walk: what the output branch adds to the running gradients
  BS_W_STEP_BACK,    // walk: the weight step backwards up to its pair sum
  BS_W_PAIRSUM,      // walk: pair sum of it
  BS_W_LN,           // walk: second-order pass through the fused LayerNorm loss
  BS_W_LN_BARRIER,   // walk: barrier after it
  BS_W_MLP_BACK,     // walk: inner MLP backwards (to the second wave-level fence)
  BS_W_UPDATES,      // walk: updates of the running gradients
  BS_W_DXK,          // walk: grad_L_XK with its pair sum (not with a grad_L_XK workgroup)
  BS_PUBLISH,        // counters for the other workgroups
  BS_X_GROUP,        // grad_L_XK workgroup, per checkpoint group: waits for the walk to have finished the group
  BS_X_PRODUCTS,     // grad_L_XK workgroup: operands of the mini-batch from HBM, G1 and the products, to the pair sum
  BS_X_SUMS,         // grad_L_XK workgroup: pair sum, grad_L_XK / grad_L_XV, token sums of the norm gradients, barrier
  BS_COUNT
};
// The recurrence and the walk on two workgroups: their waves 0-3 (compute) and 4-7 (helpers) go through stages of their own.
enum FwdWideStage {
  FWC_BLOCK0,        // compute: checkpoint store, Z1 (unless it was started early), GELU and partial Z2 of token block 0
  FWC_B1,            // compute: barrier behind it
  FWC_BLOCK1,        // compute: the same for block 1, W2's terms transposed, the last state's images stored
  FWC_B2,            // compute: barrier behind it (block 0's sums have crossed and been normalised)
  FWC_STEP0,         // compute: G1 of block 0 and its share of the weight step
  FWC_B3,            // compute: barrier behind it (the same for block 1's sums)
  FWC_STEP1,         // compute: the same for block 1, the new state split into its terms
  FWH_ASK,           // helpers: the next inputs asked for, what the last mini-batch left in flight waited for
  FWH_B1,            // helpers: wait for block 0's partial sums
  FWH_SEND0,         // helpers: sum over this CU's hidden columns, sent to the other CU
  FWH_TAKE0,         // helpers: wait for the other CU's share of block 0
  FWH_LN0,           // helpers: LayerNorm and loss gradient of block 0, G2 to LDS, free ring slot waited for
  FWH_B2,            // helpers: wait for block 1's partial sums
  FWH_SEND1,         // helpers: as for block 0, with block 0's token sums for b2
  FWH_TAKE1,         // helpers: wait for the other CU's share of block 1
  FWH_LN1,           // helpers: LayerNorm and loss gradient of block 1, G2 to LDS
  FWH_B3,            // helpers: wait for block 0's weight step
  FWH_B2STEP,        // helpers: state announced, step of b2
  FWX_COUNT
};
// The recurrence on four workgroups.
enum FwdQuadStage {
  FQC_SUMS,          // compute: Z1, GELU and partial Z2
  FQC_B1,            // compute: barrier behind it
  FQC_OUTPUT,        // compute: the output branch of the mini-batch before, operands of the step, checkpoint
  FQC_B2,            // compute: barrier behind it (the sums have crossed and been normalised)
  FQC_G1,            // compute: G1, W2's step, G1 split
  FQC_B3,            // compute: barrier behind it
  FQC_STEP,          // compute: W1's step and the split of the new state
  FQC_B4,            // compute: barrier behind it
  FQH_TOP,           // helpers: marks of the last mini-batch waited for
  FQH_B1,            // helpers: wait for the partial sums
  FQH_SEND,          // helpers: sum over this CU's hidden columns, sent to the CUs that normalise it
  FQH_TAKE,          // helpers, two of the four: wait for the other CUs' shares
  FQH_LN,            // helpers, two of the four: LayerNorm and loss gradient of 8 tokens, G2 sent
  FQH_OUTPUT,        // helpers, the other two: Out of the mini-batch before the last
  FQH_TAKE2,         // helpers: marks, share of the step of b2; wait for the other CUs' G2
  FQH_B2,            // helpers: barrier behind it
  FQH_GIVE,          // helpers: Out's partial sums gathered, step of b2
  FQH_B3,            // helpers: wait for G1
  FQH_NEXT,          // helpers: Out's partial sums sent, the next inputs asked for
  FQH_B4,            // helpers: wait for the new state
  FQX_COUNT
};
enum BwdWideStage {
  BWC_BAR_TERMS,     // compute: what the output branch adds to the running gradients
  BWC_STEP0,         // compute: weight step backwards, partial sums of token block 0
  BWC_B1,            // compute: barrier behind it
  BWC_STEP1,         // compute: the same for block 1
  BWC_B2,            // compute: barrier behind it (block 0's sums have crossed, dZ2 of block 0 is there)
  BWC_PRODUCTS,      // compute: products of the inner MLP backwards that do not need the sums
  BWC_MLP0,          // compute: inner MLP backwards and updates, block 0
  BWC_B3,            // compute: barrier behind it (the same for block 1's sums)
  BWC_MLP1,          // compute: inner MLP backwards and updates, block 1
  BWH_ASK,           // helpers: next group waited for, gradient wrt b2, the next mini-batch's tiles asked for
  BWH_B1,            // helpers: wait for block 0's partial sums
  BWH_SEND0,         // helpers: last mini-batch announced, sum over this CU's hidden columns, sent to the other CU
  BWH_TAKE0,         // helpers: wait for the other CU's share of block 0
  BWH_LN0,           // helpers: second-order LayerNorm pass of block 0, dZ2 to LDS
  BWH_B2,            // helpers: wait for block 1's partial sums
  BWH_SEND1,         // helpers: as for block 0, with block 0's outputs stored and the next mini-batch's tiles put into LDS
  BWH_TAKE1,         // helpers: wait for the other CU's share of block 1
  BWH_LN1,           // helpers: second-order LayerNorm pass of block 1, dZ2 to LDS
  BWH_B3,            // helpers: wait for block 0's inner MLP backwards
  BWH_STORE1,        // helpers: block 1's outputs stored, gradient wrt b2
  BWX_COUNT
};
// The walk on four workgroups.
enum BwdQuadStage {
  BQC_BAR,           // compute: what the output branch adds to the running gradients
  BQC_BX,            // compute: barrier behind it
  BQC_STEP,          // compute: weight step backwards, shares of the sums
  BQC_B1,            // compute: barrier behind it
  BQC_PRODUCTS,      // compute: products that do not need the sums
  BQC_B2,            // compute: barrier behind it (the sums have crossed, dZ2 is there)
  BQC_MLP,           // compute: inner MLP backwards, the next mini-batch's output-branch images asked for
  BQC_B3,            // compute: barrier behind it
  BQC_UPDATE,        // compute: gradient wrt W1, shares of grad_L_XK, the next mini-batch's other images asked for
  BQC_BE,            // compute: barrier behind it
  BQH_GATHER,        // helpers: grad_L_XK's shares of the mini-batch before summed, XK and dl/dZ2 to LDS
  BQH_BX,            // helpers: barrier behind it
  BQH_ASK,           // helpers: those sums sent, marks, own tokens' inputs asked for, gradient wrt b2, next group waited for
  BQH_B1,            // helpers: wait for the shares of the sums
  BQH_SEND,          // helpers: sum over this CU's hidden columns, sent to the CUs that take it through the LayerNorm
  BQH_TAKE,          // helpers, two of the four: wait for the other CUs' shares
  BQH_LN,            // helpers, two of the four: second-order LayerNorm pass of 8 tokens, dZ2 sent
  BQH_DXK,           // helpers, the other two: grad_L_XK of the mini-batch before
  BQH_TAKE2,         // helpers: norm gradients; wait for the other CUs' dZ2
  BQH_B2,            // helpers: barrier behind it
  BQH_PUT,           // helpers: the next mini-batch's tiles asked for, gradient wrt b2
  BQH_B3,            // helpers: wait for dZ1
  BQH_NORM,          // helpers: per checkpoint group, the replays' norm-gradient sums; XQ and gZ2_bar to LDS, outputs
  BQH_BE,            // helpers: wait for the end of the mini-batch
  BQX_COUNT
};
static_assert(FS_COUNT <= STAGE_SLOTS && BS_COUNT <= STAGE_SLOTS && FWX_COUNT <= STAGE_SLOTS && FQX_COUNT <= STAGE_SLOTS && BWX_COUNT <= STAGE_SLOTS && BQX_COUNT <= STAGE_SLOTS, "stage slots");

}  // namespace ttt

#ifdef TTT_STAGE_CLOCKS
// Device buffers the next launches write their stage clocks to (nullptr: none): [B*NH][STAGE_ROLES][8][STAGE_SLOTS]
// unsigned ints each, zero-filled by the caller.
extern "C" void ttt_mlp_set_stage_clocks(unsigned* forward, unsigned* backward);
#endif

// The kernels that do a call's work: one is compiled per combination of roles.  X(number, kernel); the kernel's text is also its name
// in a trace.
#define TTT_FWD_KERNELS(X) \
  X(FWD_ONE, ttt_mlp_fwd_kernel) X(FWD_SPLIT_8, ttt_mlp_fwd_split_kernel<8>) X(FWD_SPLIT_32, ttt_mlp_fwd_split_kernel<32>)
#define TTT_FWD_WIDE_KERNELS(X) X(FWD_WIDE, ttt_mlp_fwd_wide_kernel) X(FWD_WIDE_EARLY, ttt_mlp_fwd_wide_early_kernel)
#define TTT_BWD_KERNELS(X) \
  X(BWD_ONE, ttt_mlp_bwd_kernel) X(BWD_HELPED, ttt_mlp_bwd_helped_kernel) \
  X(BWD_SPLIT_1, ttt_mlp_bwd_split_kernel<1>) X(BWD_SPLIT_2, ttt_mlp_bwd_split_kernel<2>)
#define TTT_BWD_GANG_KERNELS(X)                                                                                                    \
  X(BWD_GANG_AHEAD, ttt_mlp_bwd_gang_kernel<true, true, true, true, true>)                                                         \
  X(BWD_GANG_PARTS, ttt_mlp_bwd_gang_kernel<true, false, false, true, true>)                                                       \
  X(BWD_GANG_WIDE, ttt_mlp_bwd_gang_kernel<true, false, false, true, false>)                                                       \
  X(BWD_GANG_WIDE_SHARED, ttt_mlp_bwd_gang_kernel<true, false, false, false, false>)                                               \
  X(BWD_GANG, ttt_mlp_bwd_gang_kernel<false, true, false, true, false>)                                                            \
  X(BWD_GANG_SHARED, ttt_mlp_bwd_gang_kernel<false, true, false, false, false>)
#define TTT_KERNEL_NUMBER(number, ...) number,
enum TttKernel {
  TTT_FWD_KERNELS(TTT_KERNEL_NUMBER) TTT_FWD_WIDE_KERNELS(TTT_KERNEL_NUMBER)
  TTT_BWD_KERNELS(TTT_KERNEL_NUMBER) TTT_BWD_GANG_KERNELS(TTT_KERNEL_NUMBER)
};
#undef TTT_KERNEL_NUMBER
// A case of a switch over TttKernel.
#define TTT_KERNEL_LAUNCH(number, ...) case number: return launch(ttt::__VA_ARGS__);
// `grid` workgroups of `kernel`, behind a small kernel that clears the synchronisation words where p.sync is set.  FWD_ONE, FWD_SPLIT_*: one
// workgroup per (batch, head), or two (state recurrence / output branch).
hipError_t ttt_mlp_fwd_enqueue(const ttt::FwdParams& p, TttKernel kernel, int grid, hipStream_t stream);
// FWD_WIDE: the recurrence of every pair on four workgroups, or (p.quad == 0) on two beside one that computes Out; FWD_WIDE_EARLY: on four.
hipError_t ttt_mlp_fwd_wide_enqueue(const ttt::FwdParams& p, TttKernel kernel, int grid, hipStream_t stream);
hipError_t ttt_mlp_fwd_clear_words(int* words, int n, hipStream_t stream);   // zeroes n ints with a small kernel
// BWD_ONE, BWD_HELPED, BWD_SPLIT_*: one workgroup per (batch, head), with helpers, or two or three (replays / reverse walk).
hipError_t ttt_mlp_bwd_enqueue(const ttt::BwdParams& p, TttKernel kernel, int grid, hipStream_t stream);
// BWD_GANG*: p.gang_pairs pairs per XCD, walked by one or two workgroups each (p.wide), and workgroups that serve all of them.
hipError_t ttt_mlp_bwd_gang_enqueue(const ttt::BwdParams& p, TttKernel kernel, int grid, hipStream_t stream);
// Replays checkpoint group 0 and writes the sixteen per-group tensors row-major (side path, one workgroup per pair).
hipError_t ttt_mlp_export_group0_enqueue(const ttt::BwdParams& p, hipStream_t stream);
extern "C" int ttt_mlp_fwd_lds_bytes();
extern "C" int ttt_mlp_bwd_lds_bytes();
extern "C" int ttt_mlp_fwd_threads();
extern "C" int ttt_mlp_bwd_threads();
