// extern "C" entry points declared in include/ttt_mlp.h: argument validation on the host, then
// one asynchronous kernel launch.  Nothing here allocates or synchronises.
#include <atomic>

#include "ttt_mlp_operator.h"
#include "ttt_mlp_kernels.hpp"

namespace {

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <typename... P>
inline bool any_null(P... ptrs) { return ((ptrs == nullptr) || ...); }

template <typename... P>
inline bool all_aligned(P... ptrs) { return (aligned16(ptrs) && ...); }

int check_sizes(int B, int NH, int NC, int K, int cgs) {
  if (B <= 0 || NH <= 0 || NC <= 0 || K <= 0 || cgs <= 0) return TTT_MLP_ERR_BAD_ARG;
  if ((long long)K != ((long long)NC + cgs - 1) / cgs) return TTT_MLP_ERR_BAD_CKPT;
  if ((long long)B * NH > 0x7fffffffLL) return TTT_MLP_ERR_TOO_LARGE;
  // the kernels address one (batch, head) with 32-bit byte offsets: 8 KiB per mini-batch, 32 KiB per group slot
  if (NC > (1 << 18) || cgs > (1 << 16)) return TTT_MLP_ERR_TOO_LARGE;
  // ... and one checkpoint slot (64 KiB) with a 32-bit byte offset too
  if (K > (1 << 15)) return TTT_MLP_ERR_TOO_LARGE;
  return TTT_MLP_OK;
}

unsigned long long g_wait_limit = 2000000000ull;   // 20 s of the 100 MHz clock
int g_cu_budget = 0;   // CUs the caller says these launches can count on (0: all the device reports)

inline const __bf16* bf(const uint16_t* p) { return reinterpret_cast<const __bf16*>(p); }
inline __bf16* bf(uint16_t* p) { return reinterpret_cast<__bf16*>(p); }

}  // namespace

extern "C" int ttt_mlp_abi_version(void) { return TTT_MLP_ABI_VERSION; }

extern "C" void ttt_mlp_set_wait_limit(unsigned long long ticks_100mhz) { g_wait_limit = ticks_100mhz; }

extern "C" void ttt_mlp_set_compute_units(int compute_units) { g_cu_budget = compute_units > 0 ? compute_units : 0; }

extern "C" const char* ttt_mlp_error_string(int code) {
  switch (code) {
    case TTT_MLP_OK: return "success";
    case TTT_MLP_ERR_BAD_ARG: return "ttt_mlp: null pointer or non-positive size";
    case TTT_MLP_ERR_BAD_CKPT: return "ttt_mlp: number of checkpoints K must equal ceil(NC / checkpoint_group_size)";
    case TTT_MLP_ERR_ALIGN: return "ttt_mlp: every tensor pointer must be 16-byte aligned";
    case TTT_MLP_ERR_TOO_LARGE: return "ttt_mlp: B*NH exceeds the launch grid limit, or NC > 262144, or checkpoint_group_size > 65536, or more than 32768 checkpoints";
    case TTT_MLP_ERR_NO_ROOM: return "ttt_mlp: two workgroups per (batch, head) do not fit the compute units of this device; use ttt_mlp_fwd_launch / ttt_mlp_bwd_launch";
    case TTT_MLP_ERR_WORKSPACE: return "ttt_mlp: workspace smaller than ttt_mlp_fwd_workspace_bytes() / ttt_mlp_bwd_workspace_bytes()";
    case TTT_MLP_ERR_SCRATCH: return "ttt_mlp: ttt_mlp_fwd_launch_static serves at most 8 (batch, head) pairs (B*NH <= 8): its workspace is a fixed array in device memory";
    default: return hipGetErrorString(static_cast<hipError_t>(code));
  }
}

#ifdef TTT_STAGE_CLOCKS
namespace {
unsigned* g_stage_clocks_fwd = nullptr;
unsigned* g_stage_clocks_bwd = nullptr;
}  // namespace
extern "C" void ttt_mlp_set_stage_clocks(unsigned* forward, unsigned* backward) {
  g_stage_clocks_fwd = forward;
  g_stage_clocks_bwd = backward;
}
#endif

namespace {
int make_fwd_params(const ttt_mlp_fwd_args* a, ttt::FwdParams& p) {
  if (a == nullptr) return TTT_MLP_ERR_BAD_ARG;
  if (any_null(a->XQ, a->XK, a->XV, a->last_eta, a->ttt_norm_weight, a->ttt_norm_bias, a->W1, a->b1, a->W2, a->b2,
               a->W1_checkpoints, a->b1_checkpoints, a->W2_checkpoints, a->b2_checkpoints, a->Out))
    return TTT_MLP_ERR_BAD_ARG;
  if (int rc = check_sizes(a->B, a->NH, a->NC, a->K, a->checkpoint_group_size)) return rc;
  if (!all_aligned(a->XQ, a->XK, a->XV, a->last_eta, a->ttt_norm_weight, a->ttt_norm_bias, a->W1, a->b1, a->W2,
                   a->b2, a->W1_checkpoints, a->b1_checkpoints, a->W2_checkpoints, a->b2_checkpoints, a->Out))
    return TTT_MLP_ERR_ALIGN;
  p = ttt::FwdParams{};
  p.XQ = bf(a->XQ); p.XK = bf(a->XK); p.XV = bf(a->XV); p.last_eta = bf(a->last_eta);
  p.ttt_norm_weight = a->ttt_norm_weight; p.ttt_norm_bias = a->ttt_norm_bias;
  p.W1 = a->W1; p.b1 = a->b1; p.W2 = a->W2; p.b2 = a->b2;
  p.W1_ck = a->W1_checkpoints; p.b1_ck = a->b1_checkpoints; p.W2_ck = a->W2_checkpoints; p.b2_ck = a->b2_checkpoints;
  p.Out = bf(a->Out);
  p.B = a->B; p.NH = a->NH; p.NC = a->NC; p.K = a->K; p.cgs = a->checkpoint_group_size;
#ifdef TTT_STAGE_CLOCKS
  p.stage_clocks = g_stage_clocks_fwd;
#endif
  return TTT_MLP_OK;
}
}  // namespace

namespace {

// Validates the backward arguments and translates them for the kernels.
int make_bwd_params(const ttt_mlp_bwd_args* a, ttt::BwdParams& p) {
  if (a == nullptr) return TTT_MLP_ERR_BAD_ARG;
  if (any_null(a->XQ, a->XK, a->XV, a->last_eta, a->ttt_norm_weight, a->ttt_norm_bias, a->W1_checkpoints,
               a->b1_checkpoints, a->W2_checkpoints, a->b2_checkpoints, a->W1_init_group, a->b1_init_group,
               a->W2_init_group, a->b2_init_group, a->x_hat_ln_group, a->std_ln_group, a->X2_group, a->Z1_group,
               a->Z1_bar_group, a->X2_bar_group, a->grad_l_wrt_Z2_group, a->grad_l_wrt_Z1_group, a->x_hat_fused_group,
               a->grad_x_hat_fused_group, a->grad_output_fused_group, a->std_fused_group, a->grad_L_W1_last,
               a->grad_L_b1_last, a->grad_L_W2_last, a->grad_L_b2_last, a->grad_L_XQW_mini_batch,
               a->grad_L_ttt_norm_weight, a->grad_L_ttt_norm_bias, a->grad_L_W1_init, a->grad_L_b1_init,
               a->grad_L_W2_init, a->grad_L_b2_init, a->grad_L_last_eta, a->grad_L_XQ, a->grad_L_XK, a->grad_L_XV))
    return TTT_MLP_ERR_BAD_ARG;  // `Out` is unused and may be null
  if (int rc = check_sizes(a->B, a->NH, a->NC, a->K, a->checkpoint_group_size)) return rc;
  if (!all_aligned(a->XQ, a->XK, a->XV, a->last_eta, a->ttt_norm_weight, a->ttt_norm_bias, a->W1_checkpoints,
                   a->b1_checkpoints, a->W2_checkpoints, a->b2_checkpoints, a->W1_init_group, a->b1_init_group,
                   a->W2_init_group, a->b2_init_group, a->x_hat_ln_group, a->std_ln_group, a->X2_group, a->Z1_group,
                   a->Z1_bar_group, a->X2_bar_group, a->grad_l_wrt_Z2_group, a->grad_l_wrt_Z1_group, a->x_hat_fused_group,
                   a->grad_x_hat_fused_group, a->grad_output_fused_group, a->std_fused_group, a->grad_L_W1_last, a->grad_L_b1_last, a->grad_L_W2_last, a->grad_L_b2_last,
                   a->grad_L_XQW_mini_batch, a->grad_L_ttt_norm_weight, a->grad_L_ttt_norm_bias, a->grad_L_W1_init,
                   a->grad_L_b1_init, a->grad_L_W2_init, a->grad_L_b2_init, a->grad_L_last_eta, a->grad_L_XQ,
                   a->grad_L_XK, a->grad_L_XV))
    return TTT_MLP_ERR_ALIGN;
  p = ttt::BwdParams{};
  p.XQ = bf(a->XQ); p.XK = bf(a->XK); p.XV = bf(a->XV); p.last_eta = bf(a->last_eta);
  p.ttt_norm_weight = a->ttt_norm_weight; p.ttt_norm_bias = a->ttt_norm_bias;
  p.W1_ck = a->W1_checkpoints; p.b1_ck = a->b1_checkpoints; p.W2_ck = a->W2_checkpoints; p.b2_ck = a->b2_checkpoints;
  p.W1_init_group = a->W1_init_group; p.b1_init_group = a->b1_init_group;
  p.W2_init_group = a->W2_init_group; p.b2_init_group = a->b2_init_group;
  p.x_hat_ln_group = bf(a->x_hat_ln_group); p.std_ln_group = a->std_ln_group;
  p.X2_group = bf(a->X2_group); p.Z1_group = bf(a->Z1_group);
  p.Z1_bar_group = bf(a->Z1_bar_group); p.X2_bar_group = bf(a->X2_bar_group);
  p.grad_l_wrt_Z2_group = bf(a->grad_l_wrt_Z2_group); p.grad_l_wrt_Z1_group = bf(a->grad_l_wrt_Z1_group);
  p.x_hat_fused_group = bf(a->x_hat_fused_group); p.grad_x_hat_fused_group = bf(a->grad_x_hat_fused_group);
  p.grad_output_fused_group = bf(a->grad_output_fused_group); p.std_fused_group = a->std_fused_group;
  p.grad_L_W1_last = a->grad_L_W1_last; p.grad_L_b1_last = a->grad_L_b1_last;
  p.grad_L_W2_last = a->grad_L_W2_last; p.grad_L_b2_last = a->grad_L_b2_last;
  p.grad_L_XQW = bf(a->grad_L_XQW_mini_batch);
  p.grad_L_ttt_norm_weight = a->grad_L_ttt_norm_weight; p.grad_L_ttt_norm_bias = a->grad_L_ttt_norm_bias;
  p.grad_L_W1_init = a->grad_L_W1_init; p.grad_L_b1_init = a->grad_L_b1_init;
  p.grad_L_W2_init = a->grad_L_W2_init; p.grad_L_b2_init = a->grad_L_b2_init;
  p.grad_L_last_eta = bf(a->grad_L_last_eta);
  p.grad_L_XQ = bf(a->grad_L_XQ); p.grad_L_XK = bf(a->grad_L_XK); p.grad_L_XV = bf(a->grad_L_XV);
  p.B = a->B; p.NH = a->NH; p.NC = a->NC; p.K = a->K; p.cgs = a->checkpoint_group_size;
  p.overwrite = a->overwrite != 0;
#ifdef TTT_STAGE_CLOCKS
  p.stage_clocks = g_stage_clocks_bwd;
#endif
  return TTT_MLP_OK;
}

// Several workgroups per (batch, head) wait for each other, so all of them must be resident at once: one
// workgroup fills a CU (LDS), hence such a launch may not exceed the CUs of the current device.  The
// (batch, head) pairs are therefore covered by two launches in a row: as many full rounds of one
// workgroup per pair as there are (a multiple of the CU count), then the rest - with several workgroups per
// pair if two each fit the device (split), otherwise with one.
// With the recurrence (walk) of a pair on two CUs (wide), or workgroups that serve several pairs (gang), the workgroups of a
// pair share an XCD: the grid is padded to a multiple of 8 pairs and dealt to the 8 XCDs in turn, so those of
// ceil(pairs / 8) pairs must fit an eighth of the CUs.
struct LaunchPlan {
  long long n_single = 0;   // pairs 0 .. n_single-1: one workgroup each
  long long n_rest = 0;     // pairs n_single .. n_single+n_rest-1
  bool rest_split = false;
  bool wide = false;
  bool quad = false;        // wide: the recurrence (walk) of a pair, and what hangs on it, on four CUs; else on two
  int gang = 0;             // backward: pairs of an XCD that share workgroups, 0: whole ones, that replay or walk, for each pair
  int n_replay = 0;         // backward: that replay checkpoint groups, of a gang or of a pair
  int n_finish = 0;         // backward, of a gang: for grad_L_XK / grad_L_XV
  int sets = 0;             // backward: sets of the per-group tensors
  int shared = 0;           // backward: groups, the first ones walked, that several workgroups at once replay
  int parts = 1;            // backward: that many, a stretch of the group each
  int helpers = 0;          // backward, one workgroup per pair: further ones that replay groups for all of them
  bool waits() const { return rest_split || helpers > 0; }                    // workgroups that wait for each other, in a workspace
  long long first_waiting() const { return helpers > 0 ? 0 : n_single; }      // of these pairs
  long long n_waiting() const { return helpers > 0 ? n_single : n_rest; }
  // Workgroups of an XCD: of a gang, or of the pairs that a forward with the recurrence on two CUs deals to it.
  int slots(bool backward) const {
    return backward ? (quad ? 4 : wide ? 2 : 1) * gang + n_finish + n_replay : static_cast<int>((n_rest + 7) / 8) * per_pair(false);
  }
  // The launch behind the full rounds of one workgroup per pair: its kernel and its workgroups.
  TttKernel kernel(bool backward, int NC) const {
    if (!backward && wide) return quad && NC <= 256 && n_rest * NC <= 6144 ? FWD_WIDE_EARLY : FWD_WIDE;   // (ttt_mlp_fwd_wide.hip)
    if (!backward) return NC >= 512 ? FWD_SPLIT_32 : FWD_SPLIT_8;   // (mini-batches per hand-over)
    if (helpers > 0) return BWD_HELPED;
    if (!gang) return n_replay == 2 ? BWD_SPLIT_2 : BWD_SPLIT_1;
    const bool own = n_finish == gang;
    if (quad) return n_replay % gang == 0 ? BWD_GANG_AHEAD : BWD_GANG_PARTS;
    if (wide) return own ? BWD_GANG_WIDE : BWD_GANG_WIDE_SHARED;
    return own ? BWD_GANG : BWD_GANG_SHARED;
  }
  long long grid(bool backward) const {
    if (helpers > 0) return n_single + helpers;
    if (wide || gang) return 8LL * slots(backward);
    return n_rest * (backward ? n_replay + 1 : 2);
  }
  // Workgroups per pair of the rest, whole ones where some are shared.
  int per_pair(bool backward) const {
    if (!rest_split) return 0;
    if (backward && gang) return slots(true) / gang;
    return backward ? n_replay + 1 : !wide ? 2 : quad ? 4 : 3;
  }
};
// Clocks per mini-batch, in hundreds, that the roles of a backward gang are busy for (stage clocks, 56 and 96 pairs x 512): the replay
// of a mini-batch and its finishing; with the GELU family evaluated by the replay, and so not by the others; the walk of one on two CUs, on
// one, and on one that does the finishing too.  Then what a group costs each role whatever its length (fitted, with the last of the walks, to
// 273 calls of 49 to 80 pairs, groups of 1 to 64 and 2 to 16 of them).
constexpr int COST_REPLAY = 443, COST_FINISH = 200, COST_REPLAY_IMG = 488, COST_FINISH_IMG = 185;
constexpr int COST_WALK_WIDE = 215, COST_WALK = 330, COST_WALK_ALL = 400;
constexpr int COST_GROUP_REPLAY = 550, COST_GROUP_WALK = 250, COST_GROUP_FINISH = 450;
// `workers` of an XCD divided between replaying and finishing for its `pairs`, so that the slower of the two is as fast as can be;
// a finishing workgroup for each pair, which then follows its walk closely, where the replay still keeps up with `walk`.
void divide_workers(int pairs, int workers, int walk, int replay, int finish, int* n_replay, int* n_finish) {
  *n_finish = pairs;
  if (workers - pairs < pairs || replay * pairs > walk * (workers - pairs)) {
    int best = 0;
    for (int f = 1; f < pairs && workers - f >= pairs; f++) {
      const int r = workers - f, tr = replay * pairs / r, tf = finish * pairs / f, t = tr > tf ? tr : tf;
      if (best == 0 || t < best) {
        best = t;
        *n_finish = f;
      }
    }
  }
  *n_replay = workers - *n_finish;
}
// Where the stretches of a group begin, in eighths of it.  To the state at its first mini-batch a workgroup takes the half of every
// replay before that carries the state, about a third of the whole, so the stretches get shorter.
constexpr int PART_START[ttt::BWD_MAX_PARTS][ttt::BWD_MAX_PARTS + 1] = {{0, 8, 8, 8, 8}, {0, 5, 8, 8, 8}, {0, 4, 6, 8, 8}, {0, 3, 5, 7, 8}};
// One workgroup for each of 129 to 248 pairs on 256 CUs: the CUs left over replay groups for all of them (ttt_mlp_bwd.hip).  In ms,
// backward alone -> with helpers (two sets for the groups they take; with one 168 x 128 4.37, 176 x 128 4.92): 136 pairs x 128
// mini-batches 4.71 -> 3.77, 168 x 128 4.87 -> 4.20, 200 x 100 4.03 -> 3.78, 200 x 256 10.44 -> 9.52, 232 x 512 21.9 -> 21.0, 248 x 512
// 22.7 -> 22.3.  (In clocks it is twice that: a device with every CU busy runs slower, and the forward after it too, 1.20 -> 1.33 ms for
// 200 x 100; both together 5.24 -> 5.10 ms.)  Fewer than one helper per XCD gain less than that costs.
constexpr int MIN_HELPERS = 8;
LaunchPlan plan_for(long long BH, int cus, bool backward) {
  LaunchPlan pl;
  if (BH <= 0 || cus <= 0) {
    pl.n_single = BH > 0 ? BH : 0;
    return pl;
  }
  pl.n_single = BH / cus * cus;
  pl.n_rest = BH - pl.n_single;
  pl.rest_split = pl.n_rest > 0 && 2 * pl.n_rest <= cus;
  if (!pl.rest_split) {
    pl.n_single = BH;
    pl.n_rest = 0;
    if (backward && BH <= cus - MIN_HELPERS) {
      pl.helpers = static_cast<int>(cus - BH);
      pl.sets = ttt::BWD_HELP_SETS;
    }
    return pl;
  }
  const long long per_xcd = (pl.n_rest + 7) / 8;
  const auto fits_xcd = [&](int per) { return per * per_xcd <= cus / 8; };
  if (!backward) {
    pl.quad = fits_xcd(4);
    pl.wide = fits_xcd(3);
    return pl;
  }
  // Three replaying workgroups per pair or more leave the walk to itself, and it has four CUs (against two, with one more that fetched ahead for
  // them and one that finished, in ms: 2 pairs x 4 0.093 -> 0.063, 12 x 64 0.627 -> 0.540, 24 x 64 0.695 -> 0.584, 16 x 256 2.22 -> 1.87,
  // 24 x 512 4.59 -> 3.79, 32 x 512 4.87 -> 4.03; with the GELU family evaluated by the replays, three images instead of one, 24 x 512 3.94, 32 x 512
  // 4.28).  The same with 2.4 of them (against three, two walking and one finishing: 33 x 128 1.44 -> 1.35, 40 x 64 0.817 -> 0.743, 40 x 256
  // 2.79 -> 2.46): a replay takes 43 k clocks a mini-batch, the walk 16 k; with 1.3 (48 pairs) they would bound it by far.
  // What is left is the walk's wait for the first group's replay: the first groups are replayed by two to four workgroups at once, and as many groups
  // that way as it takes for a group replayed by one workgroup to be ready in time (three: replay of a group 57 k clocks a
  // mini-batch, in two parts 35 k, in four 27 k).  In ms, walk on two CUs, four replaying workgroups and whole groups -> so: 8 pairs x 64 in groups of 8
  // 0.683 -> 0.617 (four parts, eight workgroups), 24 x 64 0.733 -> 0.691 and 24 x 512 in groups of 32 4.88 -> 4.64 (three, six),
  // 32 x 512 5.12 -> 5.06 (two, four; all groups in parts: 5.25, the work done twice takes clock from the walk).
  const int on_xcd = cus / 8, pairs = static_cast<int>(per_xcd);
  if (fits_xcd(7)) {
    const int each = on_xcd / pairs - 4;
    pl.wide = pl.quad = true;
    pl.gang = pairs;
    pl.parts = each >= 8 ? 4 : each >= 6 ? 3 : each >= 4 ? 2 : 1;
    pl.shared = each >= 4 ? 3 : 0;
    pl.n_replay = (each >= 4 ? 2 * pl.parts : 3) * pairs;
    pl.sets = each >= 4 ? 6 : 5;
    return pl;
  }
  // Two replaying workgroups per pair bound a walk on two CUs (48 pairs x 4,096 mini-batches: 20 us per replayed mini-batch, 10.1 us
  // per walked one); a third for some of the pairs gained nothing (48 x 512: 5.95 ms with 12 or 14 of them on an XCD).  With less
  // room than that the workgroups of an XCD that replay and those that finish serve all of its pairs.  The walks take two CUs
  // each from 4.5 CUs per pair on (56 pairs x 512 7.75 -> 6.85 ms, 51 x 77 1.46 -> 1.22 ms against one CU each and four whole
  // workgroups per pair; but 64 x 512 8.30 ms so, 8.13 with one CU each), one from 3 CUs on (72 x 512 9.57 -> 8.96 ms, 80 x 512
  // 9.71 -> 9.35 ms against three whole workgroups per pair; but 96 x 512 11.3 ms so, 10.3 with two).
  if (3 * pairs <= on_xcd) {
    pl.wide = 9 * pairs <= 2 * on_xcd;
    pl.gang = pairs;
    if (fits_xcd(6)) {   // (33 to 40 pairs: twelve of an XCD replay for its five)
      pl.quad = true;
      pl.n_replay = on_xcd - 4 * pairs;
      pl.parts = 2;
      pl.shared = 1;
    } else if (fits_xcd(5)) {
      pl.n_finish = pairs;
      pl.n_replay = 2 * pairs;
    } else if (pl.wide) {
      divide_workers(pairs, on_xcd - 2 * pairs, COST_WALK_WIDE, COST_REPLAY, COST_FINISH, &pl.n_replay, &pl.n_finish);
    } else {
      divide_workers(pairs, on_xcd - pairs, COST_WALK, COST_REPLAY_IMG, COST_FINISH_IMG, &pl.n_replay, &pl.n_finish);
    }
    pl.sets = 4;
    return pl;
  }
  pl.n_replay = 3 * pl.n_rest <= cus ? 2 : 1;
  pl.sets = 2 * pl.n_replay;
  return pl;
}
int device_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  return g_cu_budget > 0 && g_cu_budget < cus ? g_cu_budget : cus;
}
LaunchPlan plan_launches(long long BH, bool backward) { return plan_for(BH, device_cus(), backward); }

// More (batch, head) pairs than CUs, one workgroup each: the hardware runs them in rounds, and a last round that is
// not full leaves CUs idle for a whole sequence.  The forward can cut every sequence into segments at checkpoint
// boundaries instead - a segment starts from the checkpoint before its first mini-batch, which the segment before it
// left in the caller's checkpoint tensors - and launch the (segment, pair) jobs segment-major, one launch per `cus`
// jobs: a pair's earlier segment is always in an earlier launch (pairs >= cus), and the rounds are a fraction of a
// sequence long, so 384 pairs on 256 CUs take 3 launches of half a sequence, 1.5 sequences instead of 2 (or 1.7 with
// the last 128 pairs on two workgroups each).  Same arithmetic on the same state: results do not change.
struct SegmentPlan {
  int seg_len = 0;      // mini-batches per segment, a multiple of cgs; 0 = sequences are not cut
  int groups = 0;       // checkpoint groups per segment
  int launches = 1;
  long long jobs = 0;
};
// `alt_x1000`: what the alternative costs, in thousandths of a mini-batch of one workgroup.
SegmentPlan plan_segments(long long pairs, int cus, int NC, int cgs, bool backward, long long alt_x1000) {
  SegmentPlan best;
#ifndef TTT_STAGE_CLOCKS   // the stage clocks are kept per pair and sequence
  if (pairs <= cus || pairs > (1 << 27) || cus <= 0 || NC <= 0 || cgs <= 0) return best;   // (job numbers are ints)
  const int K = (NC + cgs - 1) / cgs;
  long long best_t = alt_x1000;
  for (int S = 2; S <= 8 && S <= K; S++) {
    const int groups = (K + S - 1) / S, segs = (K + groups - 1) / groups;
    const long long len = (long long)groups * cgs, jobs = segs * pairs, launches = (jobs + cus - 1) / cus;
    // A launch takes what the longest segment in it takes.  All have `len` mini-batches except the one with the sequence's last
    // group (the forward's last, the backward's first) and the one with the groups left over (the last): how many launches
    // hold nothing but those?
    const long long left = (long long)(K - (segs - 1) * groups) * cgs, missing = (long long)K * cgs - NC;
    const long long len0 = backward ? len - missing : len, len_last = backward ? left : left - missing;
    const long long n0 = pairs / cus, n_last = launches - ((segs - 1) * pairs + cus - 1) / cus;
    // + a mini-batch's worth per launch forward, a tenth backward: gaps, state in and out (measured 0.7 to 2 forward; backward what a launch costs
    // and what a device gains that is not full all the time cancel)
    const long long t = 1000 * (n0 * len0 + n_last * len_last + (launches - n0 - n_last) * len) + (backward ? 100 : 1000) * launches;
    if (t < best_t) {
      best_t = t;
      best.seg_len = static_cast<int>(len);
      best.groups = groups;
      best.launches = static_cast<int>(launches);
      best.jobs = jobs;
    }
  }
#endif
  return best;
}
// Thousandths of a one-workgroup mini-batch that the pairs take uncut: full rounds, and the rest either one more
// round or, with several workgroups per pair, a shorter one.  Measured on 256 CUs as what the rest adds to full rounds
// (6.5 ms forward, 23.1 ms backward for 512 mini-batches), at the most pairs of a shape.  Forward: 530 per mini-batch (4 pairs; 430
// for 64), 545 (80 pairs) and 650 (128 pairs), and the mini-batches by which Out trails.  The backward's walk waits for the
// first group's replay, hence the term in 1 / K: 4 to 32 pairs 240 at K = 16, 320 at 4; 48 pairs 265 and 335, 56 pairs 290 at
// K = 16, 64 pairs 350 and 435, 80 pairs 410 at K = 16, 85 pairs 435 and 515 at 4, 128 pairs 500 and 605; and a twentieth, behind a device
// that has been full.
// A last round that is not full is 5 % shorter than a full one (400 to 456 pairs).
// What the estimate decides: 312 pairs x 101 mini-batches in 4 groups, forward 1.70 ms cut, 1.93 uncut; 384 x 31 in 16, 0.65 and
// 0.78; 276 x 329 in 22, backward 17.5 and 18.7; 330 x 395 in 18, 24.3 and 27.3; 384 x 512 in 16, 35.1 and 34.8.  Of 144 backward calls of
// 260 to 384 pairs and 20 to 300 mini-batches timed both ways it takes the slower one for 2 by more than 2 % (with a mini-batch per launch and no
// twentieth for 40, by up to 11 %: 305 x 45 in groups of 5 2.75 cut, 3.03 uncut).
long long rest_x1000(const LaunchPlan& pl, int NC, int K, bool backward) {
  if (!backward) return pl.quad ? 525LL * NC + 3000 : pl.wide ? 545LL * NC + 8000 : 650LL * NC + (NC >= 512 ? 32000 : 8000);
  const int walk = pl.quad ? 210 : pl.wide ? (pl.gang > 6 ? 290 : 235) : pl.gang > 8 ? 380 : pl.gang ? 325 : pl.n_replay == 2 ? 405 : 485;
  return (long long)(walk + 470 / K) * NC * 21 / 20;
}
long long uncut_x1000(const LaunchPlan& pl, long long pairs, int cus, int NC, int cgs, bool with_workspace, bool backward) {
  if (cus <= 0) return (long long)NC * 1000;
  if (with_workspace && pl.rest_split) return pl.n_single / cus * 1000 * NC + rest_x1000(pl, NC, (NC + cgs - 1) / cgs, backward);
  return (pairs + cus - 1) / cus * (pairs % cus != 0 ? 950 : 1000) * NC;
}
// The launches of a call with the sequences cut: `cus` jobs each, in job order, on the one stream.
template <class Params, class Enqueue>
int launch_segments(Params p, const SegmentPlan& plan, int cus, Enqueue enqueue) {
  p.sync = nullptr;
  p.bh0 = 0;
  for (long long j0 = 0; j0 < plan.jobs; j0 += cus) {
    p.job0 = static_cast<int>(j0);
    p.nbh = static_cast<int>(plan.jobs - j0 < cus ? plan.jobs - j0 : cus);
    if (hipError_t e = enqueue(p)) return static_cast<int>(e);
  }
  return TTT_MLP_OK;
}
int launch_fwd_segments(ttt::FwdParams p, const SegmentPlan& plan, int cus, hipStream_t stream) {
  p.seg_len = plan.seg_len;
  return launch_segments(p, plan, cus, [stream](const ttt::FwdParams& q) { return ttt_mlp_fwd_enqueue(q, FWD_ONE, q.nbh, stream); });
}
// Backward: segment 0 = the last groups of every sequence.
int launch_bwd_segments(ttt::BwdParams p, const SegmentPlan& plan, int cus, hipStream_t stream) {
  p.seg_groups = plan.groups;
  return launch_segments(p, plan, cus, [stream](const ttt::BwdParams& q) { return ttt_mlp_bwd_enqueue(q, BWD_ONE, q.nbh, stream); });
}
SegmentPlan plan_bwd_segments(const LaunchPlan& pl, long long pairs, int cus, int NC, int cgs, bool with_workspace) {
  // (the two norm sums that a segment leaves behind, 4 KiB each, fill one 8 KiB slot of x_hat_ln_group)
  return plan_segments(pairs, cus, NC, cgs, true, uncut_x1000(pl, pairs, cus, NC, cgs, with_workspace, true));
}

// Sets of the per-group tensors that carry replayed groups to the walk, used in turn.  Set 0 is the caller's own; a sequence of K
// groups uses K.
int bwd_sets_used(const LaunchPlan& pl, long long K) { return static_cast<int>(K < pl.sets ? K : pl.sets); }
// Whether the helpers get to a group of every pair in time: a helper replays 1.75 groups while a pair's own workgroup replays and walks
// one, and there is nothing to take in the first of a pair.  If they do not, the pairs without help end as late as
// without helpers, at a lower clock: in ms, alone -> with helpers, 184 pairs x 32 mini-batches in 2 groups 1.349 -> 1.351 and 4 %
// on the forward after it, 200 x 64 in 2 2.58 -> 2.81, 200 x 48 in 3 2.01 -> 2.00; 160 x 32 in 2 1.28 -> 1.08, 200 x 64 in 4 2.62 -> 2.48.
bool helpers_pay(const LaunchPlan& pl, long long K) { return pl.helpers > 0 && 7 * pl.helpers * (K - 1) >= 4 * pl.n_waiting(); }
// The launch with less workspace for the same pairs: two replaying workgroups per pair instead of three or four.
LaunchPlan bwd_reduced(LaunchPlan pl) {
  if (pl.quad) {
    pl.n_finish = pl.gang;
    pl.n_replay = 2 * pl.gang;
    pl.parts = 1;
    pl.shared = 0;
    pl.quad = false;
    pl.sets = 4;
  }
  return pl;
}
// Clocks, in hundreds, until a gang, or two replaying workgroups, one that walks and (`finish` > 0) one that finishes for one pair, is through
// with a sequence: its jobs in their order, each as early as its workgroup and what it waits for allow.
int backward_span(int pairs, int n_replay, int n_finish, bool wide, int walk, int replay, int finish, int NC, int cgs, int K) {
  constexpr int SETS = 4;
  int replaying[64] = {}, finishing[64] = {}, walked[64] = {}, walk_end[SETS][64] = {}, finished[SETS][64] = {}, span = 0;
  const int groups = K < 16 ? K : 16;   // (longer: nothing new)
  for (int g = 0; g < groups; g++) {
    const int n = g == 0 ? NC - (K - 1) * cgs : cgs, now = g % SETS, last = (g + SETS - 1) % SETS, set = (g + SETS - 2) % SETS;
    const bool own = n_finish == pairs, end = g == groups - 1;
    int start[64];
    for (int i = 0; i < pairs; i++) {   // (the set of `now` is free once the group that used it last is walked and finished)
      int& w = replaying[(g * pairs + i) % n_replay];
      const int free = walk_end[now][i] > finished[now][i] ? walk_end[now][i] : finished[now][i];
      w = (w > free ? w : free) + COST_GROUP_REPLAY + n * replay;
      start[i] = w > walked[i] ? w : walked[i];
      if (finish > 0 && g >= 2 && finished[set][i] > start[i]) start[i] = finished[set][i];   // (two sets of what is handed over)
      walked[i] = start[i] + COST_GROUP_WALK + n * walk;
    }
    for (int i = 0; i < pairs; i++) {
      walk_end[now][i] = walked[i];
      if (finish > 0) {   // behind the walk mini-batch by mini-batch where it says so each (on two CUs, and in the last group), else behind the group
        int& w = own ? finishing[i] : end ? replaying[i % n_replay] : finishing[(g * pairs + i) % n_finish];
        int t = g > 0 && finished[last][i] > w ? finished[last][i] : w;
        const int from = wide || end ? start[i] : walked[i];
        t = (t > from ? t : from) + n * finish;
        if (t < walked[i] + finish) t = walked[i] + finish;
        finished[now][i] = w = t + COST_GROUP_FINISH;
      } else {
        finished[now][i] = walked[i];
      }
      if (finished[now][i] > span) span = finished[now][i];
    }
  }
  return span;
}
// The launch for groups as short, or as few, as the sequence at hand has.  Where workgroups that serve several pairs have to take another
// round for what does not divide among them, or spend themselves on what a group costs whatever its length, whole ones for each pair are
// faster: with the walk on two CUs and finishing workgroups that take turns (49 to 56 pairs) four with the walk on one, with the walk on
// one CU and less than four per pair (65 to 80) three, without finishing ones.  (gang / whole, 56 pairs: groups of 1 1.16 - 1.21, 16 of 2 1.08, 6 of
// 3 0.96, two of 64 and one of them half 1.05, five of 12 0.84; 72: 8 of 3 1.02, 16 of 6 0.93, two of 64 1.05, 12 of 16 0.95; 80: 16 of 6 1.04, three and
// a half of 24 to 48 1.05 - 1.07, 5 of 16 0.99, 8 of 32 0.97.)  Of 273 such calls timed both ways the spans take the slower launch for 3 by
// more than 1 %; with thresholds in group size and number it was 39, up to 7 %.
LaunchPlan bwd_for_groups(LaunchPlan pl, int cus, long long cgs, long long K, long long NC) {
  if (cgs < 2) {   // no stretches to divide a group into
    pl.parts = 1;
    pl.shared = 0;
  }
  const bool four = 4 * pl.gang <= cus / 8, shared = four ? pl.wide && !pl.quad && pl.n_finish < pl.gang : pl.gang && !pl.wide;
  if (!shared || cus / 8 > 64) return pl;
  const int n = static_cast<int>(NC), c = static_cast<int>(cgs), k = static_cast<int>(K);
  const int gang = pl.wide ? backward_span(pl.gang, pl.n_replay, pl.n_finish, true, COST_WALK_WIDE, COST_REPLAY, COST_FINISH, n, c, k)
                           : backward_span(pl.gang, pl.n_replay, pl.n_finish, false, COST_WALK, COST_REPLAY_IMG, COST_FINISH_IMG, n, c, k);
  const int whole = backward_span(1, 2, 1, false, four ? COST_WALK : COST_WALK_ALL, COST_REPLAY_IMG, four ? COST_FINISH_IMG : 0, n, c, k);
  if (gang < whole) return pl;
  if (four) {
    pl.wide = false;
    pl.n_finish = pl.gang;
    pl.n_replay = 2 * pl.gang;
  } else {
    pl.gang = pl.n_finish = 0;
    pl.n_replay = 2;
  }
  return pl;
}
// The launch of a backward call with a workspace.
LaunchPlan plan_bwd(long long pairs, int cus, long long cgs, long long NC) {
  return bwd_for_groups(plan_for(pairs, cus, true), cus, cgs, (NC + cgs - 1) / cgs, NC);
}
// What a call enqueues to do its work: sequences cut into segments, a device's worth of them at a time, or `n` kernels in a row.
struct Call {
  SegmentPlan seg;
  int n = 1;
  TttKernel kernel[2];
  long long grid[2];
};
Call plan_call(bool backward, const LaunchPlan& pl, long long pairs, int cus, int NC, int cgs, bool with_workspace) {
  Call c;
  c.kernel[0] = backward ? BWD_ONE : FWD_ONE;
  c.seg = backward ? plan_bwd_segments(pl, pairs, cus, NC, cgs, with_workspace)
                   : plan_segments(pairs, cus, NC, cgs, false, uncut_x1000(pl, pairs, cus, NC, cgs, with_workspace, false));
  if (c.seg.seg_len > 0) {
    c.grid[0] = cus;
    return c;
  }
  c.grid[0] = pairs;
  if (!with_workspace || !pl.waits() || (pl.helpers > 0 && !helpers_pay(pl, ((long long)NC + cgs - 1) / cgs))) return c;
  c.n = 0;
  if (pl.first_waiting() > 0) c.grid[c.n++] = pl.n_single;
  c.kernel[c.n] = pl.kernel(backward, NC);
  c.grid[c.n++] = pl.grid(backward);
  return c;
}
// Workspace of the backward with several workgroups per pair, for n (batch, head) pairs of K groups: the synchronisation
// words, the replay's shares of the norm gradients (one sum per set + a running sum), a parked image, what a walk on two
// CUs exchanges, what the walk hands to the grad_L_XK workgroup (one image, dZ1, and two fp32 tiles, g_y and the norm-weight
// gradient terms, per slot, two sets), what fewer of those than pairs park between two groups, then the sets of per-group tensors beyond the caller's; each part 256-byte aligned.
static_assert(ttt::BWQ_XCHG_WORDS <= ttt::BWW_XCHG_WORDS + 2 * (TTT_MLP_CS * TTT_MLP_HID * 2 + 4 * TTT_MLP_CS * TTT_MLP_F * 2) / 8, "exchange of four CUs");
struct BwdWorkspace {
  static constexpr int PER_SET = 11;
  static constexpr int ALT_SETS = ttt::BWD_MAX_SETS - 1;
  static constexpr int FIRST_SET = 8;
  static constexpr int PARTS = FIRST_SET + PER_SET * ALT_SETS;
  size_t off[PARTS];
  size_t total;
  int alt_sets;
  BwdWorkspace(const LaunchPlan& pl, long long cgs, long long K) {
    const long long n = pl.n_waiting();
    alt_sets = bwd_sets_used(pl, K) - 1;
    const size_t slot = (size_t)n * (size_t)cgs;
    const size_t tile = TTT_MLP_CS * TTT_MLP_F * 2, img = TTT_MLP_CS * TTT_MLP_HID * 2, vec = TTT_MLP_CS * 4;
    const size_t norm = (size_t)n * 8 * 2 * TTT_MLP_F * sizeof(float);
    // per set: X2, Z1, Z1_bar, X2_bar (images), gZ2 (tile), gZ1 (image), x_hat_fused, g_x_hat_fused, g_out_fused
    // (tiles), std_fused, W1_init (two images per slot: GELU' and GELU'', which helpers leave to the walk: 200 pairs in groups
    // of 64 without it 4.7 instead of 6.3 GiB)
    const size_t per_set[PER_SET] = {slot * img, slot * img, slot * img, slot * img, slot * tile, slot * img,
                                     slot * tile, slot * tile, slot * tile, slot * vec, pl.helpers > 0 ? 0 : slot * 2 * img};
    size_t o = 0;
    auto put = [&](int i, size_t bytes) { off[i] = o; o += (bytes + 255) & ~(size_t)255; };
    put(0, ttt::bwd_sync_ints(n) * sizeof(int));
    put(1, ttt::BWD_MAX_SETS * 8 * norm);
    put(2, norm);
    put(3, (size_t)n * img);
    put(4, pl.wide ? (size_t)n * ttt::BWW_XCHG_WORDS * 8 : 0);   // (a walk on four CUs exchanges through this and the next two, which it has no other use for)
    put(5, pl.gang ? 2 * slot * img : 0);
    put(6, pl.gang ? 2 * slot * 4 * tile : 0);
    put(7, !pl.quad && pl.n_finish < pl.gang ? (size_t)n * ttt::FIN_PARK_FLOATS * sizeof(float) : 0);
    for (int s = 0; s < ALT_SETS; s++)
      for (int t = 0; t < PER_SET; t++) put(FIRST_SET + PER_SET * s + t, s < alt_sets ? per_set[t] : 0);
    total = o;
  }
};

// Workspace of the forward with several workgroups per pair: synchronisation words, then per (batch, head) a ring of
// 2 * FWD_RING_MAX slots of state images and of bias vectors.
// With the recurrence on two workgroups the ring has FWD_WIDE_RING slots, and the exchange follows.
struct FwdWorkspace {
  size_t off[4];
  size_t total;
  explicit FwdWorkspace(const LaunchPlan& pl) {
    const long long n = pl.n_rest;
    const size_t slots = (size_t)n * (pl.quad ? 0 : pl.wide ? ttt::FWD_WIDE_RING : 2 * ttt::FWD_RING_MAX);
    const size_t bytes[4] = {ttt::bwd_sync_ints(n) * sizeof(int), slots * ttt::FWD_IMG_BYTES,
                             slots * ttt::FWD_BIAS_FLOATS * sizeof(float),
                             pl.wide ? (size_t)n * (pl.quad ? ttt::FWD_QUAD_XCHG_WORDS : ttt::FWD_XCHG_WORDS) * 8 : 0};
    size_t o = 0;
    for (int i = 0; i < 4; i++) { off[i] = o; o += (bytes[i] + 255) & ~(size_t)255; }
    total = o;
  }
};

int check_workspace(const void* workspace) {
  if (workspace == nullptr) return TTT_MLP_ERR_BAD_ARG;
  if ((reinterpret_cast<uintptr_t>(workspace) & 255u) != 0) return TTT_MLP_ERR_ALIGN;
  return TTT_MLP_OK;
}

}  // namespace

extern "C" int ttt_mlp_bwd_launch(const ttt_mlp_bwd_args* a, void* stream) {
  ttt::BwdParams p;
  if (int rc = make_bwd_params(a, p)) return rc;
  const int cus = device_cus();
  const Call call = plan_call(true, LaunchPlan{}, (long long)p.B * p.NH, cus, p.NC, p.cgs, false);
  if (call.seg.seg_len > 0) return launch_bwd_segments(p, call.seg, cus, static_cast<hipStream_t>(stream));
  p.bh0 = 0;
  p.nbh = p.B * p.NH;
  return static_cast<int>(ttt_mlp_bwd_enqueue(p, call.kernel[0], static_cast<int>(call.grid[0]), static_cast<hipStream_t>(stream)));
}

extern "C" int ttt_mlp_bwd_export_group0(const ttt_mlp_bwd_args* a, void* stream) {
  ttt::BwdParams p;
  if (int rc = make_bwd_params(a, p)) return rc;
  p.bh0 = 0;
  p.nbh = p.B * p.NH;
  return static_cast<int>(ttt_mlp_export_group0_enqueue(p, static_cast<hipStream_t>(stream)));
}

extern "C" size_t ttt_mlp_bwd_workspace_bytes(int B, int NH, int checkpoint_group_size) {
  if (B <= 0 || NH <= 0 || checkpoint_group_size <= 0 || checkpoint_group_size > (1 << 16)) return 0;
  const LaunchPlan pl = plan_launches((long long)B * NH, true);
  return pl.waits() ? BwdWorkspace(pl, checkpoint_group_size, ttt::BWD_MAX_SETS).total : 0;
}

namespace {
void bwd_range(const LaunchPlan& pl, long long cgs, long long K, size_t* least, size_t* most) {
  *least = *most = 0;
  if (!pl.waits() || (pl.helpers > 0 && !helpers_pay(pl, K))) return;
  *least = BwdWorkspace(bwd_reduced(pl), cgs, K).total;
  *most = BwdWorkspace(pl, cgs, K).total;
}
}  // namespace

extern "C" int ttt_mlp_bwd_workspace_range(int B, int NH, int checkpoint_group_size, int K, size_t* least, size_t* most) {
  if (least == nullptr || most == nullptr || B <= 0 || NH <= 0 || checkpoint_group_size <= 0 || checkpoint_group_size > (1 << 16) || K <= 0)
    return TTT_MLP_ERR_BAD_ARG;
  bwd_range(plan_launches((long long)B * NH, true), checkpoint_group_size, K, least, most);
  return TTT_MLP_OK;
}

extern "C" int ttt_mlp_bwd_workspace_for(int B, int NH, int checkpoint_group_size, int NC, size_t* least, size_t* most) {
  if (least == nullptr || most == nullptr || B <= 0 || NH <= 0 || checkpoint_group_size <= 0 || checkpoint_group_size > (1 << 16) || NC <= 0)
    return TTT_MLP_ERR_BAD_ARG;
  bwd_range(plan_bwd((long long)B * NH, device_cus(), checkpoint_group_size, NC), checkpoint_group_size,
            ((long long)NC + checkpoint_group_size - 1) / checkpoint_group_size, least, most);
  return TTT_MLP_OK;
}

extern "C" size_t ttt_mlp_bwd_status_offset(int B, int NH) {
  if (B <= 0 || NH <= 0) return 0;
  const LaunchPlan pl = plan_launches((long long)B * NH, true);
  return pl.waits() ? (size_t)pl.n_waiting() * ttt::BWD_SYNC_STRIDE * sizeof(int) : 0;
}

extern "C" int ttt_mlp_bwd_launch_overlapped(const ttt_mlp_bwd_args* a, void* workspace, size_t workspace_bytes, void* stream) {
  ttt::BwdParams p;
  if (int rc = make_bwd_params(a, p)) return rc;
  if (int rc = check_workspace(workspace)) return rc;
  const LaunchPlan pl = plan_launches((long long)p.B * p.NH, true);
  if (!pl.waits()) return TTT_MLP_ERR_NO_ROOM;
  if (workspace_bytes < BwdWorkspace(pl, p.cgs, ttt::BWD_MAX_SETS).total) return TTT_MLP_ERR_WORKSPACE;
  return ttt_mlp_bwd_launch_within(a, workspace, workspace_bytes, stream);
}

namespace {
int bwd_launch(const ttt_mlp_bwd_args* a, void* workspace, size_t workspace_bytes, void* stream, bool scatter, int* report) {
  ttt::BwdParams p;
  if (int rc = make_bwd_params(a, p)) return rc;
  if (int rc = check_workspace(workspace)) return rc;
  const int cus = device_cus();
  LaunchPlan pl = plan_bwd((long long)p.B * p.NH, cus, p.cgs, p.NC);
  if (!pl.waits()) return TTT_MLP_ERR_NO_ROOM;
  if (workspace_bytes < BwdWorkspace(pl, p.cgs, p.K).total) pl = bwd_reduced(pl);
  const BwdWorkspace w(pl, p.cgs, p.K);
  if (workspace_bytes < w.total) return TTT_MLP_ERR_WORKSPACE;
  char* base = static_cast<char*>(workspace);
  const Call call = plan_call(true, pl, (long long)p.B * p.NH, cus, p.NC, p.cgs, true);
  const TttKernel kernel = call.kernel[call.n - 1];
  const int grid = static_cast<int>(call.grid[call.n - 1]);
  // cut sequences where they beat a last round on several workgroups per pair (see the forward)
  if (kernel == BWD_ONE) {
    if (hipError_t e = ttt_mlp_fwd_clear_words(reinterpret_cast<int*>(base + w.off[0]), static_cast<int>(ttt::bwd_sync_ints(pl.n_waiting())),
                                               static_cast<hipStream_t>(stream)))
      return static_cast<int>(e);
    if (call.seg.seg_len > 0) return launch_bwd_segments(p, call.seg, cus, static_cast<hipStream_t>(stream));
    p.bh0 = 0;
    p.nbh = p.B * p.NH;
    return static_cast<int>(ttt_mlp_bwd_enqueue(p, kernel, grid, static_cast<hipStream_t>(stream)));
  }
  if (call.n > 1) {
    p.bh0 = 0;
    p.nbh = static_cast<int>(pl.n_single);
    if (hipError_t e = ttt_mlp_bwd_enqueue(p, call.kernel[0], p.nbh, static_cast<hipStream_t>(stream))) return static_cast<int>(e);
  }
  // The kernels index the workspace by the global pair number: every pointer is moved back by bh0 entries.
  const size_t b0 = (size_t)pl.first_waiting();
  const size_t tile = (size_t)p.cgs * TTT_MLP_CS * TTT_MLP_F, img = (size_t)p.cgs * TTT_MLP_CS * TTT_MLP_HID, vec = (size_t)p.cgs * TTT_MLP_CS;
  const size_t norm = 8 * 2 * TTT_MLP_F;
  p.bh0 = static_cast<int>(pl.first_waiting());
  p.nbh = static_cast<int>(pl.n_waiting());
  p.n_helpers = pl.helpers;
  p.gang_pairs = pl.gang;
  p.n_replay = pl.n_replay;
  p.n_sets = pl.helpers > 0 ? w.alt_sets + 1 : pl.sets;
  p.n_shared = pl.shared;
  p.n_parts = pl.parts;
  for (int i = 0; i <= ttt::BWD_MAX_PARTS; i++) p.part_start[i] = PART_START[pl.parts - 1][i];
  p.n_finish = pl.n_finish;
  p.wide = pl.wide ? 1 : 0;
  p.wait_limit = g_wait_limit;
  p.report = report;
  if (pl.gang) {
    p.fin_dz = reinterpret_cast<__bf16*>(base + w.off[5]) - b0 * 2 * img;
    p.fin_gy = reinterpret_cast<float*>(base + w.off[6]) - b0 * 2 * 2 * tile;
    p.fin_park = reinterpret_cast<float*>(base + w.off[7]) - b0 * ttt::FIN_PARK_FLOATS;
  }
  int* words = reinterpret_cast<int*>(base + w.off[0]);
  p.status = words + (size_t)pl.n_waiting() * ttt::BWD_SYNC_STRIDE;
  p.sync = words - b0 * ttt::BWD_SYNC_STRIDE;
  p.norm_partial = reinterpret_cast<float*>(base + w.off[1]) - b0 * ttt::BWD_MAX_SETS * 8 * norm;
  p.norm_park = reinterpret_cast<float*>(base + w.off[2]) - b0 * norm;
  p.walk_park = reinterpret_cast<__bf16*>(base + w.off[3]) - b0 * (TTT_MLP_CS * TTT_MLP_HID);
  // (sets that a sequence this short does not come to: the walk asks for operands of the group behind its last one and drops
  // them, so their pointers are the caller's own tensors)
  for (int s = w.alt_sets; s < ttt::BWD_MAX_SETS - 1; s++) {
    p.alt_X2_group[s] = p.X2_group; p.alt_Z1_group[s] = p.Z1_group;
    p.alt_Z1_bar_group[s] = p.Z1_bar_group; p.alt_X2_bar_group[s] = p.X2_bar_group;
    p.alt_grad_l_wrt_Z2_group[s] = p.grad_l_wrt_Z2_group; p.alt_grad_l_wrt_Z1_group[s] = p.grad_l_wrt_Z1_group;
    p.alt_x_hat_fused_group[s] = p.x_hat_fused_group; p.alt_grad_x_hat_fused_group[s] = p.grad_x_hat_fused_group;
    p.alt_grad_output_fused_group[s] = p.grad_output_fused_group; p.alt_std_fused_group[s] = p.std_fused_group;
    p.alt_W1_init_group[s] = p.W1_init_group;
  }
  for (int s = 0; s < w.alt_sets; s++) {
    const size_t* o = w.off + BwdWorkspace::FIRST_SET + BwdWorkspace::PER_SET * s;
    p.alt_X2_group[s] = reinterpret_cast<__bf16*>(base + o[0]) - b0 * img;
    p.alt_Z1_group[s] = reinterpret_cast<__bf16*>(base + o[1]) - b0 * img;
    p.alt_Z1_bar_group[s] = reinterpret_cast<__bf16*>(base + o[2]) - b0 * img;
    p.alt_X2_bar_group[s] = reinterpret_cast<__bf16*>(base + o[3]) - b0 * img;
    p.alt_grad_l_wrt_Z2_group[s] = reinterpret_cast<__bf16*>(base + o[4]) - b0 * tile;
    p.alt_grad_l_wrt_Z1_group[s] = reinterpret_cast<__bf16*>(base + o[5]) - b0 * img;
    p.alt_x_hat_fused_group[s] = reinterpret_cast<__bf16*>(base + o[6]) - b0 * tile;
    p.alt_grad_x_hat_fused_group[s] = reinterpret_cast<__bf16*>(base + o[7]) - b0 * tile;
    p.alt_grad_output_fused_group[s] = reinterpret_cast<__bf16*>(base + o[8]) - b0 * tile;
    p.alt_std_fused_group[s] = reinterpret_cast<float*>(base + o[9]) - b0 * vec;
    // [cgs][64][256] floats = 2 images per slot; not in the sets of helpers, and not touched by them
    p.alt_W1_init_group[s] = pl.helpers > 0 ? p.W1_init_group : reinterpret_cast<float*>(base + o[10]) - b0 * img;
  }
  if (pl.helpers > 0) {
    p.help_sets[0] = {p.X2_group, p.Z1_group, p.Z1_bar_group, p.X2_bar_group, p.grad_l_wrt_Z2_group, p.grad_l_wrt_Z1_group,
                      p.x_hat_fused_group, p.grad_x_hat_fused_group, p.grad_output_fused_group, p.std_fused_group, p.W1_init_group};
    for (int s = 0; s < ttt::BWD_HELP_SETS - 1; s++)
      p.help_sets[s + 1] = {p.alt_X2_group[s], p.alt_Z1_group[s], p.alt_Z1_bar_group[s], p.alt_X2_bar_group[s], p.alt_grad_l_wrt_Z2_group[s],
                            p.alt_grad_l_wrt_Z1_group[s], p.alt_x_hat_fused_group[s], p.alt_grad_x_hat_fused_group[s],
                            p.alt_grad_output_fused_group[s], p.alt_std_fused_group[s], p.alt_W1_init_group[s]};
  }
  if (pl.gang) {
    p.xchg = reinterpret_cast<unsigned long long*>(base + w.off[4]) - b0 * (pl.quad ? ttt::BWQ_XCHG_WORDS : ttt::BWW_XCHG_WORDS);
    p.scatter = scatter ? 1 : 0;
    return static_cast<int>(ttt_mlp_bwd_gang_enqueue(p, kernel, grid, static_cast<hipStream_t>(stream)));
  }
  return static_cast<int>(ttt_mlp_bwd_enqueue(p, kernel, grid, static_cast<hipStream_t>(stream)));
}
}  // namespace

extern "C" int ttt_mlp_bwd_launch_within(const ttt_mlp_bwd_args* a, void* workspace, size_t workspace_bytes, void* stream) {
  return bwd_launch(a, workspace, workspace_bytes, stream, false, nullptr);
}

extern "C" int ttt_mlp_fwd_launch(const ttt_mlp_fwd_args* a, void* stream) {
  ttt::FwdParams p;
  if (int rc = make_fwd_params(a, p)) return rc;
  const int cus = device_cus();
  const Call call = plan_call(false, LaunchPlan{}, (long long)p.B * p.NH, cus, p.NC, p.cgs, false);
  if (call.seg.seg_len > 0) return launch_fwd_segments(p, call.seg, cus, static_cast<hipStream_t>(stream));
  p.bh0 = 0;
  p.nbh = p.B * p.NH;
  return static_cast<int>(ttt_mlp_fwd_enqueue(p, call.kernel[0], static_cast<int>(call.grid[0]), static_cast<hipStream_t>(stream)));
}

extern "C" size_t ttt_mlp_fwd_workspace_bytes(int B, int NH) {
  if (B <= 0 || NH <= 0) return 0;
  const LaunchPlan pl = plan_launches((long long)B * NH, false);
  return pl.rest_split ? FwdWorkspace(pl).total : 0;
}

extern "C" size_t ttt_mlp_fwd_status_offset(int B, int NH) {
  if (B <= 0 || NH <= 0) return 0;
  const LaunchPlan pl = plan_launches((long long)B * NH, false);
  return pl.rest_split ? (size_t)pl.n_rest * ttt::BWD_SYNC_STRIDE * sizeof(int) : 0;
}

namespace {
int fwd_launch(const ttt_mlp_fwd_args* a, void* workspace, size_t workspace_bytes, void* stream, bool scatter, int* report) {
  ttt::FwdParams p;
  if (int rc = make_fwd_params(a, p)) return rc;
  if (int rc = check_workspace(workspace)) return rc;
  const int cus = device_cus();
  const LaunchPlan pl = plan_for((long long)p.B * p.NH, cus, false);
  if (!pl.rest_split) return TTT_MLP_ERR_NO_ROOM;
  const FwdWorkspace w(pl);
  if (workspace_bytes < w.total) return TTT_MLP_ERR_WORKSPACE;
  char* base = static_cast<char*>(workspace);
  const Call call = plan_call(false, pl, (long long)p.B * p.NH, cus, p.NC, p.cgs, true);
  const TttKernel kernel = call.kernel[call.n - 1];
  const int grid = static_cast<int>(call.grid[call.n - 1]);
  if (call.seg.seg_len > 0) {
    // cut sequences beat a last round on two workgroups per pair where there are full rounds before it: the
    // workspace then only has its words cleared (callers read the status word behind them)
    if (hipError_t e = ttt_mlp_fwd_clear_words(reinterpret_cast<int*>(base + w.off[0]), static_cast<int>(ttt::bwd_sync_ints(pl.n_rest)),
                                               static_cast<hipStream_t>(stream)))
      return static_cast<int>(e);
    return launch_fwd_segments(p, call.seg, cus, static_cast<hipStream_t>(stream));
  }
  if (call.n > 1) {
    p.bh0 = 0;
    p.nbh = static_cast<int>(pl.n_single);
    if (hipError_t e = ttt_mlp_fwd_enqueue(p, call.kernel[0], p.nbh, static_cast<hipStream_t>(stream))) return static_cast<int>(e);
  }
  const size_t b0 = (size_t)pl.n_single;
  p.bh0 = static_cast<int>(pl.n_single);
  p.nbh = static_cast<int>(pl.n_rest);
  int* words = reinterpret_cast<int*>(base + w.off[0]);
  p.status = words + (size_t)pl.n_rest * ttt::BWD_SYNC_STRIDE;
  p.sync = words - b0 * ttt::BWD_SYNC_STRIDE;
  p.wait_limit = g_wait_limit;
  p.report = report;
  if (pl.wide) {
    p.quad = pl.quad ? 1 : 0;
    p.state_img = reinterpret_cast<__bf16*>(base + w.off[1]) - b0 * ttt::FWD_WIDE_RING * (ttt::FWD_IMG_BYTES / 2);
    p.bias_img = reinterpret_cast<float*>(base + w.off[2]) - b0 * ttt::FWD_WIDE_RING * ttt::FWD_BIAS_FLOATS;
    p.xchg = reinterpret_cast<unsigned long long*>(base + w.off[3]) - b0 * (pl.quad ? ttt::FWD_QUAD_XCHG_WORDS : ttt::FWD_XCHG_WORDS);
    p.scatter = scatter ? 1 : 0;
    return static_cast<int>(ttt_mlp_fwd_wide_enqueue(p, kernel, grid, static_cast<hipStream_t>(stream)));
  }
  p.ring_log2 = kernel == FWD_SPLIT_32 ? 5 : 3;
  p.state_img = reinterpret_cast<__bf16*>(base + w.off[1]) - b0 * 2 * ttt::FWD_RING_MAX * (ttt::FWD_IMG_BYTES / 2);
  p.bias_img = reinterpret_cast<float*>(base + w.off[2]) - b0 * 2 * ttt::FWD_RING_MAX * ttt::FWD_BIAS_FLOATS;
  return static_cast<int>(ttt_mlp_fwd_enqueue(p, kernel, grid, static_cast<hipStream_t>(stream)));
}
}  // namespace

extern "C" int ttt_mlp_fwd_launch_overlapped(const ttt_mlp_fwd_args* a, void* workspace, size_t workspace_bytes, void* stream) {
  return fwd_launch(a, workspace, workspace_bytes, stream, false, nullptr);
}

extern "C" int ttt_mlp_launch_reporting(int which, const void* args, void* workspace, size_t workspace_bytes, int* report, void* stream) {
  if (which == 0) return fwd_launch(static_cast<const ttt_mlp_fwd_args*>(args), workspace, workspace_bytes, stream, false, report);
  if (which == 1) return bwd_launch(static_cast<const ttt_mlp_bwd_args*>(args), workspace, workspace_bytes, stream, false, report);
  return TTT_MLP_ERR_BAD_ARG;
}

extern "C" int ttt_mlp_launch_scattered(int which, const void* args, void* workspace, size_t workspace_bytes, void* stream) {
  if (which == 0) return fwd_launch(static_cast<const ttt_mlp_fwd_args*>(args), workspace, workspace_bytes, stream, true, nullptr);
  if (which == 1) return bwd_launch(static_cast<const ttt_mlp_bwd_args*>(args), workspace, workspace_bytes, stream, true, nullptr);
  return TTT_MLP_ERR_BAD_ARG;
}

// ---------------------------------------------------------------------------------------------------------
// The two-workgroup forward for callers that cannot allocate and have no workspace to bring: its workspace
// is this fixed array (one copy per GPU, held until the process ends).  Host code never passes the array's
// name to a kernel - the name is a host-side stand-in, not a device address; the address on each device
// comes from hipGetSymbolAddress, once per device.
namespace {
constexpr int STATIC_MAX_PAIRS = 8;
constexpr size_t static_scratch_bytes() {
  // FwdWorkspace(STATIC_MAX_PAIRS): synchronisation words, state images, bias vectors; each part 256-byte aligned
  const size_t slots = (size_t)STATIC_MAX_PAIRS * 2 * ttt::FWD_RING_MAX;
  const size_t a = ((STATIC_MAX_PAIRS * ttt::BWD_SYNC_STRIDE + 32) * sizeof(int) + 255) & ~(size_t)255;
  const size_t b = (slots * ttt::FWD_IMG_BYTES + 255) & ~(size_t)255;
  const size_t c = (slots * ttt::FWD_BIAS_FLOATS * sizeof(float) + 255) & ~(size_t)255;
  return a + b + c;
}
static __device__ __align__(256) unsigned char scratch[static_scratch_bytes()];   // 32.6 MiB

constexpr int MAX_DEVICES = 64;
// address of `scratch` on each device, looked up at the first call there; host threads may race to the first
// call - every one of them finds the same address, so an atomic slot per device is all the guard it needs
std::atomic<void*> g_scratch_ptr[MAX_DEVICES] = {};

// The current device's copy of the array (the device that the launch goes to).  Looked up once per device.
int static_scratch(void** ptr) {
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev)) return static_cast<int>(e);
  if (dev < 0 || dev >= MAX_DEVICES) return TTT_MLP_ERR_BAD_ARG;
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    if (hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch))) return static_cast<int>(e);
    if (p == nullptr) return TTT_MLP_ERR_BAD_ARG;
    g_scratch_ptr[dev].store(p, std::memory_order_release);
  }
  *ptr = p;
  return TTT_MLP_OK;
}

__global__ void ttt_mlp_or_status(const int* status, int* sticky) {
  if (*status != 0) *sticky = 1;
}
}  // namespace

extern "C" int ttt_mlp_status_accumulate(const void* status_word, int* sticky_word, void* stream) {
  if (status_word == nullptr || sticky_word == nullptr) return TTT_MLP_ERR_BAD_ARG;
  hipLaunchKernelGGL(ttt_mlp_or_status, dim3(1), dim3(1), 0, static_cast<hipStream_t>(stream),
                     static_cast<const int*>(status_word), sticky_word);
  return static_cast<int>(hipGetLastError());
}

extern "C" int ttt_mlp_fwd_launch_static(const ttt_mlp_fwd_args* a, int* sticky_word, void* stream) {
  ttt::FwdParams p;
  if (int rc = make_fwd_params(a, p)) return rc;
  const long long pairs = (long long)p.B * p.NH;
  if (pairs > STATIC_MAX_PAIRS) return TTT_MLP_ERR_SCRATCH;
  const LaunchPlan pl = plan_launches(pairs, false);
  if (!pl.rest_split || pl.n_single != 0) return TTT_MLP_ERR_NO_ROOM;
  const FwdWorkspace w(pl);
  static_assert(static_scratch_bytes() % 256 == 0, "scratch parts are 256-byte aligned");
  if (w.total > static_scratch_bytes()) return TTT_MLP_ERR_SCRATCH;
  void* ws = nullptr;
  if (int rc = static_scratch(&ws)) return rc;
  // From here on as ttt_mlp_fwd_launch_overlapped with `ws` as the workspace: the launch clears the
  // synchronisation words and the status word itself (a small kernel ahead of the main one), everything
  // else in the workspace is written before it is read.
  if (int rc = ttt_mlp_fwd_launch_overlapped(a, ws, static_scratch_bytes(), stream)) return rc;
  if (sticky_word != nullptr) {
    const int* status = reinterpret_cast<const int*>(static_cast<const char*>(ws) + w.off[0]) + (size_t)pl.n_rest * ttt::BWD_SYNC_STRIDE;
    return ttt_mlp_status_accumulate(status, sticky_word, stream);
  }
  return TTT_MLP_OK;
}

extern "C" int ttt_mlp_launch_plan(int which, long long pairs, int compute_units, long long* one_workgroup_pairs,
                                   long long* other_pairs, int* workgroups_per_other_pair) {
  if (one_workgroup_pairs == nullptr || other_pairs == nullptr || workgroups_per_other_pair == nullptr || (which != 0 && which != 1))
    return TTT_MLP_ERR_BAD_ARG;
  const LaunchPlan pl = plan_for(pairs, compute_units, which == 1);
  *one_workgroup_pairs = pl.n_single;
  *other_pairs = pl.n_rest;
  *workgroups_per_other_pair = pl.per_pair(which == 1);
  return TTT_MLP_OK;
}

extern "C" int ttt_mlp_segment_plan(int which, long long pairs, int compute_units, int NC, int checkpoint_group_size, int with_workspace,
                                    int* segment_minibatches, int* launches) {
  if (compute_units == 0) compute_units = device_cus();   // the current device's, or the budget set for it
  if (segment_minibatches == nullptr || launches == nullptr || pairs <= 0 || compute_units <= 0 || NC <= 0 ||
      checkpoint_group_size <= 0 || (which != 0 && which != 1))
    return TTT_MLP_ERR_BAD_ARG;
  *segment_minibatches = 0;
  *launches = 1;
  if (pairs <= compute_units) return TTT_MLP_OK;   // (asked ahead of every call of the operators)
  const LaunchPlan pl = which == 1 ? plan_bwd(pairs, compute_units, checkpoint_group_size, NC)
                                   : plan_for(pairs, compute_units, false);
  const Call call = plan_call(which == 1, pl, pairs, compute_units, NC, checkpoint_group_size, with_workspace != 0);
  *segment_minibatches = call.seg.seg_len;
  *launches = call.seg.seg_len > 0 ? call.seg.launches : call.n;
  return TTT_MLP_OK;
}

extern "C" const char* ttt_mlp_launched_kernel(int which, long long pairs, int compute_units, int NC, int checkpoint_group_size, int with_workspace,
                                               int index, long long* workgroups, int* dispatches, int* resident) {
  if (pairs <= 0 || compute_units <= 0 || NC <= 0 || checkpoint_group_size <= 0 || (which != 0 && which != 1) || index < 0) return nullptr;
  const LaunchPlan pl = which == 1 ? plan_bwd(pairs, compute_units, checkpoint_group_size, NC)
                                   : plan_for(pairs, compute_units, false);
  const Call call = plan_call(which == 1, pl, pairs, compute_units, NC, checkpoint_group_size, with_workspace != 0);
  if (index >= call.n) return nullptr;
  const TttKernel kernel = call.kernel[index];
  if (workgroups != nullptr) *workgroups = call.grid[index];
  if (dispatches != nullptr) *dispatches = call.seg.seg_len > 0 ? call.seg.launches : 1;
  if (resident != nullptr) *resident = kernel != FWD_ONE && kernel != BWD_ONE && kernel != BWD_HELPED;
  switch (kernel) {
#define TTT_KERNEL_NAME(number, ...) case number: return #__VA_ARGS__;
    TTT_FWD_KERNELS(TTT_KERNEL_NAME) TTT_FWD_WIDE_KERNELS(TTT_KERNEL_NAME) TTT_BWD_KERNELS(TTT_KERNEL_NAME) TTT_BWD_GANG_KERNELS(TTT_KERNEL_NAME)
#undef TTT_KERNEL_NAME
  }
  return nullptr;
}

extern "C" int ttt_mlp_kernel_info(int which, int* lds_bytes, int* threads_per_workgroup) {
  if (lds_bytes == nullptr || threads_per_workgroup == nullptr) return TTT_MLP_ERR_BAD_ARG;
  if (which == 0) { *lds_bytes = ttt_mlp_fwd_lds_bytes(); *threads_per_workgroup = ttt_mlp_fwd_threads(); return TTT_MLP_OK; }
  if (which == 1) { *lds_bytes = ttt_mlp_bwd_lds_bytes(); *threads_per_workgroup = ttt_mlp_bwd_threads(); return TTT_MLP_OK; }
  return TTT_MLP_ERR_BAD_ARG;
}
