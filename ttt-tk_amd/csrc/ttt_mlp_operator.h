/* Entry points of libttt_mlp.so for the operator module in this folder and for the tests; not part of the C ABI in
 * include/ttt_mlp.h.  The first four let the operator take a workspace that fits the call at hand instead of one that fits
 * every call of its B, NH and checkpoint_group_size, and learn without a copy whether a wait gave up. */
#ifndef TTT_MLP_OPERATOR_H_
#define TTT_MLP_OPERATOR_H_

#include "../../include/ttt_mlp.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Workspace of the backward over a sequence of K checkpoint groups.  ttt_mlp_bwd_workspace_bytes() serves every length, with a set of
 * per-group tensors for each group that may be under way at once; a short sequence has fewer groups than that.  *most: the
 * launch of the plan; *least: the launch with the fewest sets (two workgroups that recompute instead of three or four;
 * the same as *most where the plan has no more than two).  Both 0 when the mode does not apply.  _for: over one of NC mini-batches, whose launch may
 * be one that takes less. */
int ttt_mlp_bwd_workspace_range(int32_t B, int32_t NH, int32_t checkpoint_group_size, int32_t K, size_t* least, size_t* most);
int ttt_mlp_bwd_workspace_for(int32_t B, int32_t NH, int32_t checkpoint_group_size, int32_t NC, size_t* least, size_t* most);

/* As ttt_mlp_bwd_launch_overlapped, with any workspace of at least *least bytes (ttt_mlp_bwd_workspace_range, _for): the launch
 * of the plan from *most bytes on, the one with fewer sets below.  Same results, bit for bit. */
int ttt_mlp_bwd_launch_within(const ttt_mlp_bwd_args* args, void* workspace, size_t workspace_bytes, void* stream);

/* ttt_mlp_fwd_launch_overlapped (which = 0, args a ttt_mlp_fwd_args) / ttt_mlp_bwd_launch_within (1) whose workgroups, if a wait
 * gives up, also set *report, an int that the device can write and the host reads once the stream has been waited for (host
 * memory; not written otherwise; nullptr: none). */
int ttt_mlp_launch_reporting(int which, const void* args, void* workspace, size_t workspace_bytes, int* report, void* stream);

/* ttt_mlp_fwd_launch_overlapped (which = 0, args a ttt_mlp_fwd_args) / ttt_mlp_bwd_launch_overlapped (1) with the workgroups
 * of a pair on consecutive XCDs where the recurrence or the walk takes two: what they do if a device does not place them on
 * one.  For tests: same results, slower. */
int ttt_mlp_launch_scattered(int which, const void* args, void* workspace, size_t workspace_bytes, void* stream);

/* The kernels that a forward (which = 0) or backward (1) of this shape enqueues on a device with `compute_units` CUs, in order and
 * without the small ones that clear words: the name of number `index` as a trace has it, NULL from the first one on that there is not.  *workgroups:
 * the most of one dispatch; *dispatches: how many of it in a row (more than one: sequences cut at checkpoints); *resident: 1 if its workgroups
 * wait for others that may not have started, so that all of them have to fit the device at once.  with_workspace as in ttt_mlp_segment_plan, 1: of
 * the size that ttt_mlp_*_workspace_bytes() say.  Any of the pointers may be NULL.  No device needed. */
const char* ttt_mlp_launched_kernel(int which, long long pairs, int compute_units, int NC, int checkpoint_group_size, int with_workspace,
                                    int index, long long* workgroups, int* dispatches, int* resident);

#ifdef __cplusplus
}
#endif
#endif /* TTT_MLP_OPERATOR_H_ */
