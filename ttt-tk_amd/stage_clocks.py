#!/usr/bin/env python3
"""Per-stage clock budget of one forward and one backward mini-batch of the TTT-MLP kernels.

    python ttt-tk_amd/build.py --stages                       # once, no GPU needed: libttt_mlp_stages.so
    python ttt-tk_amd/stage_clocks.py --workload c4 [--out profiles/ttt_mlp_c4_stage_clocks.txt]

Loads the library built with -DTTT_STAGE_CLOCKS (the product library contains no clocks), runs the forward and the
backward of the workload once each the way the operator module would (same launch plan, workspace from torch), and
prints for every kind of workgroup - forward: recurrence / output branch; backward: replay / reverse walk / grad_L_XK
workgroup - the clocks per mini-batch that its waves spent in each stage, averaged over the (batch, head) pairs: the mean
over the 8 waves and the slowest wave.  Where the recurrence or the walk runs on two workgroups, their compute waves and
their helper waves go through stages of their own and get a table each.  The stage names and their descriptions are read
from the enums in csrc/ttt_mlp_kernels.hpp.  --shape B,NH,NC,CGS takes another shape than the benchmark's.  Reading the clock is a scalar-memory operation that also waits for the wave's
outstanding LDS reads, so an instrumented kernel runs some 10 % slower than the product kernel; the launch times of
both are printed side by side.
"""
from __future__ import annotations

import argparse
import ctypes
import os
import re
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
SLOTS = 24
ROLES = 8     # of a workgroup: csrc/ttt_mlp_kernels.hpp
OUT, HALF, WALK, DXK, WALK_HALF = 1, 3, 4, 5, 6
WAVES = 8
WORKLOADS = {   # B, NH, NC, checkpoint_group_size, std of the eta logits
    "c3": (1, 48, 256, 16, 1.0),
    "c4": (1, 48, 4096, 64, 1.0),
    "c5": (8, 48, 512, 32, 2.0),
}


def stage_names(header_text: str, enum: str):
    """[(name, description)] of `enum` in the kernels' header, in order, without the closing *_COUNT."""
    body = re.search(r"enum\s+" + enum + r"\s*\{(.*?)\};", header_text, re.S).group(1)
    out = []
    for line in body.splitlines():
        m = re.match(r"\s*(\w+)\s*,?\s*(?://\s*(.*))?$", line)
        if m and m.group(1) and not m.group(1).endswith("_COUNT"):
            out.append((m.group(1), (m.group(2) or "").strip()))
    return out


PER_WAVE = False


def table(title, clocks, names, per_mb):
    """clocks: tensor [pairs][waves][SLOTS] of summed clocks; per_mb: mini-batches each wave went through."""
    mean_w = clocks.double().mean(dim=0) / per_mb          # [waves][SLOTS]
    tot = mean_w.sum(dim=1)                                # per wave
    lines = [f"{title}: {tot.mean().item():9.0f} clocks per mini-batch (mean over the waves; slowest wave {tot.max().item():.0f})"]
    for i, (name, desc) in enumerate(names):
        m, mx = mean_w[:, i].mean().item(), mean_w[:, i].max().item()
        if mx <= 0:
            continue
        if PER_WAVE:
            lines.append(f"  {name:18s} {m:8.0f}   wave by wave: " + " ".join(f"{x:6.0f}" for x in mean_w[:, i].tolist()))
        else:
            lines.append(f"  {name:18s} {m:8.0f} {100 * m / tot.mean().item():5.1f} %   slowest wave {mx:8.0f}   {desc}")
    return lines


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--workload", choices=sorted(WORKLOADS), default="c4")
    ap.add_argument("--shape", default=None, metavar="B,NH,NC,CGS", help="this shape instead of a named workload")
    ap.add_argument("--out", default=None, help="also write the tables to this file")
    ap.add_argument("--per-wave", action="store_true", help="every stage's clocks wave by wave instead of share and description")
    a = ap.parse_args()
    global PER_WAVE
    PER_WAVE = a.per_wave
    import torch
    sys.path.insert(0, ROOT)
    sys.path.insert(0, HERE)
    import ttt_mlp_host as host
    from bench import make_device_inputs
    from build import STAGES_LIB, LIB

    if not os.path.exists(STAGES_LIB) or os.path.getmtime(STAGES_LIB) < os.path.getmtime(LIB):
        raise SystemExit(f"{STAGES_LIB} is missing or older than the product library: run  python ttt-tk_amd/build.py --stages  first")
    header = open(os.path.join(HERE, "csrc", "ttt_mlp_kernels.hpp")).read()
    fwd_names, bwd_names = stage_names(header, "FwdStage"), stage_names(header, "BwdStage")
    fwd_wide_names, bwd_wide_names = stage_names(header, "FwdWideStage"), stage_names(header, "BwdWideStage")
    fwd_quad_names, bwd_quad_names = stage_names(header, "FwdQuadStage"), stage_names(header, "BwdQuadStage")
    if a.shape:
        B, NH, NC, cgs, eta_std = *(int(x) for x in a.shape.split(",")), 1.0
        label, option = "custom", f"--shape {a.shape}"
    else:
        B, NH, NC, cgs, eta_std = WORKLOADS[a.workload]
        label, option = a.workload, f"--workload {a.workload}"
    BH, K = B * NH, host.num_checkpoints(NC, cgs)
    dev = torch.device("cuda:0")
    t = make_device_inputs(B, NH, NC, eta_std, dev)
    t.update(host.alloc_forward_buffers(B, NH, NC, cgs, dev))
    t.update(host.alloc_backward_buffers(B, NH, NC, cgs, dev))

    class FwdArgs(ctypes.Structure):
        _fields_ = [(n, ctypes.c_void_p) for n in host.FWD_ORDER] + [(n, ctypes.c_int32) for n in ("cgs", "B", "NH", "NC", "K")]

    class BwdArgs(ctypes.Structure):
        _fields_ = [(n, ctypes.c_void_p) for n in host.BWD_ORDER] + [(n, ctypes.c_int32) for n in ("cgs", "B", "NH", "NC", "K", "overwrite")]

    fa = FwdArgs(*[t[k].data_ptr() for k in host.FWD_ORDER], cgs, B, NH, NC, K)
    ba = BwdArgs(*[t[k].data_ptr() for k in host.BWD_ORDER], cgs, B, NH, NC, K, 0)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def launches(lib):
        lib.ttt_mlp_fwd_workspace_bytes.restype = ctypes.c_size_t
        lib.ttt_mlp_bwd_workspace_bytes.restype = ctypes.c_size_t
        nf, nb = lib.ttt_mlp_fwd_workspace_bytes(B, NH), lib.ttt_mlp_bwd_workspace_bytes(B, NH, cgs)
        wf = torch.empty(max(nf, 1), dtype=torch.uint8, device=dev)
        wb = torch.empty(max(nb, 1), dtype=torch.uint8, device=dev)

        def fwd():
            if nf:
                return lib.ttt_mlp_fwd_launch_overlapped(ctypes.byref(fa), ctypes.c_void_p(wf.data_ptr()), ctypes.c_size_t(nf), stream)
            return lib.ttt_mlp_fwd_launch(ctypes.byref(fa), stream)

        def bwd():
            if nb:
                return lib.ttt_mlp_bwd_launch_overlapped(ctypes.byref(ba), ctypes.c_void_p(wb.data_ptr()), ctypes.c_size_t(nb), stream)
            return lib.ttt_mlp_bwd_launch(ctypes.byref(ba), stream)
        return fwd, bwd, (wf, wb)

    def timed(fn):
        rc = fn()   # warm-up
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        rc |= fn()
        e1.record()
        torch.cuda.synchronize()
        if rc:
            raise SystemExit(f"launch failed: code {rc}")
        return e0.elapsed_time(e1)

    plain = ctypes.CDLL(LIB)
    pf, pb, keep0 = launches(plain)
    plain_ms = (timed(pf), timed(pb))

    lib = ctypes.CDLL(STAGES_LIB)
    cf = torch.zeros(BH, ROLES, WAVES, SLOTS, dtype=torch.int32, device=dev)
    cb = torch.zeros(BH, ROLES, WAVES, SLOTS, dtype=torch.int32, device=dev)
    lib.ttt_mlp_set_stage_clocks.restype = None
    sf, sb, keep1 = launches(lib)
    lib.ttt_mlp_set_stage_clocks(ctypes.c_void_p(0), ctypes.c_void_p(0))
    sf(); sb()   # warm-up without clocks
    lib.ttt_mlp_set_stage_clocks(ctypes.c_void_p(cf.data_ptr()), ctypes.c_void_p(cb.data_ptr()))
    torch.cuda.synchronize()
    e0, e1, e2 = (torch.cuda.Event(enable_timing=True) for _ in range(3))
    e0.record(); rc = sf(); e1.record(); rc |= sb(); e2.record()
    torch.cuda.synchronize()
    if rc:
        raise SystemExit(f"launch failed: code {rc}")
    stage_ms = (e0.elapsed_time(e1), e1.elapsed_time(e2))
    cf, cb = cf.cpu().long() & 0xFFFFFFFF, cb.cpu().long() & 0xFFFFFFFF

    props = torch.cuda.get_device_properties(0)
    out = [f"Stage clocks of the TTT-MLP kernels, workload {label}: B={B} NH={NH} NC={NC} checkpoint_group_size={cgs} on {props.name} ({props.multi_processor_count} CUs)",
           f"Command: python ttt-tk_amd/build.py --stages && python ttt-tk_amd/stage_clocks.py {option}",
           f"Launch times: forward {plain_ms[0]:.2f} ms, backward {plain_ms[1]:.2f} ms (product library); "
           f"{stage_ms[0]:.2f} ms, {stage_ms[1]:.2f} ms with the clocks compiled in",
           "Clocks are shader clocks per mini-batch and wave, averaged over the (batch, head) pairs whose workgroup of that kind ran;",
           "a stage's share is of the workgroup's own total.  Barrier waits are part of the stage that ends with the barrier.", ""]

    def present(x):   # pairs whose workgroup of this kind wrote anything
        return x[x.sum(dim=(1, 2)) > 0]

    def ran(x):       # which pairs had a workgroup of this kind
        return x.sum(dim=(1, 2)) > 0

    def halves(clocks, role):   # both workgroups of every pair, as if they were pairs of their own
        return torch.cat((present(clocks[:, role]), present(clocks[:, role + 1])))

    wide_f, split_f = ran(cf[:, HALF]), ran(cf[:, OUT]) & ~ran(cf[:, HALF])
    one_f = ran(cf[:, 0]) & ~split_f
    if one_f.any():
        out += table(f"forward, one workgroup per pair ({int(one_f.sum())} pairs)", cf[one_f, 0], fwd_names, NC) + [""]
    if split_f.any():
        out += table(f"forward, recurrence workgroup ({int(split_f.sum())} pairs)", cf[split_f, 0], fwd_names, NC) + [""]
        out += table(f"forward, output-branch workgroup ({int(split_f.sum())} pairs)", cf[split_f, OUT], fwd_names, NC) + [""]
    if wide_f.any() and not ran(cf[:, OUT]).any():   # (of the four workgroups the first two keep clocks)
        both = halves(cf, HALF)
        out += table(f"forward, recurrence on four workgroups, compute waves ({int(wide_f.sum())} pairs)", both[:, :4], fwd_quad_names, NC) + [""]
        out += table("forward, recurrence on four workgroups, helper waves", both[:, 4:], fwd_quad_names, NC) + [""]
    elif wide_f.any():
        both = halves(cf, HALF)
        n_out = 2 if ran(cf[:, OUT + 1]).any() else 1
        out += table(f"forward, recurrence on two workgroups, compute waves ({int(wide_f.sum())} pairs)", both[:, :4], fwd_wide_names, NC) + [""]
        out += table("forward, recurrence on two workgroups, helper waves", both[:, 4:], fwd_wide_names, NC) + [""]
        out += table(f"forward, output-branch workgroup 0 of {n_out}", cf[wide_f, OUT], fwd_names, -(-NC // n_out)) + [""]
    wide_b, rep0 = ran(cb[:, WALK_HALF]), ran(cb[:, 0])
    walk_b = ran(cb[:, WALK])
    if (walk_b & ~rep0).any():
        one_b = walk_b & ~rep0
        out += table(f"backward, one workgroup per pair ({int(one_b.sum())} pairs)", cb[one_b, WALK], bwd_names, NC) + [""]
    if rep0.any():
        out += table(f"backward, replaying workgroups, all that worked for a pair ({int(rep0.sum())} pairs)", cb[rep0, 0], bwd_names, NC) + [""]
    if (walk_b & rep0).any():
        out += table(f"backward, reverse-walk workgroup ({int((walk_b & rep0).sum())} pairs)", cb[walk_b & rep0, WALK], bwd_names, NC) + [""]
    if wide_b.any() and not ran(cb[:, DXK]).any():   # (of the four workgroups the first two keep clocks)
        both = halves(cb, WALK_HALF)
        out += table(f"backward, walk on four workgroups, compute waves ({int(wide_b.sum())} pairs)", both[:, :4], bwd_quad_names, NC) + [""]
        out += table("backward, walk on four workgroups, helper waves", both[:, 4:], bwd_quad_names, NC) + [""]
    elif wide_b.any():
        both = halves(cb, WALK_HALF)
        out += table(f"backward, walk on two workgroups, compute waves ({int(wide_b.sum())} pairs)", both[:, :4], bwd_wide_names, NC) + [""]
        out += table("backward, walk on two workgroups, helper waves", both[:, 4:], bwd_wide_names, NC) + [""]
    if ran(cb[:, DXK]).any():
        out += table(f"backward, grad_L_XK workgroup ({int(ran(cb[:, DXK]).sum())} pairs)", present(cb[:, DXK]), bwd_names, NC) + [""]
    text = "\n".join(out)
    print(text)
    if a.out:
        os.makedirs(os.path.dirname(os.path.abspath(a.out)), exist_ok=True)
        with open(a.out, "w") as f:
            f.write(text + "\n")
    del keep0, keep1
    return 0


if __name__ == "__main__":
    sys.exit(main())
