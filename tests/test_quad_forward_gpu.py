"""The forward with the recurrence of a pair, and Out, on four workgroups (up to 64 pairs on 256 CUs), against the one-workgroup launch, bit
for bit: the shortest sequences, where the slots of the exchange are first used, come round and are used last; ragged numbers of
pairs per XCD; and inputs with infinities and NaNs, which pass through the exchange like any other value."""
import os
import sys

import pytest
import torch

from oracle import ttt_mlp_oracle as orc

FWD_KEYS = ("XQ", "XK", "XV", "last_eta", "ttt_norm_weight", "ttt_norm_bias", "W1", "b1", "W2", "b2")
OUT_KEYS = ("Out", "W1_checkpoints", "b1_checkpoints", "W2_checkpoints", "b2_checkpoints")


def _both(B, NH, NC, cgs, spoil=None):
    import ttt_mlp_host as host
    import test_time_training as ext
    print(f"case B={B} NH={NH} NC={NC} cgs={cgs}", flush=True)
    dev = torch.device("cuda:0")
    d = orc.make_inputs(B, NH, NC, seed=5 + NC, with_grads=False)
    if spoil is not None:
        spoil(d)
    res = []
    for overlap in (False, True):
        t = {k: d[k].to(dev).contiguous() for k in FWD_KEYS}
        t.update(host.alloc_forward_buffers(B, NH, NC, cgs, dev))
        for k in OUT_KEYS:
            t[k].fill_(7.0)
        ext.set_overlap(overlap)
        try:
            host.forward(t, cgs)
        finally:
            ext.set_overlap(True)
        assert ext.last_forward_mode() == int(overlap)
        res.append({k: t[k].float().cpu() for k in OUT_KEYS})
    return res


@pytest.mark.gpu
@pytest.mark.parametrize("B,NH,NC,cgs", [(1, 2, 2, 2), (2, 1, 3, 1), (1, 9, 4, 3), (3, 17, 5, 5), (1, 63, 6, 4), (1, 64, 7, 2), (1, 5, 513, 64)])
def test_recurrence_on_four_workgroups_is_bit_identical(B, NH, NC, cgs):
    one, four = _both(B, NH, NC, cgs)
    for k in OUT_KEYS:
        assert torch.isfinite(four[k]).all() and torch.equal(one[k], four[k]), k


@pytest.mark.gpu
def test_a_single_mini_batch():
    """(through the C interface: the operator takes one workgroup per pair for it)"""
    import ctypes
    import ttt_mlp_host as host
    from test_overlapped_abi_gpu import _args, _lib
    lib, dev, NH = _lib(), torch.device("cuda:0"), 3
    print("case NC=1", flush=True)
    d = orc.make_inputs(1, NH, 1, seed=6, with_grads=False)
    t = {k: d[k].to(dev).contiguous() for k in FWD_KEYS}
    t.update(host.alloc_forward_buffers(1, NH, 1, 1, dev))
    host.forward(t, 1)
    ref = {k: t[k].clone() for k in OUT_KEYS}
    for k in OUT_KEYS:
        t[k].fill_(7.0)
    nbytes = lib.ttt_mlp_fwd_workspace_bytes(1, NH)
    ws = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=dev)
    a = _args(host.FWD_ORDER, t, 1, 1, NH, 1, 1)
    assert lib.ttt_mlp_fwd_launch_overlapped(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(nbytes),
                                             ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    for k in OUT_KEYS:
        assert torch.equal(t[k], ref[k]), k


@pytest.mark.gpu
def test_infinities_and_nans_stay_where_they_are():
    def spoil(d):
        d["XV"][0, 0, 1, 5, 3] = float("nan")
        d["XK"][0, 1, 2, 60, 63] = float("inf")
        d["XQ"][0, 2, 3, 17, 0] = float("-inf")
        d["W2"][0, 3, 7, 7] = float("nan")
    one, four = _both(1, 6, 8, 3, spoil)
    for k in OUT_KEYS:
        assert torch.equal(torch.isnan(one[k]), torch.isnan(four[k])), k
        assert torch.equal(one[k].nan_to_num(), four[k].nan_to_num()), k
    assert torch.isfinite(four["Out"][0, 4:]).all() and not torch.isfinite(four["Out"][0, :4]).all()


def test_leaving_is_decided_between_barriers_by_all_waves_alike():
    """As for the recurrence on two workgroups: the word that says that a wait gave up is not written between two barriers between
    which a wave reads it, and both kinds of waves pass the same barriers."""
    import re
    sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
    import test_wait_protocol_cpu as wp
    text = re.sub(r"//[^\n]*", "", open(os.path.join(wp.CSRC, "ttt_mlp_fwd_quad.hpp")).read())
    body, _ = wp._block(text, text.index("TTT_DEV void fwd_quad_recurrence"))
    compute, end = wp._block(body, re.search(r"if \(compute\) ", body).end())
    kinds = [wp._intervals(wp._inline(kind), "for (int mb = 0; mb < p.NC; mb++") for kind in (compute, body[end:])]
    assert len(kinds[0]) == len(kinds[1]) == 2 + 2 * 4 + 2 + 1
    assert any("W" in x for x in kinds[1]) and any("R" in x for x in kinds[0])
    for i, (a, b) in enumerate(zip(*kinds)):
        assert not ("W" in a + b and "R" in a + b), f"interval {i}: the word is written while it is read ({a!r}, {b!r})"


def test_the_stages_of_the_recurrence_on_four_workgroups_are_marked():
    import re
    pkg = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ttt-tk_amd")
    sys.path.insert(0, pkg)
    import stage_clocks as sc
    names = sc.stage_names(open(os.path.join(pkg, "csrc", "ttt_mlp_kernels.hpp")).read(), "FwdQuadStage")
    text = open(os.path.join(pkg, "csrc", "ttt_mlp_fwd_quad.hpp")).read()
    assert set(re.findall(r"TTT_STAGE\((\w+)\)", text)) == {n for n, _ in names} and all(desc for _, desc in names) and len(names) <= sc.SLOTS
