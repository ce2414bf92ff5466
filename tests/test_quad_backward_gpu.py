"""The remat backward with the walk of a pair on four workgroups (up to 40 pairs on 256 CUs), against the one-workgroup launch, bit for bit:
the shortest sequences, where the slots of the exchange are first used, come round and are used last; groups of one mini-batch, ragged ones and
more groups than sets; ragged numbers of pairs per XCD, behind a full round of one workgroup per pair too; gradients stored
and added to; and inputs with infinities and NaNs, which pass through the exchange like any other value."""
import os
import sys

import pytest
import torch

from oracle import ttt_mlp_oracle as orc

FWD_KEYS = ("XQ", "XK", "XV", "last_eta", "ttt_norm_weight", "ttt_norm_bias", "W1", "b1", "W2", "b2")
UP_KEYS = ("grad_L_W1_last", "grad_L_b1_last", "grad_L_W2_last", "grad_L_b2_last", "grad_L_XQW_mini_batch")


def _both(B, NH, NC, cgs, accumulate, spoil=None):
    import ttt_mlp_host as host
    import test_time_training as ext
    print(f"case B={B} NH={NH} NC={NC} cgs={cgs}", flush=True)
    dev = torch.device("cuda:0")
    d = orc.make_inputs(B, NH, NC, seed=19 + NC)
    g = torch.Generator().manual_seed(119)
    d["b1"] = 0.02 * torch.randn(B, NH, 1, 256, generator=g)
    d["ttt_norm_weight"] = 1 + 0.1 * torch.randn(1, NH, 1, 64, generator=g)
    if spoil is not None:
        spoil(d)
    t = {k: d[k].to(dev).contiguous() for k in FWD_KEYS + UP_KEYS}
    t.update(host.alloc_forward_buffers(B, NH, NC, cgs, dev))
    host.forward(t, cgs)
    res = []
    for overlap in (False, True):
        t.update(host.alloc_backward_buffers(B, NH, NC, cgs, dev))
        for k in ("grad_L_last_eta", "grad_L_XQ", "grad_L_XK", "grad_L_XV"):
            t[k].fill_(0.25)
        ext.set_overlap(overlap)
        ext.set_accumulate(accumulate)
        try:
            host.backward(t, cgs)
        finally:
            ext.set_overlap(True)
            ext.set_accumulate(True)
        assert ext.last_backward_mode() == int(overlap)
        res.append({k: t[k].float().cpu() for k in host.GRAD_NAMES})
    return res


@pytest.mark.gpu
@pytest.mark.parametrize("B,NH,NC,cgs,accumulate", [
    (1, 1, 2, 1, True), (1, 2, 3, 2, False), (3, 1, 4, 2, True), (1, 9, 5, 3, False), (1, 17, 7, 1, True), (2, 13, 10, 4, False), (1, 32, 6, 5, True),
    (1, 31, 19, 8, False), (1, 4, 66, 64, True), (3, 13, 8, 3, False), (1, 40, 11, 2, True), (4, 67, 3, 2, True)])
def test_walk_on_four_workgroups_is_bit_identical(B, NH, NC, cgs, accumulate):
    one, four = _both(B, NH, NC, cgs, accumulate)
    for k in one:
        assert torch.isfinite(four[k]).all() and torch.equal(one[k], four[k]), k


@pytest.mark.gpu
def test_infinities_and_nans_stay_where_they_are():
    def spoil(d):
        d["XV"][0, 0, 1, 5, 3] = float("nan")
        d["XK"][0, 1, 2, 60, 63] = float("inf")
        d["grad_L_XQW_mini_batch"][0, 2, 3, 17, 0] = float("-inf")
        d["grad_L_W2_last"][0, 3, 7, 7] = float("nan")
    one, four = _both(1, 6, 8, 3, True, spoil)
    for k in one:
        assert torch.equal(torch.isnan(one[k]), torch.isnan(four[k])), k
        assert torch.equal(one[k].nan_to_num(), four[k].nan_to_num()), k
    assert torch.isfinite(four["grad_L_XK"][0, 4:]).all() and not torch.isfinite(four["grad_L_XK"][0, 3]).all()


def test_leaving_is_decided_between_barriers_by_all_waves_alike():
    """As for the walk on two workgroups: the word that says that a wait gave up is not written between two barriers between
    which a wave reads it, and both kinds of waves pass the same barriers."""
    import re
    sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
    import test_wait_protocol_cpu as wp
    text = re.sub(r"//[^\n]*", "", open(os.path.join(wp.CSRC, "ttt_mlp_bwd_quad.hpp")).read())
    body, _ = wp._block(text, text.index("TTT_DEV void bwd_quad_walk"))
    compute, end = wp._block(body, re.search(r"if \(w < 4\) ", body).end())
    kinds = [wp._intervals(wp._inline(kind), "for (int j = n_mb - 1; j >= 0; j--") for kind in (compute, body[end:])]
    assert len(kinds[0]) == len(kinds[1])
    assert any("W" in x for x in kinds[1]) and any("R" in x for x in kinds[0])
    for i, (a, b) in enumerate(zip(*kinds)):
        assert not ("W" in a + b and "R" in a + b), f"interval {i}: the word is written while it is read ({a!r}, {b!r})"


def test_the_stages_of_the_walk_on_four_workgroups_are_marked():
    import re
    pkg = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ttt-tk_amd")
    sys.path.insert(0, pkg)
    import stage_clocks as sc
    names = sc.stage_names(open(os.path.join(pkg, "csrc", "ttt_mlp_kernels.hpp")).read(), "BwdQuadStage")
    text = open(os.path.join(pkg, "csrc", "ttt_mlp_bwd_quad.hpp")).read()
    assert set(re.findall(r"TTT_STAGE\((\w+)\)", text)) == {n for n, _ in names} and all(desc for _, desc in names) and len(names) <= sc.SLOTS
