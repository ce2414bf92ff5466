"""The backward with the walk of a pair on two workgroups, against the one-workgroup launch, bit for bit: groups of one mini-batch,
ragged and single groups, more groups than sets, and the pair counts where the launch changes shape (four replaying
workgroups per pair up to 32 pairs, two up to 48, the launch with the walk on one workgroup beyond)."""
import pytest
import torch

from oracle import ttt_mlp_oracle as orc

pytestmark = pytest.mark.gpu

FWD_KEYS = ("XQ", "XK", "XV", "last_eta", "ttt_norm_weight", "ttt_norm_bias", "W1", "b1", "W2", "b2")
UP_KEYS = ("grad_L_W1_last", "grad_L_b1_last", "grad_L_W2_last", "grad_L_b2_last", "grad_L_XQW_mini_batch")


@pytest.mark.parametrize("B,NH,NC,cgs,accumulate", [
    (1, 1, 9, 1, True), (1, 3, 17, 2, False), (1, 9, 29, 3, True), (2, 4, 33, 4, False), (1, 5, 16, 8, True), (1, 2, 24, 23, True),
    (4, 8, 13, 4, True), (1, 33, 14, 3, False), (1, 48, 11, 2, True), (7, 7, 9, 4, True)])
def test_walk_on_two_workgroups_is_bit_identical(B, NH, NC, cgs, accumulate):
    import ttt_mlp_host as host
    import test_time_training as ext
    print(f"case B={B} NH={NH} NC={NC} cgs={cgs}", flush=True)
    dev = torch.device("cuda:0")
    d = orc.make_inputs(B, NH, NC, seed=81)
    g = torch.Generator().manual_seed(181)
    d["b1"] = 0.02 * torch.randn(B, NH, 1, 256, generator=g)
    d["ttt_norm_weight"] = 1 + 0.1 * torch.randn(1, NH, 1, 64, generator=g)
    t = {k: d[k].to(dev).contiguous() for k in FWD_KEYS + UP_KEYS}
    t.update(host.alloc_forward_buffers(B, NH, NC, cgs, dev))
    host.forward(t, cgs)
    res = []
    for overlap in (False, True):
        t.update(host.alloc_backward_buffers(B, NH, NC, cgs, dev))
        if accumulate:
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
    for k in res[0]:
        assert torch.isfinite(res[1][k]).all(), k
        assert torch.equal(res[0][k], res[1][k]), k
