"""The forward with the recurrence of a pair on two workgroups, against the one-workgroup launch, bit for bit: where the ring
of states wraps, at the smallest sequences, and at the pair counts where the launch changes shape (two output workgroups
per pair up to 64 pairs, one up to 80, the older two-workgroup launch beyond), and on both sides of the lengths up to which the products
of a mini-batch are started in the one before."""
import pytest
import torch

from oracle import ttt_mlp_oracle as orc

pytestmark = pytest.mark.gpu

FWD_KEYS = ("XQ", "XK", "XV", "last_eta", "ttt_norm_weight", "ttt_norm_bias", "W1", "b1", "W2", "b2")


@pytest.mark.parametrize("B,NH,NC,cgs", [(1, 1, 2, 1), (1, 7, 3, 2), (1, 9, 8, 8), (1, 5, 9, 4), (2, 4, 17, 5), (1, 3, 70, 16),
                                         (1, 64, 11, 4), (5, 13, 11, 4), (1, 80, 10, 4), (1, 81, 3, 2),
                                         (1, 3, 256, 50), (1, 3, 257, 50), (1, 64, 96, 16), (1, 64, 97, 97)])
def test_recurrence_on_two_workgroups_is_bit_identical(B, NH, NC, cgs):
    import ttt_mlp_host as host
    import test_time_training as ext
    print(f"case B={B} NH={NH} NC={NC} cgs={cgs}", flush=True)
    dev = torch.device("cuda:0")
    d = orc.make_inputs(B, NH, NC, seed=71, with_grads=False)
    g = torch.Generator().manual_seed(171)
    d["b1"] = 0.02 * torch.randn(B, NH, 1, 256, generator=g)
    d["b2"] = 0.02 * torch.randn(B, NH, 1, 64, generator=g)
    d["ttt_norm_weight"] = 1 + 0.1 * torch.randn(1, NH, 1, 64, generator=g)
    d["ttt_norm_bias"] = 0.1 * torch.randn(1, NH, 1, 64, generator=g)
    res = []
    for overlap in (False, True):
        t = {k: d[k].to(dev).contiguous() for k in FWD_KEYS}
        t.update(host.alloc_forward_buffers(B, NH, NC, cgs, dev))
        for k in ("Out", "W1_checkpoints", "b1_checkpoints", "W2_checkpoints", "b2_checkpoints"):
            t[k].fill_(float("nan"))
        ext.set_overlap(overlap)
        try:
            host.forward(t, cgs)
        finally:
            ext.set_overlap(True)
        assert ext.last_forward_mode() == int(overlap)
        res.append({k: t[k].float().cpu() for k in ("Out", "W1_checkpoints", "b1_checkpoints", "W2_checkpoints", "b2_checkpoints")})
    for k in res[0]:
        assert torch.isfinite(res[1][k]).all(), k
        assert torch.equal(res[0][k], res[1][k]), k
