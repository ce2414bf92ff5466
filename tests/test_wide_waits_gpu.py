"""Launches with the recurrence (walk) of a pair on two workgroups whose waits give up somewhere in the sequence, forced from
the host by limits between one tick and longer than any wait takes: the call ends and says so, or its results are those of an
undisturbed call, and the device is fine afterwards."""
import pytest
import torch

from oracle import ttt_mlp_oracle as orc

pytestmark = pytest.mark.gpu

FWD_KEYS = ("XQ", "XK", "XV", "last_eta", "ttt_norm_weight", "ttt_norm_bias", "W1", "b1", "W2", "b2")
UP_KEYS = ("grad_L_W1_last", "grad_L_b1_last", "grad_L_W2_last", "grad_L_b2_last", "grad_L_XQW_mini_batch")
LIMITS = (1, 100, 200, 400, 800, 1600, 2400, 3200, 4800, 10000, 2_000_000_000)   # ticks of 10 ns


# a group per mini-batch (the walk waits for a replay at every one) with four replaying workgroups per pair, and with two
@pytest.mark.parametrize("NH,NC,cgs", [(2, 24, 1), (40, 24, 1), (8, 24, 5)])
def test_waits_that_give_up_anywhere_end_the_launch(NH, NC, cgs):
    import ttt_mlp_host as host
    import test_time_training as ext
    dev = torch.device("cuda:0")
    d = orc.make_inputs(1, NH, NC, seed=91)
    t = {k: d[k].to(dev).contiguous() for k in FWD_KEYS + UP_KEYS}
    t.update(host.alloc_forward_buffers(1, NH, NC, cgs, dev))
    t.update(host.alloc_backward_buffers(1, NH, NC, cgs, dev))

    def call(fn, keys, limit):
        print(f"NH={NH} NC={NC} cgs={cgs} {fn.__name__} limit={limit}", flush=True)
        host.zero_accumulating_grads(t)
        ext.set_wait_limit(limit)
        try:
            fn(t, cgs)
        except RuntimeError as e:
            assert "gave up" in str(e) and limit < 2_000_000_000
            return None
        finally:
            ext.set_wait_limit(2_000_000_000)
        return {k: t[k].clone() for k in keys}

    for fn, keys in ((host.forward, ("Out", "W1_checkpoints", "b2_checkpoints")), (host.backward, host.GRAD_NAMES)):
        ref = call(fn, keys, 2_000_000_000)
        gave_up = 0
        for limit in LIMITS:
            got = call(fn, keys, limit)
            gave_up += got is None
            for k in got or ():
                assert torch.equal(got[k], ref[k]), (limit, k)
        assert gave_up > 0, "no limit was short enough"
        # the checkpoints as an undisturbed forward leaves them, for the backward
        got = call(fn, keys, 2_000_000_000)
        assert all(torch.equal(got[k], ref[k]) for k in keys)
