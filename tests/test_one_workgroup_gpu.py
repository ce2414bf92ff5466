"""The backward with one workgroup per pair on both sides of the line between cached and streamed stores of the replay, against the
launches with several workgroups per pair, bit for bit: groups of one mini-batch, ragged last groups."""
import pytest
import torch

from test_wide_placement_gpu import _reference, _tensors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("NH", [79, 80])
@pytest.mark.parametrize("NC,cgs", [(3, 1), (7, 3), (9, 5)])
def test_one_workgroup_per_pair_is_bit_identical(NH, NC, cgs):
    import test_time_training as ext
    import ttt_mlp_host as host
    print(f"case NH={NH} NC={NC} cgs={cgs}", flush=True)
    t = _tensors(host, NH, NC, cgs, torch.device("cuda:0"))
    ref = _reference(host, ext, t, cgs)   # one workgroup per pair
    host.zero_accumulating_grads(t)
    for k in host.GRAD_NAMES[:6]:
        t[k].fill_(float("nan"))
    host.backward(t, cgs)
    assert ext.last_backward_mode() == 1   # several
    for k in host.GRAD_NAMES:
        assert torch.equal(t[k], ref[k]), k
