"""The backward whose first groups are replayed by several workgroups at once, a stretch of the group's mini-batches each, against the
one-workgroup launch, bit for bit: two, three and four stretches, groups of fewer mini-batches than stretches, ragged ones whose
stretches are empty, stretches of one mini-batch and of many, and fewer groups than are shared."""
import pytest
import torch

from test_wide_placement_gpu import _reference, _tensors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("NH,NC,cgs", [(1, 70, 64), (3, 19, 9), (9, 33, 16), (17, 40, 12), (24, 18, 16), (24, 5, 1), (25, 35, 32), (32, 29, 7),
                                       (33, 25, 8), (40, 11, 10), (40, 6, 2)])
def test_groups_replayed_in_parts_are_bit_identical(NH, NC, cgs):
    import test_time_training as ext
    import ttt_mlp_host as host
    print(f"case NH={NH} NC={NC} cgs={cgs}", flush=True)
    t = _tensors(host, NH, NC, cgs, torch.device("cuda:0"))
    ref = _reference(host, ext, t, cgs)
    host.zero_accumulating_grads(t)
    for k in host.GRAD_NAMES[:6]:
        t[k].fill_(float("nan"))
    host.backward(t, cgs)
    assert ext.last_backward_mode() == 1
    for k in host.GRAD_NAMES:
        assert torch.equal(t[k], ref[k]), k
