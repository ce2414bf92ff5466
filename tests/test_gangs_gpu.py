"""The backward whose replaying and finishing workgroups serve several (batch, head) pairs, against the one-workgroup launch, bit
for bit: gangs of unequal size, more and fewer groups than sets and workgroups, groups of one mini-batch, ragged and single
groups, the pair counts at both ends of the walk on two CUs (49 to 56 pairs) and on one (57 to 80), and a wait that gives up.  Groups too
short or few for that have whole workgroups for each pair, which are among the cases."""
import ctypes

import pytest
import torch

from test_overlapped_abi_gpu import _args, _lib
from test_wide_placement_gpu import _reference, _tensors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("NH,NC,cgs,scatter", [(49, 9, 2, 0), (53, 7, 1, 1), (56, 25, 4, 0), (56, 3, 4, 0), (57, 5, 2, 0), (64, 6, 4, 0),
                                               (65, 9, 4, 0), (75, 11, 2, 0), (80, 8, 1, 1), (80, 2, 3, 0),
                                               (53, 13, 4, 1), (55, 31, 10, 0), (65, 93, 8, 0), (72, 95, 24, 0), (80, 91, 10, 1), (80, 99, 30, 0),
                                               (65, 36, 4, 1), (73, 97, 7, 1), (79, 130, 9, 0), (80, 160, 32, 0)])
def test_shared_workgroups_are_bit_identical(NH, NC, cgs, scatter):
    import test_time_training as ext
    import ttt_mlp_host as host
    lib = _lib()
    dev = torch.device("cuda:0")
    K = host.num_checkpoints(NC, cgs)
    print(f"case NH={NH} NC={NC} cgs={cgs}", flush=True)
    t = _tensors(host, NH, NC, cgs, dev)
    ref = _reference(host, ext, t, cgs)
    host.zero_accumulating_grads(t)
    for k in host.GRAD_NAMES[:6]:
        t[k].fill_(float("nan"))
    a = _args(host.BWD_ORDER, t, cgs, 1, NH, NC, K)
    nbytes = lib.ttt_mlp_bwd_workspace_bytes(1, NH, cgs)
    ws = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=dev)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    ptr = ctypes.c_void_p(ws.data_ptr())
    launch = (lambda: lib.ttt_mlp_launch_scattered(1, ctypes.byref(a), ptr, ctypes.c_size_t(nbytes), stream)) if scatter else \
             (lambda: lib.ttt_mlp_bwd_launch_overlapped(ctypes.byref(a), ptr, ctypes.c_size_t(nbytes), stream))
    assert launch() == 0
    torch.cuda.synchronize()
    assert ws.view(torch.int32)[NH * 32].item() == 0, "a workgroup gave up waiting for another"
    for k in host.GRAD_NAMES:
        assert torch.equal(t[k], ref[k]), k


@pytest.mark.parametrize("NH,NC,cgs", [(52, 12, 2), (76, 12, 2), (52, 12, 4), (76, 92, 10)])
def test_a_shared_workgroup_that_gives_up_ends_the_launch(NH, NC, cgs):
    import test_time_training as ext
    import ttt_mlp_host as host
    t = _tensors(host, NH, NC, cgs, torch.device("cuda:0"))
    ref = _reference(host, ext, t, cgs)
    for limit in (1, 1000, 3000, 2_000_000_000):
        print(f"case NH={NH} limit={limit}", flush=True)
        host.zero_accumulating_grads(t)
        ext.set_wait_limit(limit)
        try:
            host.backward(t, cgs)
        except RuntimeError as e:
            assert "gave up" in str(e) and limit < 2_000_000_000
            continue
        finally:
            ext.set_wait_limit(2_000_000_000)
        for k in host.GRAD_NAMES:
            assert torch.equal(t[k], ref[k]), (limit, k)
