"""The launches with the recurrence (walk) of a pair on two workgroups where a device does not place them on one XCD: forced by
a grid that deals the workgroups of a pair to consecutive XCDs.  And the one with three replaying workgroups, which only a
number of CUs between 56 and 63 per 8 pairs leads to.  Against the one-workgroup launch, bit for bit."""
import ctypes

import pytest
import torch

from oracle import ttt_mlp_oracle as orc

pytestmark = pytest.mark.gpu

FWD_KEYS = ("XQ", "XK", "XV", "last_eta", "ttt_norm_weight", "ttt_norm_bias", "W1", "b1", "W2", "b2")
UP_KEYS = ("grad_L_W1_last", "grad_L_b1_last", "grad_L_W2_last", "grad_L_b2_last", "grad_L_XQW_mini_batch")
OUT_KEYS = ("Out", "W1_checkpoints", "b1_checkpoints", "W2_checkpoints", "b2_checkpoints")


def _tensors(host, NH, NC, cgs, dev):
    d = orc.make_inputs(1, NH, NC, seed=101)
    t = {k: d[k].to(dev).contiguous() for k in FWD_KEYS + UP_KEYS}
    t.update(host.alloc_forward_buffers(1, NH, NC, cgs, dev))
    t.update(host.alloc_backward_buffers(1, NH, NC, cgs, dev))
    return t


def _reference(host, ext, t, cgs):
    ext.set_overlap(False)
    try:
        host.forward(t, cgs)
        host.backward(t, cgs)
    finally:
        ext.set_overlap(True)
    return {k: t[k].clone() for k in OUT_KEYS + host.GRAD_NAMES}


# forward / backward: two output and eight replaying workgroups per pair, two and two, one and two replaying with the walk on one CU; and a
# forward too long for an early start of the next mini-batch
@pytest.mark.parametrize("NH,NC,cgs", [(3, 21, 4), (8, 30, 3), (41, 19, 2), (70, 12, 4), (2, 259, 64)])
def test_workgroups_of_a_pair_on_different_xcds(NH, NC, cgs):
    import test_time_training as ext
    import ttt_mlp_host as host
    from test_overlapped_abi_gpu import _args, _lib
    lib = _lib()
    dev = torch.device("cuda:0")
    K = host.num_checkpoints(NC, cgs)
    print(f"case NH={NH} NC={NC} cgs={cgs}", flush=True)
    t = _tensors(host, NH, NC, cgs, dev)
    ref = _reference(host, ext, t, cgs)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for which, order, nbytes in ((0, host.FWD_ORDER, lib.ttt_mlp_fwd_workspace_bytes(1, NH)),
                                 (1, host.BWD_ORDER, lib.ttt_mlp_bwd_workspace_bytes(1, NH, cgs))):
        host.zero_accumulating_grads(t)
        for k in OUT_KEYS if which == 0 else host.GRAD_NAMES[:6]:
            t[k].fill_(float("nan"))
        a = _args(order, t, cgs, 1, NH, NC, K)
        ws = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=dev)
        assert lib.ttt_mlp_launch_scattered(which, ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(nbytes), stream) == 0
        torch.cuda.synchronize()
        assert ws.view(torch.int32)[NH * 32].item() == 0, "a workgroup gave up waiting for another"
        for k in OUT_KEYS if which == 0 else host.GRAD_NAMES:
            assert torch.equal(t[k], ref[k]), k
    assert lib.ttt_mlp_launch_scattered(2, ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(nbytes), stream) == 1001


@pytest.mark.parametrize("NH,NC,cgs,cus", [(8, 23, 4, 56), (3, 17, 2, 63), (16, 9, 1, 112)])
def test_three_replaying_workgroups(NH, NC, cgs, cus):
    import test_time_training as ext
    import ttt_mlp_host as host
    lib = ctypes.CDLL(__import__("test_overlapped_abi_gpu").LIB)
    one, rest, per = ctypes.c_longlong(), ctypes.c_longlong(), ctypes.c_int()
    assert lib.ttt_mlp_launch_plan(1, ctypes.c_longlong(NH), cus, ctypes.byref(one), ctypes.byref(rest), ctypes.byref(per)) == 0
    assert per.value == 7 and one.value == 0
    print(f"case NH={NH} NC={NC} cgs={cgs} cus={cus}", flush=True)
    t = _tensors(host, NH, NC, cgs, torch.device("cuda:0"))
    ref = _reference(host, ext, t, cgs)
    host.zero_accumulating_grads(t)
    ext.set_compute_units(cus)
    try:
        host.backward(t, cgs)
    finally:
        ext.set_compute_units(0)
    assert ext.last_backward_mode() == 1
    for k in host.GRAD_NAMES:
        assert torch.equal(t[k], ref[k]), k
