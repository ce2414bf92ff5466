"""What the backward does with the four outputs that it adds to, in every launch that shares workgroups between (batch, head) pairs or between
roles: adding to values that are there, and overwriting whatever is there, against the one-workgroup launch under the same policy, bit for
bit.  And the launch with helpers on two streams at a time."""
import ctypes

import pytest
import torch

from test_overlapped_abi_gpu import _args, _lib
from test_wide_placement_gpu import _reference, _tensors

pytestmark = pytest.mark.gpu

ADDED = ("grad_L_last_eta", "grad_L_XQ", "grad_L_XK", "grad_L_XV")
GANG = "ttt_mlp_bwd_gang_kernel<%s>"


def _prefill(t, old):
    for k in ADDED:
        t[k].copy_(old[k]) if isinstance(old, dict) else t[k].fill_(old)


@pytest.mark.parametrize("NH,NC,cgs,cus,kernel", [
    (9, 33, 16, 256, GANG % "true, true, true, true, true"),
    (40, 11, 10, 256, GANG % "true, false, false, true, true"),
    (44, 13, 4, 256, GANG % "true, false, false, true, false"),
    (53, 13, 4, 256, GANG % "true, false, false, false, false"),
    (49, 9, 2, 256, GANG % "false, true, false, true, false"),     # four whole workgroups per pair
    (60, 13, 3, 256, GANG % "false, true, false, true, false"),    # shared replaying ones
    (72, 48, 4, 256, GANG % "false, true, false, true, false"),
    (80, 91, 10, 256, GANG % "false, true, false, false, false"),  # and finishing ones
    (80, 13, 3, 256, "ttt_mlp_bwd_split_kernel<2>"),
    (96, 9, 2, 256, "ttt_mlp_bwd_split_kernel<1>"),
    (136, 24, 4, 256, "ttt_mlp_bwd_helped_kernel"),
    (200, 30, 3, 256, "ttt_mlp_bwd_helped_kernel"),
    (16, 50, 10, 24, "ttt_mlp_bwd_helped_kernel")])
def test_added_to_and_overwritten_outputs_in_every_launch(NH, NC, cgs, cus, kernel):
    import test_time_training as ext
    import ttt_mlp_host as host
    lib = _lib()
    lib.ttt_mlp_launched_kernel.restype = ctypes.c_char_p
    dev = torch.device("cuda:0")
    K = host.num_checkpoints(NC, cgs)
    assert lib.ttt_mlp_launched_kernel(1, ctypes.c_longlong(NH), cus, NC, cgs, 1, 0, None, None, None).decode() == kernel
    t = _tensors(host, NH, NC, cgs, dev)
    g = torch.Generator(device=dev).manual_seed(3)
    old = {k: torch.empty_like(t[k]).normal_(0.0, 0.5, generator=g) for k in ADDED}
    for accumulate, before in ((True, old), (False, float("nan")), (False, old)):
        print(f"case NH={NH} NC={NC} cgs={cgs} cus={cus} accumulate={accumulate}", flush=True)
        host.set_accumulate(accumulate)
        ext.set_compute_units(cus)
        try:
            _prefill(t, before)
            ref = _reference(host, ext, t, cgs)
            _prefill(t, before)
            for k in host.GRAD_NAMES[:6]:
                t[k].fill_(float("nan"))
            nbytes = lib.ttt_mlp_bwd_workspace_bytes(1, NH, cgs)
            ws = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=dev)
            a = _args(host.BWD_ORDER, t, cgs, 1, NH, NC, K)
            a.overwrite = 0 if accumulate else 1
            stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
            assert lib.ttt_mlp_bwd_launch_overlapped(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(nbytes), stream) == 0
            torch.cuda.synchronize()
            words = ws.view(torch.int32)[:NH * 32 + 1].cpu()
            assert words[NH * 32] == 0, "a workgroup gave up waiting for another"
            if "helped" in kernel:   # (the group last replayed into a pair's sets 1 and 2)
                assert words[:NH * 32].view(NH, 32)[:, 1:3].max() > 0, "no helper took a group"
            for k in host.GRAD_NAMES:
                assert torch.equal(t[k], ref[k]), k
            if accumulate:
                assert not torch.equal(ref["grad_L_XK"], old["grad_L_XK"]) and torch.isfinite(ref["grad_L_XK"]).all()
            # the operator, which takes its workspace by the call's own sizes
            _prefill(t, before)
            host.backward(t, cgs)
            assert ext.last_backward_mode() == 1
            for k in host.GRAD_NAMES:
                assert torch.equal(t[k], ref[k]), ("operator", k)
        finally:
            ext.set_compute_units(0)
            host.set_accumulate(True)


@pytest.mark.parametrize("NH,NC,cgs", [(136, 24, 4), (200, 30, 3)])
def test_helpers_on_two_streams(NH, NC, cgs):
    """No workgroup of this launch waits for one that is not running, so two of them may share the device."""
    import test_time_training as ext
    import ttt_mlp_host as host
    print(f"case NH={NH} NC={NC} cgs={cgs}", flush=True)
    dev = torch.device("cuda:0")
    ts = [_tensors(host, NH, NC, cgs, dev) for _ in range(2)]
    ts[1]["grad_L_XQW_mini_batch"].mul_(-0.5)
    refs = [_reference(host, ext, t, cgs) for t in ts]
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    host.set_synchronize(False)
    try:
        for _ in range(3):
            for t, s in zip(ts, streams):
                with torch.cuda.stream(s):
                    host.zero_accumulating_grads(t)
                    host.backward(t, cgs)
                    assert ext.last_backward_mode() == 1
        torch.cuda.synchronize()
        ext.check_last_status()
    finally:
        host.set_synchronize(True)
    for t, ref in zip(ts, refs):
        for k in host.GRAD_NAMES:
            assert torch.equal(t[k], ref[k]), k
