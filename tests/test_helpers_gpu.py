"""The backward of more pairs than half the CUs, whose idle CUs replay checkpoint groups for all of them, against the one-workgroup
launch alone, bit for bit: one and two sets for the taken groups, two groups (one to take), groups of one mini-batch, ragged ones,
many more groups than sets, few CUs, and the fewest and most pairs."""
import ctypes

import pytest
import torch

from test_wide_placement_gpu import _reference, _tensors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("NH,NC,cgs,cus", [(129, 13, 3, 256), (170, 9, 2, 256), (171, 21, 4, 256), (200, 17, 4, 256), (248, 20, 1, 256), (150, 40, 1, 256),
                                           (9, 33, 16, 17), (9, 7, 4, 17), (13, 24, 7, 21), (16, 50, 3, 24), (17, 70, 32, 25), (20, 11, 5, 28),
                                           (200, 17, 9, 256), (15, 6, 3, 23)])   # (the last two: too few groups for all, so no helpers)
def test_groups_replayed_by_helpers_are_bit_identical(NH, NC, cgs, cus):
    import test_time_training as ext
    import ttt_mlp_host as host
    from test_overlapped_abi_gpu import _args, _lib
    lib = _lib()
    dev = torch.device("cuda:0")
    K = host.num_checkpoints(NC, cgs)
    print(f"case NH={NH} NC={NC} cgs={cgs} cus={cus}", flush=True)
    t = _tensors(host, NH, NC, cgs, dev)
    ref = _reference(host, ext, t, cgs)
    ext.set_compute_units(cus)

    def check():
        for k in host.GRAD_NAMES:
            assert torch.equal(t[k], ref[k]), k

    def clear():
        host.zero_accumulating_grads(t)
        for k in host.GRAD_NAMES[:6]:
            t[k].fill_(float("nan"))
    try:
        for _ in range(3):   # (who takes which group differs from run to run)
            clear()
            host.backward(t, cgs)
            assert ext.last_backward_mode() == (1 if 7 * (cus - NH) * (K - 1) >= 4 * NH else 0)
            check()
        nbytes = lib.ttt_mlp_bwd_workspace_bytes(1, NH, cgs)
        ws = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=dev)
        clear()
        a = _args(host.BWD_ORDER, t, cgs, 1, NH, NC, K)
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert lib.ttt_mlp_bwd_launch_overlapped(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(nbytes), stream) == 0
        torch.cuda.synchronize()
        assert ws.view(torch.int32)[lib.ttt_mlp_bwd_status_offset(1, NH) // 4].item() == 0, "a workgroup gave up waiting for another"
        check()
    finally:
        ext.set_compute_units(0)


@pytest.mark.parametrize("NH", [129, 200])
def test_sets_of_helpers_hold_what_a_helper_writes(NH):
    """Two further sets of five images, four tiles and a vector per mini-batch of a group: the GELU images of the other launches have no
    place in them."""
    from test_overlapped_abi_gpu import _lib
    lib = _lib()
    for cgs in (4, 16, 64):
        assert lib.ttt_mlp_bwd_workspace_bytes(1, NH, 2 * cgs) - lib.ttt_mlp_bwd_workspace_bytes(1, NH, cgs) == NH * cgs * 2 * (5 * 32768 + 4 * 8192 + 256)


@pytest.mark.parametrize("NH,NC,cgs", [(136, 24, 4), (200, 30, 3)])
def test_a_pair_that_gives_up_ends_the_launch(NH, NC, cgs):
    """A pair that stops waiting for a taken group ends the launch with an error; a helper that stops waiting for one to take only leaves."""
    import test_time_training as ext
    import ttt_mlp_host as host
    t = _tensors(host, NH, NC, cgs, torch.device("cuda:0"))
    ref = _reference(host, ext, t, cgs)
    for limit in (1, 1000, 2_000_000_000):
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
