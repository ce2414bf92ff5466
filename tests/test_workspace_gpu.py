"""A caller-owned workspace for the operator module: with `set_workspace(tensor)` the two operators allocate nothing
(the upstream operator takes every tensor, scratch included, from its caller: kernels/ttt_backward/ttt.cu:1451-1917)
and give the same results, bit for bit, as with a workspace from torch's allocator."""
import pytest
import torch

from oracle import ttt_mlp_oracle as orc

pytestmark = pytest.mark.gpu

FWD_KEYS = ("XQ", "XK", "XV", "last_eta", "ttt_norm_weight", "ttt_norm_bias", "W1", "b1", "W2", "b2")
UP_KEYS = ("grad_L_W1_last", "grad_L_b1_last", "grad_L_W2_last", "grad_L_b2_last", "grad_L_XQW_mini_batch")


def _run(host, t, cgs):
    host.zero_accumulating_grads(t)
    host.forward(t, cgs)
    host.backward(t, cgs)
    torch.cuda.synchronize()
    return {k: t[k].clone() for k in ("Out", "W1_checkpoints", "b1_checkpoints") + host.GRAD_NAMES}


def test_operators_allocate_nothing_with_a_caller_workspace():
    import test_time_training as ext
    import ttt_mlp_host as host
    dev = torch.device("cuda:0")
    B, NH, NC, cgs = 1, 8, 24, 4
    print(f"case B={B} NH={NH} NC={NC} cgs={cgs}", flush=True)
    d = orc.make_inputs(B, NH, NC, seed=5)
    t = {k: d[k].to(dev).contiguous() for k in FWD_KEYS + UP_KEYS}
    t.update(host.alloc_forward_buffers(B, NH, NC, cgs, dev))
    t.update(host.alloc_backward_buffers(B, NH, NC, cgs, dev))
    ext.set_workspace(None)
    ref = _run(host, t, cgs)                       # workspace from torch's allocator
    assert ext.last_forward_mode() == 1 and ext.last_backward_mode() == 1
    nbytes = host.workspace_bytes(B, NH, cgs)
    assert nbytes > 0
    ws = torch.full((nbytes,), 0x5A, dtype=torch.uint8, device=dev)
    try:
        host.set_workspace(ws)
        for call in range(2):
            for k in ("Out",) + host.GRAD_NAMES[:6]:
                t[k].fill_(7.0)
            host.zero_accumulating_grads(t)
            torch.cuda.synchronize()
            before, peak0 = torch.cuda.memory_allocated(dev), torch.cuda.max_memory_allocated(dev)
            torch.cuda.reset_peak_memory_stats(dev)
            host.forward(t, cgs)
            host.backward(t, cgs)
            torch.cuda.synchronize()
            assert torch.cuda.memory_allocated(dev) == before, "the operators kept memory"
            assert torch.cuda.max_memory_allocated(dev) == before, "the operators allocated during the calls"
            assert ext.last_forward_mode() == 1 and ext.last_backward_mode() == 1, "the caller's workspace was not used"
            for k, r in ref.items():
                assert torch.equal(t[k], r), (call, k)
        # a workspace that is too small for the shape: one workgroup per pair, still nothing allocated, same results
        host.set_workspace(ws[:4096])
        host.zero_accumulating_grads(t)
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated(dev)
        torch.cuda.reset_peak_memory_stats(dev)
        host.forward(t, cgs)
        host.backward(t, cgs)
        torch.cuda.synchronize()
        assert torch.cuda.max_memory_allocated(dev) == before
        assert ext.last_forward_mode() == 0 and ext.last_backward_mode() == 0
        for k, r in ref.items():
            assert torch.equal(t[k], r), ("small", k)
        with pytest.raises(RuntimeError):
            ext.set_workspace(torch.zeros(16, dtype=torch.float32, device=dev))
    finally:
        host.set_workspace(None)


def test_compute_unit_budget_turns_the_waiting_launches_off():
    """Workgroups that wait for each other must all be resident; a host that cannot promise the whole device says how
    many CUs there are, and shapes that no longer fit run with one workgroup per (batch, head) - same results."""
    import test_time_training as ext
    import ttt_mlp_host as host
    dev = torch.device("cuda:0")
    B, NH, NC, cgs = 1, 8, 12, 4
    print(f"case B={B} NH={NH} NC={NC} cgs={cgs}", flush=True)
    d = orc.make_inputs(B, NH, NC, seed=6)
    t = {k: d[k].to(dev).contiguous() for k in FWD_KEYS + UP_KEYS}
    t.update(host.alloc_forward_buffers(B, NH, NC, cgs, dev))
    t.update(host.alloc_backward_buffers(B, NH, NC, cgs, dev))
    ref = _run(host, t, cgs)
    assert ext.last_forward_mode() == 1 and ext.last_backward_mode() == 1
    try:
        ext.set_compute_units(15)             # 2 x 8 workgroups do not fit 15 CUs
        assert host.workspace_bytes(B, NH, cgs) == 0
        got = _run(host, t, cgs)
        assert ext.last_forward_mode() == 0 and ext.last_backward_mode() == 0
        for k, r in ref.items():
            assert torch.equal(got[k], r), k
        ext.set_compute_units(16)             # two per pair fit, more do not
        assert host.workspace_bytes(B, NH, cgs) > 0
        got = _run(host, t, cgs)
        assert ext.last_forward_mode() == 1 and ext.last_backward_mode() == 1
        for k, r in ref.items():
            assert torch.equal(got[k], r), k
    finally:
        ext.set_compute_units(0)


@pytest.mark.parametrize("NH,NC,cgs", [(8, 3, 4), (8, 7, 4), (3, 9, 4), (8, 48, 4), (40, 5, 4), (8, 5, 1)])
def test_short_sequences_and_small_workspaces(NH, NC, cgs):
    """One set of per-group tensors per checkpoint group is enough for a short sequence (K groups, the caller's own set among
    them), and a workspace too small for three or four recomputing workgroups still serves two; results do not change."""
    import ctypes
    import os
    import test_time_training as ext
    import ttt_mlp_host as host
    from test_overlapped_abi_gpu import LIB, _args
    lib = ctypes.CDLL(LIB)
    lib.ttt_mlp_bwd_workspace_bytes.restype = ctypes.c_size_t
    dev = torch.device("cuda:0")
    B, K = 1, host.num_checkpoints(NC, cgs)
    print(f"case B={B} NH={NH} NC={NC} cgs={cgs} K={K}", flush=True)
    d = orc.make_inputs(B, NH, NC, seed=7)
    t = {k: d[k].to(dev).contiguous() for k in FWD_KEYS + UP_KEYS}
    t.update(host.alloc_forward_buffers(B, NH, NC, cgs, dev))
    t.update(host.alloc_backward_buffers(B, NH, NC, cgs, dev))
    ext.set_overlap(False)
    try:
        ref = _run(host, t, cgs)
    finally:
        ext.set_overlap(True)
    least, most = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib.ttt_mlp_bwd_workspace_range(B, NH, cgs, K, ctypes.byref(least), ctypes.byref(most)) == 0
    full = lib.ttt_mlp_bwd_workspace_bytes(B, NH, cgs)
    sets = 6 if NH <= 32 else 4
    per_set = NH * cgs * (7 * 32768 + 4 * 8192 + 256)      # seven images, four tiles, a vector per slot
    assert full - most.value == max(0, sets - K) * per_set
    assert most.value - least.value == (min(sets, K) - min(4, K)) * per_set
    ba = _args(host.BWD_ORDER, t, cgs, B, NH, NC, K)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for nbytes in (most.value, least.value):
        host.zero_accumulating_grads(t)
        for k in host.GRAD_NAMES[:6]:
            t[k].fill_(7.0)
        ws = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=dev)
        assert lib.ttt_mlp_bwd_launch_within(ctypes.byref(ba), ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(least.value - 1), stream) == 1006
        assert lib.ttt_mlp_bwd_launch_within(ctypes.byref(ba), ctypes.c_void_p(ws.data_ptr()), ctypes.c_size_t(nbytes), stream) == 0
        torch.cuda.synchronize()
        for k in host.GRAD_NAMES:
            assert torch.equal(t[k], ref[k]), (nbytes, k)
    # the operator: what it allocates, and what it does with a caller's tensor of either size
    if K >= 2:
        del ws
        host.zero_accumulating_grads(t)
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated(dev)
        torch.cuda.reset_peak_memory_stats(dev)
        host.backward(t, cgs)
        assert ext.last_backward_mode() == 1
        # (the caching allocator rounds to 512 bytes and hands out a block of up to 1 MiB more rather than split it; a set is 2 MiB or more)
        assert torch.cuda.max_memory_allocated(dev) - before <= most.value + 512 + (1 << 20)
        try:
            for nbytes, mode in ((least.value, 1), (least.value - 1, 0)):
                host.set_workspace(torch.empty(nbytes, dtype=torch.uint8, device=dev))
                host.zero_accumulating_grads(t)
                host.backward(t, cgs)
                assert ext.last_backward_mode() == mode
                for k in host.GRAD_NAMES:
                    assert torch.equal(t[k], ref[k]), (nbytes, k)
        finally:
            host.set_workspace(None)
