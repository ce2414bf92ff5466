"""How a call learns that a wait gave up, and where it gets its workspace: more waiting calls in a row than there are words to report
to, and an allocator without room, which leaves one workgroup per (batch, head) and the same results."""
import pytest
import torch

from test_wide_placement_gpu import _reference, _tensors

pytestmark = pytest.mark.gpu


def test_a_failed_call_neither_keeps_its_word_nor_taints_the_next():
    import test_time_training as ext
    import ttt_mlp_host as host
    t = _tensors(host, 2, 3, 1, torch.device("cuda:0"))
    ref = _reference(host, ext, t, 1)
    for call in range(150):
        ext.set_wait_limit(1 if call % 2 else 2_000_000_000)
        try:
            if call % 2:
                with pytest.raises(RuntimeError, match="gave up"):
                    host.forward(t, 1)
            else:
                host.forward(t, 1)
                assert torch.equal(t["Out"], ref["Out"])
        finally:
            ext.set_wait_limit(2_000_000_000)
    ext.check_last_status()


def test_an_allocator_without_room_leaves_one_workgroup_per_pair():
    import test_time_training as ext
    import ttt_mlp_host as host
    t = _tensors(host, 3, 8, 2, torch.device("cuda:0"))
    ref = _reference(host, ext, t, 2)
    host.zero_accumulating_grads(t)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved() / total)
        host.forward(t, 2)
        host.backward(t, 2)
        assert ext.last_backward_mode() == 0
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    for k, r in ref.items():
        assert torch.equal(t[k], r), k
