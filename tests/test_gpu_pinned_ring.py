"""Staging buffers taken in turn (worker/pinned_ring.py): copies whose device side is still to come keep what was staged for them."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("slots", [1, 2, 4])
def test_copies_behind_a_busy_device(slots):
    from swiftllm_amd.worker.pinned_ring import PinnedRing
    ring, out = PinnedRing(slots, floor=4), []
    work = torch.randn(2048, 2048, device="cuda")
    for i in range(3 * slots + 1):
        for _ in range(4):
            work @ work
        n = 3 + 5 * (i % 4)
        staged, enqueued = ring.fill(n, [(0, np.full(2, 1000 + i, dtype=np.int32)), (2, np.arange(n - 2, dtype=np.int32) + i)])
        dev = torch.empty(n, dtype=torch.int32, device="cuda")
        dev.copy_(staged, non_blocking=True)
        enqueued()
        out.append((i, n, dev))
    for i, n, dev in out:
        assert dev.tolist() == [1000 + i] * 2 + [i + k for k in range(n - 2)]


def test_buffers_are_as_large_as_the_largest_so_far():
    """One large step (memory profiling) sizes every buffer: those after it are not made anew as steps grow up to its size."""
    from swiftllm_amd.worker.pinned_ring import PinnedRing
    ring, made = PinnedRing(3, floor=4), set()
    for n in [900] + list(range(3, 900, 40)):
        staged, enqueued = ring.fill(n, [(0, np.arange(n, dtype=np.int32))])
        assert staged.numel() == n and staged.tolist() == list(range(n))
        enqueued()
        made.add(staged.data_ptr())
    assert len(made) == 3
