"""Pinned staging buffers of small host-to-device copies, taken in turn."""
import numpy as np
import torch


class PinnedRing:
    """`slots` pinned int32 buffers. A buffer is handed out again once the copy out of it is done: with one buffer a caller that
    prepares a step waits for the copy that the step before it enqueued, which on the device comes after everything enqueued in
    front of it; with several it prepares the next step while the device still works. Steps in a row that nobody waits for, one buffer
    and several: rokevik's prompts (4 x 2000 tokens) 2350 and 2166 us, vafozen's prompts beside decoded tokens 1345 and 1251, the prompts of
    kekapel, lorulix and ratilorn 2635 and 2556, 2555 and 2436, 3041 and 2965. The number of buffers bounds how far it gets ahead. A caller
    that reads a step's results before it prepares the next gains nothing by them. A buffer that is made is as large as the largest so far:
    each is made anew only where the steps themselves grow."""

    def __init__(self, slots: int, floor: int = 1024):
        self._slots = [[None, None, None] for _ in range(slots)]        # tensor, its numpy view, event
        self._next, self._floor = 0, floor

    def fill(self, total: int, arrays) -> "tuple":
        """Writes the arrays (offset, values) into the next buffer -> (its first `total` elements, what to call once the copy out of
        them is enqueued on the current stream)."""
        slot = self._slots[self._next]
        self._next = (self._next + 1) % len(self._slots)
        if slot[2] is not None:
            slot[2].synchronize()
        if slot[0] is None or slot[0].numel() < total:
            self._floor = max(self._floor, 1 << (max(total, 1) - 1).bit_length())
            slot[0] = torch.empty(self._floor, dtype=torch.int32, pin_memory=True)
            slot[1] = slot[0].numpy()
        host: np.ndarray = slot[1]
        for at, values in arrays:
            host[at:at + values.size] = values
        if slot[2] is None:
            slot[2] = torch.cuda.Event()
        return slot[0][:total], slot[2].record
