"""Pinned words through which kernels report to the host (ptv3_index_wait): no copy, no event, and what was queued behind
the reporting kernel runs while the host reads."""
import collections
import ctypes
import itertools

import torch

from . import _lib

DATA = 3   # PTV3_SLOT_DATA


class _Slot:
    def __init__(self, words):
        self.tensor = torch.zeros(words, dtype=torch.int64, pin_memory=True)
        self.ptr = self.tensor.data_ptr()
        self.words = (ctypes.c_int64 * words).from_address(self.ptr)


_FREE = collections.deque(maxlen=16)   # append and pop are atomic
_SEQ = itertools.count(1)


def next_seq():
    """A number no slot's words hold yet."""
    return next(_SEQ)


def take(words):
    """A slot of at least `words` words that no queued kernel writes to; give() it back once what it reported is read."""
    kept = []
    slot = None
    while slot is None:
        try:
            s = _FREE.pop()
        except IndexError:
            slot = _Slot(max(words, 256))
            break
        if len(s.words) >= words:
            slot = s
        else:
            kept.append(s)
    _FREE.extend(kept)
    return slot


def give(slot):
    _FREE.append(slot)


def wait(slot, which, seq, stream):
    """Until the kernels of stage `which` have reported `seq`."""
    _lib.check(_lib.load().ptv3_index_wait(slot.ptr, which, seq, stream), "ptv3_index_wait")
