"""Host code of the native training step: what it asks of the runtime, over a stand-in for it (tests/hip_stub.py)."""
import ctypes
import types

import hip_stub
import torch

from pointtransformerv3_amd import native_train


def test_the_second_stream_is_waited_for_where_a_call_of_the_runtime_fails(tmp_path):
    """Whatever event call fails: once the backward has returned, the caller's buffers belong to its stream again. Either that
    stream waits for an event recorded behind the last launch on the second stream, or the host has waited for that stream."""
    hip_stub.run(r'''
from train_description import Step
MAIN, SIDE = 0x100, 0x200
step = Step()
step.net.side = SIDE
size = step.sizes(lib)[2]

def joined():
    launched = [i for i, (op, a, b, failed) in enumerate(calls()) if op == "launch" and a == SIDE]
    if not launched:
        return True
    behind = [c for c in calls()[launched[-1]:] if not c[3]]
    recorded = set()
    for op, a, b, failed in behind:
        if op == "synchronize" and a == SIDE:
            return True
        if op == "record" and a == SIDE:
            recorded.add(b)
        if op == "wait" and a == MAIN and b in recorded:
            return True
    return False

clear()
assert step.backward(lib, MAIN, size) == 0 and joined()
count = {op: sum(c[0] == op for c in calls()) for op in ("create", "record", "wait", "launch", "synchronize", "destroy")}
assert count["create"] == count["destroy"] == 3 and count["synchronize"] == 0
assert any(c[0] == "launch" and c[1] == SIDE for c in calls()) and count["record"] > 4
for op in ("create", "record", "wait"):
    for nth in range(count[op]):
        clear(fail=op, nth=nth)
        rc = step.backward(lib, MAIN, size)
        assert rc != 0, (op, nth)
        assert joined(), (op, nth, [c for c in calls() if c[0] != "launch"])
        assert sum(c[0] == "create" and not c[3] for c in calls()) == sum(c[0] == "destroy" for c in calls())
''', tmp_path)


def test_a_description_without_the_second_stream_is_not_read_past_its_end(tmp_path):
    """A caller built before the field was there hands over a description that ends in front of it, here at the end of what
    may be read."""
    hip_stub.run(r'''
import mmap
from train_description import Step
from pointtransformerv3_amd import native_train as t
step = Step()
step.net.has_side = 0
size, known = step.sizes(lib)[2], t._Net.side.offset
assert known == ctypes.sizeof(t._Net) - 8 and known % 8 == 0
libc, page = ctypes.CDLL(None, use_errno=True), mmap.PAGESIZE
pages = -(-known // page)
area = mmap.mmap(-1, (pages + 1) * page)
base = ctypes.addressof(ctypes.c_char.from_buffer(area))
libc.mprotect.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
assert libc.mprotect(base + pages * page, page, 0) == 0
at = base + pages * page - known
ctypes.memmove(at, ctypes.addressof(step.net), known)
clear()
assert step.backward(lib, 0x100, size, net=at) == 0
assert {a for op, a, b, failed in calls() if op == "launch"} == {0x100}
assert not [c for c in calls() if c[0] in ("create", "record", "wait")]
assert step.sizes(lib)[2] == size
import os
sys.stdout.flush()
os._exit(0)   # the area is never unmapped: it is half protected
''', tmp_path)


def test_without_the_second_stream_the_backward_needs_less_scratch(tmp_path):
    """What it then asks for is refused by one byte, and on one stream it takes groups of weight gradients in turn."""
    hip_stub.run(r'''
from train_description import Step
for points in ((60_000, 40_000, 12_000), (300_000, 200_000, 100_000)):
    step = Step(points)
    step.net.side = 0x200
    two = step.sizes(lib)
    step.net.side = None
    one = step.sizes(lib)
    assert one[:2] == two[:2] and one[2] < 0.85 * two[2], (one, two)
    clear()
    assert step.backward(lib, 0x100, one[2] - 1) == -3 and not calls()
    assert step.backward(lib, 0x100, one[2]) == 0 and {c[1] for c in calls()} == {0x100}
''', tmp_path)


def test_a_backward_that_finds_no_memory_for_two_streams_takes_one(monkeypatch):
    """A step that fitted without the second stream still runs: the description that is handed over then names none, the
    engine's own stays as it is for the steps to come."""
    weight, seen = torch.nn.Parameter(torch.ones(1)), []

    class Lib:
        def ptv3_train_bytes(self, net, levels, acts, fwd, bwd):
            for at, size in ((acts, 512), (fwd, 512), (bwd, 4096 if net._obj.side else 2048)):
                ctypes.c_size_t.from_address(at).value = size
            return 0

        def ptv3_train_fwd(self, *args):
            return 0

        def ptv3_train_bwd(self, net, levels, dout, dt, masks, acts, scratch, nbytes, grads, stream):
            seen.append((net._obj.side, nbytes))
            ctypes.memset(grads, 0, 4)
            return 0

    lib = Lib()
    monkeypatch.setattr(native_train._lib, "load", lambda: lib)
    monkeypatch.setattr(native_train.ops, "_stream", lambda: None)
    net = native_train._Net(has_side=1, side=0x200)
    engine = types.SimpleNamespace(net=net, out_channels=4, dtype=torch.float32, total=1, params=[weight], read_back=[weight])
    engine.versions = lambda: [p._version for p in engine.read_back]
    empty, short = torch.empty, [True]

    def limited(*size, **kw):
        if short[0] and size == (4096,):
            raise torch.cuda.OutOfMemoryError("no room")
        return empty(*size, **kw)

    monkeypatch.setattr(torch, "empty", limited)
    for short[0] in (True, False):
        out = native_train._Step.apply(engine, torch.zeros(6, 6), types.SimpleNamespace(levels=None), [None], weight)
        out.sum().backward()
    assert seen == [(None, 2048), (0x200, 4096)] and net.side == 0x200
