"""Host code of the native training step: what it asks of the runtime, over a stand-in for it (tests/hip_stub.py)."""
import hip_stub


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
