"""Host-side rules of the natively queued paths that need no GPU."""
import contextlib
import types

import pytest
import torch

from pointtransformerv3_amd import native


class _Stop(Exception):
    pass


@pytest.mark.parametrize("overlap", [True, False])
def test_inputs_are_converted_where_the_index_reads_them(overlap, monkeypatch):
    """Under the overlapped schedule the index stream waits for nothing: a conversion queued on the caller's stream would
    still be pending when the index kernels read its result."""
    inside, seen = [False], []

    class Overlap:
        device = torch.device("cpu")

        @contextlib.contextmanager
        def scope(self):
            inside[0] = True
            yield
            inside[0] = False

    def build(*args, **kw):
        raise _Stop

    monkeypatch.setattr(native.ops, "_stream", lambda: None)
    monkeypatch.setattr(native, "coordinates", lambda point: seen.append(inside[0]) or (None, None, None))
    monkeypatch.setattr(native.levels, "build", build)
    engine = native.Engine.__new__(native.Engine)
    engine.layout = engine.want = None
    engine._refresh = native._Refresh()   # nothing to refresh: launches nothing
    model = types.SimpleNamespace(overlap_index_prologue=overlap, _prologue_state=Overlap(), order=("z",), shuffle_orders=False)
    with pytest.raises(_Stop):
        engine.forward(model, dict(feat=torch.zeros(4, 6), grid_coord=torch.zeros(4, 3, dtype=torch.int64), offset=torch.tensor([4])))
    assert seen == [overlap]
