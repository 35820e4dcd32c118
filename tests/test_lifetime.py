"""A context outlives the chains and operators in its memory, also where the garbage collector
finds them in one cycle (an exception that is kept holds the frames with both).  The
library is stood in for by a recorder of its calls."""
import gc

import pytest


class _Recorder:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            if name in ("qh_ctx_destroy", "qh_mps_free", "qh_mpo_free"):
                self.calls.append(name)
            return 0

        return call


@pytest.mark.parametrize("kind", ["chain", "mpo"])
@pytest.mark.parametrize("first", ["context", "object"])
def test_context_is_destroyed_last(monkeypatch, kind, first):
    import qrochet_hip as qh
    from qrochet_hip import _lib, mpo

    lib = _Recorder()
    monkeypatch.setattr(_lib, "load", lambda: lib)
    ctx = qh.Context()
    obj = qh.Chain(1, ctx) if kind == "chain" else mpo.MPOChain(1, ctx, 2, 2, [1])
    cycle = [ctx, obj] if first == "context" else [obj, ctx]
    cycle.append(cycle)
    del ctx, obj, cycle
    for _ in range(3):
        gc.collect()
    assert lib.calls == ["qh_mps_free" if kind == "chain" else "qh_mpo_free", "qh_ctx_destroy"]
