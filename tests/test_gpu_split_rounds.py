"""Jacobi rounds in three launches (Gram, eigensolver, update, where pairs of more than 256 rows
are fewer than the compute units) against rounds in one (QH_JACOBI_SPLIT=0, read when a
context is created; QH_JACOBI_DEFER_V is an older name of the same switch): the same bits from
a third of the launches."""
import numpy as np
import pytest

from oracle import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["QH_JACOBI_SPLIT", "QH_JACOBI_DEFER_V"])
def test_same_bits(qh, monkeypatch, name):
    rng = np.random.default_rng(31)
    arrays = wl.random_mps_arrays(rng, 4, 2, [150, 150, 150])
    g = wl.haar_gate4(rng)
    runs = []
    for value in ("1", "0"):
        monkeypatch.setenv(name, value)
        ctx = qh.Context()
        psi = qh.from_internal(arrays, context=ctx)
        ctx.set_timing(True)
        qh.evolve_(psi, qh.gate(g, 2, 3), maxdim=200)
        ctx.synchronize()
        ctx.set_timing(False)
        runs.append((ctx.timing("jacobi_round")["launches"], psi.lambda_(2), psi.internal_arrays()))
    (n3, lam, sites), (n1, lam1, sites1) = runs
    assert n3 == 3 * n1
    assert np.array_equal(lam, lam1)
    assert all(np.array_equal(x, y) for x, y in zip(sites, sites1))
