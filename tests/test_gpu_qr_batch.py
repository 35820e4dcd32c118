"""The batched Householder QR on a ragged batch: matrices of different heights above and below
1024 rows (the height up to which panels are held in registers; above it a launch per panel
and one for its update) go through one series of steps, and each of them gets the same bits as
alone.

Updates of 4-site chains with all bonds χ give θ of 2χ × 2χ; an SVD of more than 32 columns
takes three QR passes and one that recovers a factor, whatever the batch: the timing class
`qr` counts a series per pass."""
import numpy as np
import pytest

from oracle import workloads as wl

pytestmark = pytest.mark.gpu


def _layer(qh, chis, arrays, gates):
    ctx = qh.Context()
    ups = [(qh.from_internal(arrays[c], context=ctx), qh.gate(gates[c], 2, 3)) for c in chis]
    ctx.set_timing(True)
    qh.evolve_layer_(ups, maxdim=100, context=ctx)
    ctx.synchronize()
    ctx.set_timing(False)
    return [(psi.lambda_(2), psi.internal_arrays()) for psi, _ in ups], ctx.timing("qr")["launches"]


def test_ragged_heights_share_their_steps(qh):
    chis = [560, 90, 514, 520, 601]
    rng = np.random.default_rng(12)
    arrays = {c: wl.random_mps_arrays(rng, 4, 2, [c, c, c]) for c in chis}
    gates = {c: wl.haar_gate4(rng) for c in chis}
    batch, series = _layer(qh, chis, arrays, gates)
    for c, (lam, sites) in zip(chis, batch):
        [(lam1, sites1)], series1 = _layer(qh, [c], arrays, gates)
        assert np.array_equal(lam, lam1), c
        for x, y in zip(sites, sites1):
            assert np.array_equal(x, y), c
        assert series == series1, c
