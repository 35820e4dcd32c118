"""The sweep limit (`qh_ctx_set_jacobi`) holds for matrices of one block pair, which are solved in
one launch: a window of one sweep and a second of as many are too few for a generic matrix of
10 to 32 columns (one solve rotates, the next still finds something), and ten of them are
enough; alone, and next to a matrix of many pairs."""
import numpy as np
import pytest

from oracle import workloads as wl

pytestmark = pytest.mark.gpu


def _updates(qh, ctx, chis):
    rng = np.random.default_rng(21)
    return [(qh.from_internal(wl.random_mps_arrays(rng, 4, 2, [c, c, c]), context=ctx),
             qh.gate(wl.haar_gate4(rng), 2, 3)) for c in chis]


@pytest.mark.parametrize("chis", [[5], [8], [16], [3, 12, 7], [60, 16]])
def test_limit(qh, chis):
    ctx = qh.Context()
    ups = _updates(qh, ctx, chis)
    before = [psi.internal_arrays() for psi, _ in ups]
    ctx.set_jacobi(max_sweeps=1)
    with pytest.raises(qh.QHError, match="did not converge within 2 sweeps"):
        qh.evolve_layer_(ups, maxdim=max(chis), context=ctx)
    for (psi, _), arrays in zip(ups, before):  # (no state is written by a call that fails)
        assert all(np.array_equal(x, y) for x, y in zip(psi.internal_arrays(), arrays))
    ctx.set_jacobi(max_sweeps=10)
    kept, _ = qh.evolve_layer_(ups, maxdim=max(chis), context=ctx)
    assert kept == [min(2 * c, max(chis)) for c in chis]
