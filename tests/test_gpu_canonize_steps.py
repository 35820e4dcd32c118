"""How many factorisations a canonical form takes where a chain has bonds too wide for the site on
either side: bond 3 (30) for site 4 (at most 4 to its right), which the sweep from the right cuts
down, and bond 1 (5) for site 1 (2 to its left), which leaves the rest to the sweep of SVDs.

`canonize!` is one sweep from the right and that sweep of SVDs.  From the chain that
`canonize_site!` steps leave, it is the same with a sweep whose sites are all tall (a QR each), so
the two differ by the steps' own QRs less one for each of sites 2..n (the timing class `qr`
counts the series)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _series(ctx, f):
    ctx.reset_timing()
    ctx.set_timing(True)
    f()
    ctx.synchronize()
    ctx.set_timing(False)
    return ctx.timing("qr")["launches"]


def test_one_sweep_from_the_right(qh):
    rng = np.random.default_rng(8)
    dims = [1, 5, 7, 30, 2, 1]
    n = len(dims) - 1
    arrays = [rng.standard_normal((dims[i], 2, dims[i + 1])) / np.sqrt(2 * dims[i]) + 0j for i in range(n)]
    ctx = qh.Context()
    psi, phi = (qh.from_internal(arrays, context=ctx) for _ in range(2))
    whole = _series(ctx, lambda: qh.canonize_(psi))
    steps = _series(ctx, lambda: [qh.canonize_site_(phi, s, direction="left", method="qr") for s in range(n, 1, -1)])
    rest = _series(ctx, lambda: qh.canonize_(phi))
    assert whole == steps + rest - (n - 1)
    for b in range(1, n):
        assert psi.lambda_(b).shape == phi.lambda_(b).shape
        assert np.allclose(psi.lambda_(b), phi.lambda_(b), rtol=0, atol=1e-13 * phi.lambda_(b)[0])
