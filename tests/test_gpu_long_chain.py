"""The canonical form of a chain of 65,600 sites, more bonds than a launch grid's second
dimension holds workgroups.

A product of unit vectors: every Λ is 1 and every Γ the site's vector up to a phase.  Each of
the n factorisations a value passes through adds a few ε to it: 8·n·ε."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_product_state(qh):
    n = 65600
    rng = np.random.default_rng(3)
    v = rng.standard_normal((n, 2)) + 1j * rng.standard_normal((n, 2))
    v /= np.linalg.norm(v, axis=1)[:, None]
    psi = qh.from_internal([x.reshape(1, 2, 1) for x in v], context=qh.Context())
    qh.canonize_(psi)
    tol = 8 * n * np.finfo(float).eps
    for s in (1, 2, 3, 1000, n // 2, n // 2 + 1, 65537, n - 1, n):
        got = psi.site_array(s).reshape(-1)
        assert abs(abs(np.vdot(v[s - 1], got)) - 1) <= tol, s
        assert abs(np.linalg.norm(got) - 1) <= tol, s
    for b in (1, 2, n // 2, 65536, n - 1):
        assert np.abs(psi.lambda_(b) - 1).max() <= tol, b
