"""The order of `overlap`'s arguments: overlap(a, b) = ⟨b|a⟩ (src/Ansatz/Chain.jl:737-748), its
conjugate in the other order, for contractions that start from both ends: an even and an odd
number of sites, different bonds on the two chains, with and without Λ.

Against numpy's contraction; both sum at most n·d·χ² products per value, so they agree to
8·n·√(d·χ²)·ε of the norms' product."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _state(rng, chi, lam):
    dims = [1, *chi, 1]
    arrays = [(rng.standard_normal((dims[i], 2, dims[i + 1])) + 1j * rng.standard_normal((dims[i], 2, dims[i + 1])))
              / np.sqrt(4 * dims[i]) for i in range(len(dims) - 1)]
    lams = [0.5 + 0.5 * rng.random(c) if lam else None for c in chi]
    v = np.ones((1, 1), complex)
    for i, a in enumerate(arrays):
        v = np.tensordot(v, a, (1, 0)).reshape(-1, a.shape[2])
        if lam and i < len(chi):
            v = v * lams[i]
    return arrays, lams, v[:, 0]


@pytest.mark.parametrize("lam", [False, True])
@pytest.mark.parametrize("chia,chib", [([3], [5]), ([4, 33], [7, 2]), ([2, 40, 9], [17, 31, 64]),
                                       ([16, 31, 33, 5], [3, 70, 32, 20])])
def test_order(qh, chia, chib, lam):
    rng = np.random.default_rng([len(chia), lam])
    ctx = qh.Context()
    (a, la, va), (b, lb, vb) = _state(rng, chia, lam), _state(rng, chib, lam)
    psi, phi = qh.from_internal(a, lambdas=la, context=ctx), qh.from_internal(b, lambdas=lb, context=ctx)
    top = max(*chia, *chib)
    tol = 8 * len(a) * np.sqrt(2 * top * top) * EPS * np.linalg.norm(va) * np.linalg.norm(vb)
    want = np.vdot(vb, va)
    for f in (qh.overlap, qh.overlap_noalloc):
        assert abs(f(psi, phi) - want) <= tol
        assert abs(f(phi, psi) - np.conj(want)) <= tol
