"""Both factors of the batched SVD as `evolve!` gets them (no refinement step): the factor that is
recovered by a product and a QR is the left one for an odd number of preconditioning passes
and the right one for an even number, and changes sides once more where θ is wider than tall.

θ is any matrix M: the left site holds an identity from (l, o) to the bond, the right one M, and
the gate is the identity.  U and V^H are the new sites.  Checked: Σ against LAPACK to
4·√(rows·cols)·ε·σ₁, U Σ V^H = M to 8·√(rows·cols)·ε·‖M‖_F, and both isometries: the rotations
stop where any two columns' cosine is below 16·√p·ε, so ‖W^H W − 1‖_F ≤ 16·√p·ε·k, with p the
longer and k the shorter side; the recovered side is orthonormal to rounding, well within."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _matrix(rng, rows, cols, kind):
    def g(a, b):
        return (rng.standard_normal((a, b)) + 1j * rng.standard_normal((a, b))) / np.sqrt(2 * a)

    k = min(rows, cols)
    if kind == "flat":
        return g(rows, cols)
    if kind == "graded":  # 1 to 1e-14
        return (g(rows, k) * 10.0 ** (-14 * np.arange(k) / max(k - 1, 1))) @ g(k, cols)
    if kind == "columns":
        return g(rows, cols) * 10.0 ** (-12 * rng.permutation(cols) / max(cols - 1, 1))
    return g(rows, max(1, k // 3)) @ g(max(1, k // 3), cols)


def _check(qh, cl, cr, kind, passes):
    rng = np.random.default_rng([cl, cr, passes, len(kind)])
    rows, cols = 2 * cl, 2 * cr
    m = _matrix(rng, rows, cols, kind)
    ctx = qh.Context()
    ctx.set_qr_passes(passes)
    ends = [np.ones((1, 2, cl), complex), np.ones((cr, 2, 1), complex)]
    psi = qh.from_internal([ends[0], np.eye(rows, dtype=complex).reshape(cl, 2, rows), m.reshape(rows, 2, cr), ends[1]],
                           context=ctx)
    qh.evolve_(psi, qh.gate(np.eye(4, dtype=complex), 2, 3))
    arrays, lam = psi.internal_arrays(), psi.lambda_(2)
    k, p = min(rows, cols), max(rows, cols)
    u, vh = arrays[1].reshape(rows, -1), arrays[2].reshape(-1, cols)
    assert u.shape[1] == vh.shape[0] == lam.size == k
    s = np.linalg.svd(m, compute_uv=False)
    scale = np.sqrt(rows * cols) * EPS
    assert np.max(np.abs(lam - s)) <= 4 * scale * s[0]
    assert np.linalg.norm((u * lam) @ vh - m) <= 8 * scale * np.linalg.norm(m)
    assert np.linalg.norm(u.conj().T @ u - np.eye(k)) <= 16 * np.sqrt(p) * EPS * k
    assert np.linalg.norm(vh @ vh.conj().T - np.eye(k)) <= 16 * np.sqrt(p) * EPS * k


@pytest.mark.parametrize("passes", [0, 1, 2, 3, 4])
@pytest.mark.parametrize("kind", ["flat", "graded", "columns", "deficient"])
@pytest.mark.parametrize("cl,cr", [(24, 24), (40, 19), (19, 40)])
def test_passes(qh, cl, cr, kind, passes):
    _check(qh, cl, cr, kind, passes)


@pytest.mark.parametrize("kind", ["flat", "graded", "columns", "deficient"])
@pytest.mark.parametrize("cl,cr", [(1, 3), (7, 16), (16, 17), (9, 130), (130, 128), (60, 140), (257, 20), (20, 257),
                                   (130, 300), (513, 40), (40, 513)])
def test_sizes(qh, cl, cr, kind):
    _check(qh, cl, cr, kind, 3)
