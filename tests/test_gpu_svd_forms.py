"""The batched SVD at the sizes where its form changes: with and without QR preconditioning
(32 / 33 columns), the Jacobi rounds in one launch or three (256 / 257 and 512 / 513 rows),
Gram sums over several row groups (1030 rows), the factor recovered by a QR on either side
(1 to 4 passes), for flat, graded and rank-deficient matrices.

`canonize_site!(…, :right; method = :svd)` factors the middle site of a three-site chain,
M = U Σ V^H (rows (l, o)).  Checked against LAPACK: Σ to 4·√(rows·cols)·ε·σ₁ (the backward
error of either factorisation is a small multiple of √(rows·cols)·ε·‖M‖ at most), U^H U = 1 to
8·cols·ε in Frobenius norm, and U Σ V^H = M (through the neighbour that V^H goes into) to
8·√(rows·cols)·ε·‖M‖_F."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _matrix(rng, rows, cols, kind):
    def g(a, b):
        return (rng.standard_normal((a, b)) + 1j * rng.standard_normal((a, b))) / np.sqrt(2 * a)

    if kind == "flat":
        return g(rows, cols)
    if kind == "graded":  # 1 to 1e-14
        k = min(rows, cols)
        return (g(rows, k) * 10.0 ** (-14 * np.arange(k) / max(k - 1, 1))) @ g(k, cols)
    k = max(1, min(rows, cols) // 3)
    return g(rows, k) @ g(k, cols)


def _check(qh, chil, chir, kind, passes=3):
    rng = np.random.default_rng([chil, chir, len(kind), passes])
    rows, cols = 2 * chil, chir
    m = _matrix(rng, rows, cols, kind)
    ctx = qh.Context()
    ctx.set_qr_passes(passes)
    # site 1 and site 3 are identities on their bonds, split over a physical index of 2
    first = np.zeros((1, 2, chil), complex)
    first[0, 0] = rng.standard_normal(chil)
    last = np.zeros((chir, 2, chir), complex)
    last[:, 0, :] = np.eye(chir)
    end = np.ones((chir, 2, 1), complex)
    psi = qh.from_internal([first, m.reshape(chil, 2, chir), last, end], context=ctx)
    qh.canonize_site_(psi, 2, direction="right", method="svd")
    arrays, lam = psi.internal_arrays(), psi.lambda_(2)
    k = min(rows, cols)
    u = arrays[1].reshape(rows, k)
    vh = arrays[2].reshape(k, 2, chir)[:, 0, :]
    s = np.linalg.svd(m, compute_uv=False)
    scale = np.sqrt(rows * cols) * EPS
    assert lam.shape == s.shape
    assert np.max(np.abs(lam - s)) <= 4 * scale * s[0]
    assert np.linalg.norm(u.conj().T @ u - np.eye(k)) <= 8 * k * EPS
    assert np.linalg.norm((u * lam) @ vh - m) <= 8 * scale * np.linalg.norm(m)


@pytest.mark.parametrize("kind", ["flat", "graded", "deficient"])
@pytest.mark.parametrize("chil,chir", [(1, 2), (9, 16), (16, 32), (17, 33), (300, 20), (515, 32), (24, 48), (130, 255),
                                       (129, 257), (256, 300)])
def test_svd_sizes(qh, chil, chir, kind):
    _check(qh, chil, chir, kind)


@pytest.mark.parametrize("chil,chir", [(256, 512), (257, 513), (515, 1030)])
def test_svd_tall(qh, chil, chir):
    _check(qh, chil, chir, "graded")


@pytest.mark.parametrize("passes", [1, 2, 3, 4])
@pytest.mark.parametrize("kind", ["flat", "graded", "deficient"])
def test_svd_passes(qh, kind, passes):
    _check(qh, 45, 70, kind, passes)
