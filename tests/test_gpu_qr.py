"""The batched Householder QR at the sizes where its form changes: one to three row blocks of
16, four waves or eight (64 / 65 rows), a tile of four or eight blocks a wave (512 / 513), panels
of eight columns and of four in registers (1024 / 1026, 2048 / 2050 rows), panels in memory
(4096 / 4098), and a last panel of 1 to 16 columns.

`canonize_site!(…, :right; method = :qr)` factors the second site of a chain, M = Q R (rows
(l, o)), and R goes into the third, an identity.  Householder's backward error is a small
multiple of rows·cols·ε at the very worst and about √(rows·cols)·ε in practice: checked are
Q^H Q = 1 to 8·√(rows·cols)·ε in Frobenius norm per column, and Q R = M to
8·√(rows·cols)·ε·‖M‖_F."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


TALL = [(513, 5), (514, 8), (600, 9), (1024, 16), (1024, 31), (1025, 3), (1025, 21), (2048, 20), (2049, 18), (700, 120)]


@pytest.mark.parametrize("kind", ["flat", "zero-column", "scaled"])
@pytest.mark.parametrize("chil,chir", TALL)
def test_qr_tall(qh, chil, chir, kind):
    _check(qh, chil, chir, kind)


@pytest.mark.parametrize("kind", ["flat", "zero-column", "scaled"])
@pytest.mark.parametrize("chil,chir", [(1, 1), (1, 2), (8, 15), (8, 16), (9, 17), (16, 31), (32, 33), (33, 64),
                                       (64, 63), (128, 80), (129, 100), (256, 65), (257, 47), (512, 33), (513, 33)])
def test_qr_sizes(qh, chil, chir, kind):
    _check(qh, chil, chir, kind)


def _check(qh, chil, chir, kind):
    rng = np.random.default_rng([chil, chir, len(kind)])
    rows, cols = 2 * chil, chir
    m = rng.standard_normal((rows, cols)) + 1j * rng.standard_normal((rows, cols))
    if kind == "zero-column":
        m[:, cols // 2] = 0.0
    if kind == "scaled":
        m *= 10.0 ** (-12.0 * np.arange(cols) / max(cols - 1, 1))
    first = rng.standard_normal((1, 2, chil)).astype(complex)
    last = np.zeros((chir, 2, chir), complex)
    last[:, 0, :] = np.eye(chir)
    end = np.ones((chir, 2, 1), complex)
    psi = qh.from_internal([first, m.reshape(chil, 2, chir), last, end], context=qh.Context())
    qh.canonize_site_(psi, 2, direction="right", method="qr")
    arrays = psi.internal_arrays()
    k = min(rows, cols)
    q = arrays[1].reshape(rows, k)
    r = arrays[2].reshape(k, 2, chir)[:, 0, :]
    scale = np.sqrt(rows * cols) * EPS
    assert np.linalg.norm(q.conj().T @ q - np.eye(k)) <= 8 * scale * np.sqrt(k)
    assert np.linalg.norm(q @ r - m) <= 8 * scale * np.linalg.norm(m)


# A reflector takes refined estimates where the squared norm of its column lies between 1e-280 and
# 1e280, square root and divisions beyond: on both sides of the two limits, and across them
@pytest.mark.parametrize("power", [-145, -140, -138, 138, 139, 140, 145])
@pytest.mark.parametrize("chil,chir", [(1, 2), (16, 15), (33, 40), (130, 33), (600, 17)])
def test_qr_magnitudes(qh, chil, chir, power):
    rng = np.random.default_rng([chil, chir])
    rows, cols = 2 * chil, chir
    m = rng.standard_normal((rows, cols)) + 1j * rng.standard_normal((rows, cols))
    m *= 10.0 ** rng.uniform(-1.0, 1.0, cols)
    first = rng.standard_normal((1, 2, chil)).astype(complex)
    last = np.zeros((chir, 2, chir), complex)
    last[:, 0, :] = np.eye(chir)
    end = np.ones((chir, 2, 1), complex)
    psi = qh.from_internal([first, (m * 10.0 ** power).reshape(chil, 2, chir), last, end], context=qh.Context())
    qh.canonize_site_(psi, 2, direction="right", method="qr")
    arrays = psi.internal_arrays()
    k = min(rows, cols)
    q = arrays[1].reshape(rows, k)
    r = arrays[2].reshape(k, 2, chir)[:, 0, :] / 10.0 ** power
    scale = np.sqrt(rows * cols) * EPS
    assert np.linalg.norm(q.conj().T @ q - np.eye(k)) <= 8 * scale * np.sqrt(k)
    assert np.linalg.norm(q @ r - m) <= 8 * scale * np.linalg.norm(m)
