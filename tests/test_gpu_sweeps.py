"""QR sweeps over a chain: lanes from both ends that share their launches, factors that are formed
a group at a time (28 sites of χ = 512 hold more than one group), rows in registers and in
memory (χ = 512 / 520: 1024 / 1040 rows), physical dimensions 2 and 3, and a chain with a bond
wider than its site is tall.

The state is checked by its overlap with the original, whose error is that of the contraction and
of a QR per site, at most about 8·√(rows·cols)·ε each, so 16·n·√(rows·cols)·ε relative; the
isometries by ‖Q^H Q − 1‖_F ≤ 8·√(rows·cols)·ε·√cols."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _chain(qh, chi, d, seed):
    rng = np.random.default_rng([seed, len(chi), d])
    dims = [1, *chi, 1]
    arrays = []
    for i in range(len(dims) - 1):
        shape = (dims[i], d, dims[i + 1])
        a = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
        arrays.append(a / np.sqrt(2 * d * dims[i]))
    return qh.from_internal(arrays, context=qh.Context())


def _ramp(n, d, top):
    return [min(top, d ** min(b, n - b, 40)) for b in range(1, n)]


def _check(qh, chi, d, center, seed):
    psi = _chain(qh, chi, d, seed)
    n = len(chi) + 1
    phi = psi.copy()
    qh.mixed_canonize_(phi, center)
    size = d * max(chi) * max(chi)
    tol = 16 * n * np.sqrt(size) * EPS
    a, b, ab = qh.norm(psi), qh.norm(phi), qh.overlap(psi, phi)
    assert abs(a - b) <= tol * a
    assert abs(ab - a * b) <= tol * a * b
    arrays = phi.internal_arrays()
    for s in range(1, n + 1):
        if s == center:
            continue
        m = arrays[s - 1]
        q = m.reshape(-1, m.shape[2]) if s < center else m.reshape(m.shape[0], -1).conj().T
        k = q.shape[1]
        assert np.linalg.norm(q.conj().T @ q - np.eye(k)) <= 8 * np.sqrt(q.size) * EPS * np.sqrt(k), s


@pytest.mark.parametrize("center", [2, 5, 6, 9])
@pytest.mark.parametrize("d,top", [(2, 7), (2, 12), (3, 30)])
def test_mixed(qh, d, top, center):
    _check(qh, _ramp(9, d, top), d, center, 1)


@pytest.mark.parametrize("chi", [[2, 3, 5, 4, 2], [1, 2, 1, 2], [2, 40, 3, 2], [30, 30, 30]])
def test_odd_bonds(qh, chi):
    _check(qh, chi, 2, 3, 2)


def test_groups(qh):
    _check(qh, _ramp(28, 2, 512), 2, 17, 3)


def test_rows_in_memory(qh):
    _check(qh, _ramp(23, 2, 520), 2, 12, 4)


@pytest.mark.parametrize("n,top", [(21, 500), (19, 250), (17, 100), (23, 520)])
def test_partial_panels(qh, n, top):
    """The last panel's 4 to 10 columns, factored behind an update by every wave: each site on
    its own, three times over, gives the same bits."""
    psi = _chain(qh, _ramp(n, 2, top), 2, 6)
    first = None
    for _ in range(3):
        phi = psi.copy()
        for s in range(1, n // 2 + 1):
            qh.canonize_site_(phi, s, direction="right", method="qr")
        arrays = phi.internal_arrays()
        if first is None:
            first = arrays
            tol = 16 * n * np.sqrt(2 * top * top) * EPS
            a, ab = qh.norm(psi), qh.overlap(psi, phi)
            assert abs(ab - a * a) <= tol * a * a
        assert all(np.array_equal(x, y) for x, y in zip(arrays, first))


def test_canonical_form_groups(qh):
    chi = _ramp(28, 2, 512)
    psi = _chain(qh, chi, 2, 5)
    phi = psi.copy()
    qh.canonize_(phi)
    tol = 16 * 28 * np.sqrt(2 * 512 * 512) * EPS
    a, b, ab = qh.norm(psi), qh.norm(phi), qh.overlap(psi, phi)
    assert abs(a - b) <= tol * a
    assert abs(ab - a * b) <= tol * a * b


@pytest.mark.parametrize("chi,d", [([2], 2), ([2, 2], 2), ([3, 2], 3), ([2, 4, 2], 2), ([2, 3, 4, 2], 2), ([1, 2, 1], 2),
                                   ([2, 4, 5, 3, 2], 2), ([3, 9, 17, 9, 3], 3), ([2, 4, 8, 16, 8, 4, 2], 2),
                                   ([4, 9, 4], 2), ([2, 9, 3, 2], 2)])
def test_canonical_form(qh, chi, d):
    """Λ against the singular values of the whole state's matrices, from lanes that meet at either
    kind of centre, with bonds wider than a site allows among them."""
    psi = _chain(qh, chi, d, 7)
    state = np.ones((1, 1), complex)
    for a in psi.internal_arrays():
        state = np.tensordot(state, a, (1, 0)).reshape(-1, a.shape[2])
    n, size = np.linalg.norm(state), len(chi) + 1
    tol = 16 * size * np.sqrt(state.size) * EPS * n
    phi = psi.copy()
    qh.canonize_(phi)
    for b in range(1, size):
        want = np.linalg.svd(state.reshape(d**b, -1), compute_uv=False)
        got = phi.lambda_(b)
        k = min(len(want), len(got))
        assert np.max(np.abs(got[:k] - want[:k])) <= tol
        assert np.all(got[k:] <= tol) and np.all(want[k:] <= tol)
    assert abs(qh.overlap(psi, phi) - n * n) <= tol * n
