"""Overlaps and expectation values from both ends of a chain: 2 to 5 sites, bonds on either side
of the closing product's 32 × 32 tile, operators on every site and pair of neighbours.

Against numpy's contraction of the same arrays; both sum at most n·d·χ² products per value, so
they agree to 8·n·√(d·χ²)·ε of the norms' product."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _arrays(rng, chi, d):
    dims = [1, *chi, 1]
    return [(rng.standard_normal((dims[i], d, dims[i + 1])) + 1j * rng.standard_normal((dims[i], d, dims[i + 1])))
            / np.sqrt(2 * d * dims[i]) for i in range(len(dims) - 1)]


def _sandwich(ket, bra, ops=None):
    e = np.ones((1, 1), complex)
    for i, (a, b) in enumerate(zip(ket, bra)):
        if ops and i in ops:
            a = np.einsum("uv,lvr->lur", ops[i], a)
        e = np.tensordot(b.conj(), np.tensordot(e, a, (1, 0)), ((0, 1), (0, 1)))
    return e[0, 0]


@pytest.mark.parametrize("chi,chib", [([1], [1]), ([5], [7]), ([31, 32], [33, 2]), ([33, 65, 31], [32, 64, 1]),
                                      ([40, 70, 100, 33], [64, 96, 31, 65])])
def test_overlap(qh, chi, chib):
    rng = np.random.default_rng([len(chi), *chi])
    d = 2
    ka, kb = _arrays(rng, chi, d), _arrays(rng, chib, d)
    ctx = qh.Context()
    a, b = qh.from_internal(ka, context=ctx), qh.from_internal(kb, context=ctx)
    n, top = len(chi) + 1, max(*chi, *chib)
    na, nb = np.sqrt(_sandwich(ka, ka).real), np.sqrt(_sandwich(kb, kb).real)
    tol = 8 * n * np.sqrt(d * top * top) * EPS
    assert abs(qh.norm(a) - na) <= tol * na
    want = _sandwich(ka, kb)
    assert min(abs(qh.overlap(a, b) - want), abs(qh.overlap(b, a) - want)) <= tol * na * nb


@pytest.mark.parametrize("site", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("two", [False, True])
def test_expect(qh, site, two):
    if two and site == 5:
        pytest.skip("no second site")
    rng = np.random.default_rng([site, two])
    chi = [33, 40, 65, 31]
    arrays = _arrays(rng, chi, 2)
    psi = qh.from_internal(arrays, context=qh.Context())
    z = np.diag([1.0, -1.0]).astype(complex)
    terms = [qh.gate(z, site)] + ([qh.gate(z, site + 1)] if two else [])
    ops = {site - 1: z, **({site: z} if two else {})}
    norm2 = _sandwich(arrays, arrays).real
    tol = 8 * 5 * np.sqrt(2 * 65 * 65) * EPS
    assert abs(qh.expect(psi, terms) - _sandwich(arrays, arrays, ops)) <= tol * norm2
    many = qh.expect_many(psi, [terms, terms[:1]])
    assert abs(many[0] - _sandwich(arrays, arrays, ops)) <= tol * norm2
