"""The FP64 products behind the contractions, at the sizes where their tiling can go wrong:
contractions on both sides of the split over waves (31, 32, 33 values), output edges around
the 16- and 32-wide tiles, Λ scaling of the contracted index in each operand order, launches
with more products than travel by value, and one large enough for the 32 × 32 tiles.

Tolerance: the chains are left-canonical of norm 1, so every environment entry is at most 1
in modulus and a site step adds at most 2·d·χ rounding errors of ε to it; the sum over the n
sites bounds the value's error by 4·n·d·χ·ε (twice that for the values with spectra, whose
weights lie within [1/2, 1])."""
import numpy as np
import pytest

from oracle import chain as oc
from oracle import workloads as wl

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _chain(rng, n, chi, lam):
    arrays = wl.left_canonize_normalize(wl.random_mps_arrays(rng, n, 2, wl.max_profile(n, 2, chi)))
    lams = [0.5 + 0.5 * rng.random(a.shape[2]) if lam else None for a in arrays[:-1]]
    return arrays, lams


@pytest.mark.parametrize("lam", [False, True])
@pytest.mark.parametrize("chia,chib", [(1, 3), (15, 16), (16, 17), (31, 32), (33, 31), (47, 65), (130, 40)])
def test_overlap_at_tile_edges(qh, chia, chib, lam):
    rng = np.random.default_rng([chia, chib, lam])
    n = 18
    (a, la), (b, lb) = _chain(rng, n, chia, lam), _chain(rng, n, chib, lam)
    got = qh.overlap(qh.from_internal(a, lambdas=la), qh.from_internal(b, lambdas=lb))
    want = oc.overlap(oc.Chain([x.copy() for x in a], list(la)), oc.Chain([x.copy() for x in b], list(lb)))
    assert abs(got - want) < (2 if lam else 1) * 4 * n * 2 * max(chia, chib) * EPS


@pytest.mark.parametrize("n,chi", [(7, 5), (14, 33), (13, 48)])
def test_expect_many_at_tile_edges(qh, n, chi):
    rng = np.random.default_rng([n, chi])
    a, la = _chain(rng, n, chi, True)
    psi, ref = qh.from_internal(a, lambdas=la), oc.Chain([x.copy() for x in a], list(la))
    sites = [(i,) for i in range(1, n + 1)] + [(i, i + 2) for i in range(1, n - 1)]
    got = qh.expect_many(psi, [[qh.gate(wl.Z, i) for i in t] for t in sites])
    want = [oc.expect(ref, [oc.gate1(wl.Z, i) for i in t]) for t in sites]
    assert np.max(np.abs(got - np.array(want))) < 2 * 4 * n * 2 * chi * EPS


def test_norm_with_large_tiles(qh):
    """2 × 1024 columns and 1024 rows: 32 × 32 tiles."""
    rng = np.random.default_rng(5)
    n, chi = 22, 1024
    dims = [1] + wl.max_profile(n, 2, chi) + [1]
    a = [rng.standard_normal((dims[i], 2, dims[i + 1])) / np.sqrt(2 * dims[i]) + 0j for i in range(n)]
    got = qh.norm(qh.from_internal(a))
    want = oc.norm(oc.Chain(a))
    assert abs(got - want) < 4 * n * 2 * chi * EPS * want
