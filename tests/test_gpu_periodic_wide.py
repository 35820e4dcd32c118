"""Periodic chains whose wrap bonds give enough passenger indices (at least 64 pairs) for the
contraction to run over all of them in one product: at the edge (7·9 = 63, 8·8 = 64, 8·9),
with bonds around the products' tiles, operators over one and two sites, Λ on a bond, and one
chain large enough (529 pairs, bonds of 48 and 61) for the products of 128 × 32 tiles.

Against the dense state of five sites, ψ(s) = tr Π A_i(s_i).  The value is the trace of a product
of n transfer matrices of P rows; each adds about √(d·χ²)·ε to it in Frobenius norm and the trace
takes √P of that: 8·n·√(d·χ²·P)·ε of the norms' product."""
import numpy as np
import pytest

from oracle import chain as oc
from oracle import workloads as wl

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _state(qh, ctx, rng, w, chi):
    dims = [w, *chi, w]
    arrays = [(rng.standard_normal((2, dims[i], dims[i + 1])) + 1j * rng.standard_normal((2, dims[i], dims[i + 1])))
              / np.sqrt(4 * dims[i]) for i in range(5)]
    psi = qh.pMPS(arrays, context=ctx)
    qh.evolve_(psi, qh.gate(wl.haar_gate4(rng), 3, 4), maxdim=chi[2])  # (leaves Λ on bond 3)
    return psi, oc.statevector(oc.Chain(psi.internal_arrays(), psi.lambdas(), periodic=True)).reshape([2] * 5)


@pytest.mark.parametrize("wk,chik,wb,chib", [(7, [5, 17, 16, 6], 9, [5, 16, 17, 3]), (8, [8, 15, 16, 8], 8, [3, 4, 33, 9]),
                                             (8, [31, 32, 33, 40], 9, [40, 17, 31, 7]), (12, [12, 65, 20, 1], 12, [2, 33, 64, 30]),
                                             (23, [48, 61, 61, 48], 23, [48, 61, 48, 20])])
def test_values(qh, wk, chik, wb, chib):
    rng = np.random.default_rng([wk, wb, *chik])
    ctx = qh.Context()
    a, va = _state(qh, ctx, rng, wk, chik)
    b, vb = _state(qh, ctx, rng, wb, chib)
    na, nb = np.linalg.norm(va), np.linalg.norm(vb)

    def tol(w, v, top):
        return 8 * 5 * np.sqrt(2.0 * top * top * w * v) * EPS

    assert abs(qh.norm(a) - na) <= tol(wk, wk, max(chik)) * na
    want, t = np.vdot(vb, va), tol(wk, wb, max(*chik, *chib)) * na * nb
    assert abs(qh.overlap(a, b) - want) <= t  # <b|a>
    assert abs(qh.overlap(b, a) - np.conj(want)) <= t
    z, x = np.diag([1.0, -1.0]).astype(complex), np.array([[0, 1], [1, 0]], complex)
    t = tol(wk, wk, max(chik)) * na * na
    ops = np.einsum("abcde,bB,dD,aBcDe->", va.conj(), z, x, va)
    assert abs(qh.expect(a, [qh.gate(z, 2), qh.gate(x, 4)]) - ops) <= t
    g = wl.haar_gate4(rng)
    both = np.einsum("abcde,cdCD,abCDe->", va.conj(), g, va)
    assert abs(qh.expect(a, [qh.gate(g, 3, 4)]) - both) <= t
