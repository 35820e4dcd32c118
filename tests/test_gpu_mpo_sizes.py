"""The FP64 MPO fit at the sizes where its products change form: sums over two indices of at least
32 values (split over four waves) with the first of them a multiple of four and not, across
the boundary between the two; orthonormalised sites of several QR panels, turned round with
their rows reordered; and bonds of 520, whose right factors have more than 1024 rows.

The oracle is the same fit in numpy; the device's rounding differs in each of the 2·n site
steps of a sweep by at most about √(D·d·χ²)·ε relative, so state and overlap agree to
8·2·n·√(2·D·d·χ²)·ε of the norm of φ for the states, and of its square for the overlap."""
import numpy as np
import pytest

from oracle import chain as oc
from oracle import mpo as om
from oracle import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,chi,D", [(9, 11, 3), (9, 15, 5), (10, 16, 3), (10, 17, 4), (11, 29, 5), (12, 33, 3),
                                     (12, 36, 6), (13, 48, 5), (14, 65, 2), (22, 520, 2)])
def test_fit(qh, n, chi, D):
    from qrochet_hip import mpo as qm

    rng = np.random.default_rng([n, chi, D])
    ref = oc.Chain(wl.left_canonize_normalize(wl.random_mps_arrays(rng, n, 2, wl.max_profile(n, 2, chi))))
    marr = om.random_hermitian_mpo(rng, n, 2, D)
    phi_ref, ov_ref = om.fit(om.from_arrays(marr), ref, ref.copy(), sweeps=1)
    phi, ov = qm.compress(qm.MPO(marr), qh.from_internal([a.copy() for a in ref.arrays]), sweeps=1)
    assert phi.bond_dims() == phi_ref.bond_dims()
    v, w = oc.statevector(oc.Chain(phi.internal_arrays())), oc.statevector(phi_ref)
    norm = np.linalg.norm(w)
    tol = 8 * 2 * n * np.sqrt(2 * D * 2 * chi * chi) * np.finfo(float).eps
    print(f"n={n} chi={chi} D={D}: state {np.linalg.norm(v - w) / norm:.1e}, value {abs(ov - ov_ref[-1]) / norm**2:.1e}, "
          f"bound {tol:.1e}")
    assert np.linalg.norm(v - w) <= tol * norm
    assert abs(ov - ov_ref[-1]) <= tol * norm**2
