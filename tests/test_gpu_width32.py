"""Block width 32 (`qh_ctx_set_jacobi`, 64-column pairs) on a θ of 2048 columns, and the default
width next to it: singular values against LAPACK, both new sites isometric."""
import numpy as np
import pytest

from oracle import chain as oc
from oracle import workloads as wl

pytestmark = pytest.mark.gpu


def test_width_32_and_default(qh):
    rng = np.random.default_rng(97)
    chi = 1024
    arrays = wl.random_mps_arrays(rng, 4, 2, [chi, chi, chi])
    g = wl.haar_gate4(rng)
    th = oc.theta(oc.Chain([a.copy() for a in arrays]), 2, g)
    cl, d, _, cr = th.shape
    s = np.linalg.svd(th.reshape(cl * d, d * cr), compute_uv=False)[:chi]
    for block in (32, 16):
        ctx = qh.Context()
        ctx.set_jacobi(block=block)
        psi = qh.from_internal(arrays, context=ctx)
        ctx.set_timing(True)
        qh.evolve_(psi, qh.gate(g, 2, 3), maxdim=chi)
        ctx.synchronize()
        ctx.set_timing(False)
        # (a sweep of 64-column pairs is 63 launches, one of 32-column pairs 3 · 127)
        per_sweep = ctx.timing("jacobi_round")["launches"] / ctx.timing("jacobi_sweep")["launches"]
        assert (per_sweep < 100) == (block == 32)
        a2, a3 = psi.internal_arrays()[1:3]
        u, vh = a2.reshape(-1, a2.shape[2]), a3.reshape(a3.shape[0], -1)
        assert np.max(np.abs(psi.lambda_(2) - s)) < 1e-12 * s[0]
        assert np.max(np.abs(u.conj().T @ u - np.eye(chi))) < 1e-11
        assert np.max(np.abs(vh @ vh.conj().T - np.eye(chi))) < 1e-11
