"""Arrays read back from device memory on both sides of the size up to which the device stores
them itself (512 doubles), again and again between calls that use the same memory: the bytes
that went in come out."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chi", [1, 3, 255, 256, 511, 512, 513, 1100])
def test_bytes(qh, chi):
    rng = np.random.default_rng(chi)
    lam = np.sort(rng.random(chi))[::-1].copy()
    a = rng.standard_normal((1, 2, chi)) + 1j * rng.standard_normal((1, 2, chi))
    b = rng.standard_normal((chi, 2, 1)) + 1j * rng.standard_normal((chi, 2, 1))
    psi = qh.from_internal([a, b], lambdas=[lam], context=qh.Context())
    for _ in range(20):
        assert np.array_equal(psi.lambda_(1), lam)
        left, right = psi.copy().internal_arrays()
        assert np.array_equal(left, a) and np.array_equal(right, b)


def test_many_calls(qh, monkeypatch):
    """Descriptors of hundreds of calls through an arena of 4 KB: recycled many times over."""
    monkeypatch.setenv("QH_ARENA_INITIAL_BYTES", "4096")
    ctx = qh.Context()
    rng = np.random.default_rng(0)
    arrays = [rng.standard_normal(s) + 0j for s in ((1, 2, 2), (2, 2, 4), (4, 2, 2), (2, 2, 1))]
    psi = qh.from_internal(arrays, context=ctx)
    want = qh.overlap(psi, psi)
    for _ in range(300):
        assert qh.overlap(psi, psi.copy()) == want
