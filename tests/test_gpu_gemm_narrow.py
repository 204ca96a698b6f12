"""C := C -+ A B for at most 16 columns and depth <= 128 runs a 16 x 16 tile per wave; each entry is
one FMA chain over ascending k, so it equals the same columns of a wider product bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("alpha", [-1.0, 1.0])
def test_narrow_equals_wide(dev, dtype, alpha):
    rng = np.random.default_rng(4)
    for m in (1, 15, 64, 65, 1000):
        for n in (1, 3, 16):
            for k in (1, 5, 72, 127, 128):
                print("[case]", m, n, k, alpha, dtype.__name__, flush=True)
                A = rng.standard_normal((m, k)).astype(dtype)
                B = rng.standard_normal((k, 40)).astype(dtype)
                C = rng.standard_normal((m, 40)).astype(dtype)
                wide, part = dev.to_device(C), dev.to_device(C)
                dA, dB = dev.to_device(A), dev.to_device(B)
                dev.gemm(0, 0, alpha, dA, dB, 1.0, wide)
                dev.gemm(0, 0, alpha, dA, dB[:, :n], 1.0, part[:, :n])
                assert np.array_equal(dev.to_host(part)[:, :n], dev.to_host(wide)[:, :n])
                assert np.array_equal(dev.to_host(part)[:, n:], C[:, n:])
