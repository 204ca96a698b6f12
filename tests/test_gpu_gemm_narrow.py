"""C := C -+ A B for at most 16 columns and depth <= 128 runs a 16 x 16 tile per wave; each entry is
one FMA chain over ascending k, so it equals the same columns of a wider product bit for bit."""
import numpy as np
import pytest
import torch

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


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n,k", [(1, 1, 5), (100, 4000, 7), (130, 1500, 33), (2100, 129, 50), (127, 300, 64),
                                   (1152, 1152, 64), (1300, 1300, 17), (1500, 1500, 127), (2100, 2100, 33),
                                   (3200, 3200, 16)])
def test_every_tile_of_a_ragged_product(dev, m, n, k, dtype):
    """Grids without whole tiles (K not a multiple of 16, or C smaller than one), and triangles whose
    last group of 8 tile rows has 1, 3, 4 or 8: whole-number operands, so the product is exact in any
    order, and every entry of C, inside the triangle only for syrk."""
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n + k)

    def ints(a, b):
        t = dev.colmajor_empty(a, b, dtype)
        t.copy_(torch.randint(-8, 9, (a, b), device="cuda", generator=g))
        return t

    for ta in (0, 1):
        for tb in (0, 1):
            print("[case]", m, n, k, dtype, ta, tb, flush=True)
            A, B, C = ints(*((k, m) if ta else (m, k))), ints(*((n, k) if tb else (k, n))), ints(m, n)
            want = C.cpu().double() - (A.t() if ta else A).cpu().double() @ (B.t() if tb else B).cpu().double()
            dev.gemm(ta, tb, -1.0, A, B, 1.0, C)
            assert torch.equal(C.cpu().double(), want)
        if m == n:
            for uplo in (0, 1):
                A, C = ints(*((k, m) if ta else (m, k))), ints(m, m)
                P = (A.t() if ta else A).cpu().double()
                full = C.cpu().double()
                mask = torch.ones(m, m).tril() if uplo == 0 else torch.ones(m, m).triu()
                want = torch.where(mask > 0, full - P @ P.t(), full)
                dev.syrk(uplo, ta, -1.0, A, 1.0, C)
                assert torch.equal(C.cpu().double(), want)
