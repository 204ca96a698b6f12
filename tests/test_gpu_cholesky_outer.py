"""The Cholesky's 512-column outer blocks (FP64, orders from 8192) against 64-column blocks, which have no
outer blocks. Every entry of the lower factor receives the same FMAs in column order and one
multiplication by a reciprocal whatever the blocking: bit for bit. The upper form divides in its
triangular solves and multiplies in its diagonal blocks (as the reference BLAS does), so there the
blocking changes roundings and the bar is the factorizations' 8 n u. When a pivot fails inside an
outer block, the columns right of it hold the updates of the panels completed before the failing
one, as the reference leaves them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def hpd(n, dtype, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    G = torch.randn(n, n, dtype=torch.float64, device="cuda", generator=g)
    H = G @ G.t() / n
    H.diagonal().add_(1.0)
    return (torch.tril(H) + torch.tril(H, -1).t()).to(dtype)


def colmajor(dev, a, pad):
    n = a.shape[0]
    t = torch.zeros((n, n + pad), dtype=a.dtype, device="cuda").t()[:n]
    t.copy_(a)
    return t


@pytest.mark.parametrize("uplo", [0, 1])
@pytest.mark.parametrize("n,pad", [(8192, 0), (8300, 1)])
def test_outer_blocks(dev, n, pad, uplo, dtype=torch.float64):
    H = hpd(n, dtype, n)
    # a clean factorization, and stops in the first and a later panel of an outer block
    for fail in (None, 10, 2 * 128 + 10, n - 10):
        print("[case]", n, pad, uplo, fail, flush=True)
        A = H.clone()
        if fail is not None:
            A[fail, fail] = -1e6
        a, b = colmajor(dev, A, pad), colmajor(dev, A, pad)
        ia, ib = dev.potrf(a, uplo=uplo, nb=128), dev.potrf(b, uplo=uplo, nb=64)
        assert int(ia.item()) == int(ib.item()) == (0 if fail is None else fail + 1)
        # right of the failing 128-column panel (the panel itself stops at a block edge of its own)
        c = 0 if fail is None else fail // 128 * 128 + 128
        if fail is not None and fail % 128 >= 64:
            continue  # the 64-column blocks complete half a panel more
        x, y = (a.t(), b.t()) if uplo == 0 else (a, b)  # row j: the entries of column (row) j
        if uplo == 0:
            assert torch.equal(x[c:, c:], y[c:, c:])
        else:
            x, y = x[c:, c:], y[c:, c:]
            if y.numel():
                assert float((x - y).abs().max()) <= 8 * n * 2.0 ** -53 * float(y.abs().max())
