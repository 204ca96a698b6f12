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


# Orders with one outer block and with two, one after the other (both start with at least 8192 rows left).
# Stops in the first, a later and the last panel of an outer block and behind the last outer block.
@pytest.mark.parametrize("uplo", [0, 1])
@pytest.mark.parametrize("n,pad,fails", [
    (8192, 0, (10, 2 * 128 + 10, 8192 - 10, 8192 - 256 + 10)),
    (8300, 1, (10, 2 * 128 + 10, 8300 - 10, 63 * 128 + 10)),
    (8748, 0, (3 * 128 + 10, 512 + 10, 512 + 128 + 10, 512 + 384 + 10, 1024 + 10)),
])
def test_outer_blocks(dev, n, pad, fails, uplo, dtype=torch.float64):
    H = hpd(n, dtype, n)
    for fail in (None,) + fails:
        print("[case]", n, pad, uplo, fail, flush=True)
        A = H.clone()
        if fail is not None:
            A[fail, fail] = -1e6
        a, b = colmajor(dev, A, pad), colmajor(dev, A, pad)
        ia, ib = dev.potrf(a, uplo=uplo, nb=128), dev.potrf(b, uplo=uplo, nb=64)
        assert int(ia.item()) == int(ib.item()) == (0 if fail is None else fail + 1)
        # the columns finished before the failing 128-column panel and those right of it (the panel itself
        # stops at a block edge of its own)
        p, c = (n, n) if fail is None else (fail // 128 * 128, fail // 128 * 128 + 128)
        if fail is not None and fail % 128 >= 64:
            continue  # the 64-column blocks complete half a panel more
        x, y = (a.t(), b.t()) if uplo == 0 else (a, b)  # row j: the entries of column (row) j
        assert fail is None or c < n
        for part in (slice(0, p), slice(c, n)):
            u, v = x[part], y[part]
            if u.numel() == 0:
                continue
            if uplo == 0:
                assert torch.equal(u, v)
            else:
                assert float((u - v).abs().max()) <= 8 * n * 2.0 ** -53 * float(v.abs().max())
