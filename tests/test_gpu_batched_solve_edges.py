"""The batched Cholesky solve at the edges of its 16- and 32-row blocks and 8-column chunks.

The factors hold 1 or 2 on the diagonal and -1, 0 or 1 below it, the solutions small integers:
every product, sum and reciprocal of the two sweeps (cholesky::SolveAfter,
src/lapack_like/factor/Cholesky/SolveAfter.hpp:15-43) is exact in FP32, whatever its order, so the
solutions must come back bit for bit. The strict upper triangles hold NaN and the right-hand sides
lie in wider arrays of NaN: neither may be read or written."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def padded(dev, M, dtype, rows):
    """M as a column-major view with leading dimension rows + M's own, NaN all round."""
    n, m = M.shape
    buf = torch.full((m + 1, n + rows), float("nan"), dtype=dtype, device="cuda")
    buf[:m, :n] = torch.from_numpy(np.ascontiguousarray(M.T)).to(dtype)
    return buf, buf.t()[:n, :m]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_solve_edges(dev, dtype):
    rng = np.random.default_rng(16)
    Ls, Bs, Xs, bufs = [], [], [], []
    for n in (1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 95, 97, 128, 160, 161, 511, 512):
        for r in (1, 2, 7, 8, 9, 17):
            L = np.tril(rng.integers(-1, 2, (n, n)) * (rng.random((n, n)) < 8 / n), -1).astype(float)
            L += np.diag(rng.integers(1, 3, n))
            X = rng.integers(-3, 4, (n, r)).astype(float)
            Y = L.T @ X
            # the largest partial sum of either sweep stays an exact FP32 integer
            assert max((np.abs(L) @ np.abs(Y)).max(), (np.abs(L.T) @ np.abs(X)).max()) < 2 ** 23
            _, dL = padded(dev, L + np.triu(np.full((n, n), np.nan), 1), dtype, 1)
            buf, dB = padded(dev, L @ Y, dtype, 3)
            Ls.append(dL)
            Bs.append(dB)
            Xs.append(X)
            bufs.append(buf)
    dev.potrs_vbatched(dev.Batch(Ls, dtype), dev.Batch(Bs, dtype))
    torch.cuda.synchronize()
    for X, dB, buf in zip(Xs, Bs, bufs):
        n, r = X.shape
        print("[case]", dtype, n, r, flush=True)
        assert np.array_equal(dB.cpu().numpy().astype(float), X)
        assert torch.isnan(buf[r:]).all() and torch.isnan(buf[:, n:]).all()
