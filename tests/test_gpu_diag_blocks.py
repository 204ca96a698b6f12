"""Diagonal-block kernels at the edges of their 16-entry blocks: the unblocked Cholesky (also where
it stops, and beside infinities) and triangular solves of order <= 128, bit for bit the oracle's."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 48, 127, 128])
def test_cholesky_block(dev, orc, n, dtype):
    rng = np.random.default_rng(n)
    G = rng.standard_normal((n, n))
    H = (G @ G.T / n + np.eye(n)).astype(dtype)
    H = np.tril(H) + np.tril(H, -1).T
    cases = [("hpd", H)]
    for j in sorted({0, n // 2, n - 1}):
        S = H.copy()
        S[j, j] = -1
        cases.append((f"stops at {j}", S))
    D = np.diag(np.arange(1, n + 1)).astype(dtype)  # exact zeros beside an infinity
    D[n - 1, 0] = D[0, n - 1] = np.inf
    cases.append(("inf beside zeros", D))
    for name, A in cases:
        for uplo in (0, 1):
            print("[case]", n, dtype.__name__, name, uplo, flush=True)
            F_ref, info_ref = orc.cholesky(A, uplo=uplo, bsize=128)
            dA = dev.to_device(A)
            info = dev.potrf(dA, uplo=uplo, nb=128)
            tri = np.tril if uplo == 0 else np.triu
            assert int(info.item()) == info_ref
            assert np.array_equal(tri(dev.to_host(dA)), tri(F_ref), equal_nan=True)


@pytest.mark.parametrize("side", [0, 1])
def test_trsm_block_edges(dev, orc, side):
    rng = np.random.default_rng(side)
    for order in (15, 16, 31, 113, 127, 128):
        for other in (4, 64, 65, 130):
            for uplo in (0, 1):
                for orient in (0, 1):
                    for diag in (0, 1):
                        print("[case]", side, order, other, uplo, orient, diag, flush=True)
                        T = rng.standard_normal((order, order)) / np.sqrt(order) + 2 * np.eye(order)
                        B = rng.standard_normal((order, other) if side == 0 else (other, order))
                        dB = dev.to_device(B)
                        dev.trsm(side, uplo, orient, diag, 1.0, dev.to_device(T), dB)
                        ref = orc.trsm("LR"[side], "LU"[uplo], "NT"[orient], "NU"[diag], 1.0,
                                       np.asfortranarray(T), np.asfortranarray(B))
                        assert np.array_equal(dev.to_host(dB), ref)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("order", [1, 2, 8, 33, 64, 128])
def test_trsm_block_small_orders_and_range(dev, orc, order, dtype):
    """Orders below and between the 16-entry blocks, vectors down to the smallest subnormals and
    divisors far from 1."""
    rng = np.random.default_rng(order)
    low, high = (-1070, 500) if dtype == np.float64 else (-146, 60)
    for other in (1, 5, 66):
        for spread in (0, 70 if dtype == np.float32 else 450):
            T = rng.standard_normal((order, order)) / order
            T[np.diag_indices(order)] = np.ldexp(1 + rng.random(order), rng.integers(-spread, spread + 1, order))
            T = T.astype(dtype)
            for side in (0, 1):
                V = np.ldexp(rng.standard_normal((order, other)), rng.integers(low, high, other))
                B = (V if side == 0 else V.T).astype(dtype)
                for uplo in (0, 1):
                    for orient in (0, 1):
                        for diag in (0, 1):
                            print("[case]", dtype.__name__, order, other, spread, side, uplo, orient, diag, flush=True)
                            dB = dev.to_device(np.ascontiguousarray(B))
                            dev.trsm(side, uplo, orient, diag, 1.0, dev.to_device(T), dB)
                            ref = orc.trsm("LR"[side], "LU"[uplo], "NT"[orient], "NU"[diag], 1.0,
                                           np.asfortranarray(T), np.asfortranarray(B))
                            assert np.array_equal(dev.to_host(dB), ref, equal_nan=True)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [1, 16, 17, 100, 128])
def test_factored_solves_of_one_block(dev, orc, n, dtype):
    """potrs and getrs of one block: the bits of their triangular solves, one after the other."""
    rng = np.random.default_rng(n)
    T = rng.standard_normal((n, n)) / n + 2 * np.eye(n)
    dT, dests = dev.to_device(T.astype(dtype)), None
    for nrhs in (1, 4, 5, 40):
        B = rng.standard_normal((n, nrhs)).astype(dtype)
        for name, forms in (("potrs lower", [(0, 0, 0), (0, 1, 0)]), ("potrs upper", [(1, 1, 0), (1, 0, 0)]),
                            ("getrs", [(0, 0, 1), (1, 0, 0)])):
            print("[case]", dtype.__name__, n, nrhs, name, flush=True)
            got, wide = dev.to_device(B), np.zeros((n, 130), dtype)
            wide[:, :nrhs] = B
            one = dev.to_device(wide)
            if name == "getrs":
                dev.getrs(dT, dests, got)
                dev.getrs(dT, dests, one)
            else:
                dev.potrs(dT, got, uplo=forms[0][0])
                dev.potrs(dT, one, uplo=forms[0][0])
            x = dev.to_host(got)
            assert np.array_equal(x, dev.to_host(one)[:, :nrhs])
            r = B.astype(np.float64)
            for uplo, orient, diag in reversed(forms):
                M = np.tril(T) if uplo == 0 else np.triu(T)
                M = M.astype(dtype).astype(np.float64)
                if diag:
                    M = M - np.diag(np.diag(M)) + np.eye(n)
                x = (M.T if orient else M) @ x
            u = np.finfo(dtype).eps / 2
            assert np.abs(x - r).max() <= 64 * n * u * np.abs(r).max()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_trsm_block_under_capture(dev, dtype):
    """The order-128 forms captured and replayed, eager solves between the replays."""
    rng = np.random.default_rng(3)
    dT = dev.to_device((rng.standard_normal((128, 128)) / 128 + 2 * np.eye(128)).astype(dtype))
    B = torch.from_numpy(rng.standard_normal((128, 70)).astype(dtype)).cuda()
    forms = [(uplo, orient, diag) for uplo in (0, 1) for orient in (0, 1) for diag in (0, 1)]
    outs = [dev.colmajor_empty(128, 70, B.dtype) for _ in forms]
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for out, (uplo, orient, diag) in zip(outs, forms):
            dev.trsm(0, uplo, orient, diag, 1.0, dT, out)
    for _ in range(3):
        for out in outs:
            out.copy_(B)
        g.replay()
        torch.cuda.synchronize()
        for out, (uplo, orient, diag) in zip(outs, forms):
            eager = dev.colmajor_empty(128, 70, B.dtype)
            eager.copy_(B)
            dev.trsm(0, uplo, orient, diag, 1.0, dT, eager)
            assert torch.equal(out, eager)
