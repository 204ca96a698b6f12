"""The chained triangular solve (left side, order above 128, up to 128 right-hand sides): every
orientation at the edges of its 128-row blocks, 16-row sub-blocks and groups of 16 right-hand
sides. Substitution in any order satisfies |b - T x| <= gamma_n |T| |x| entry by entry
(gamma_n ~ n u); evaluating that residual in FP64 costs as much again, hence the factor 2."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def residual_ok(T, x, b, u):
    n = T.shape[0]
    r = np.abs(b - T @ x)
    return bool((r <= 2 * n * u * (np.abs(T) @ np.abs(x)) + np.finfo(np.float64).tiny).all())


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,nrhs,pad", [(129, 1, 0), (143, 16, 1), (256, 3, 2), (300, 17, 0),
                                        (1000, 1, 3), (1153, 33, 1), (2200, 128, 0)])
def test_all_orientations(dev, n, nrhs, pad, dtype):
    rng = np.random.default_rng(n)
    u = 2.0 ** -53 if dtype == np.float64 else 2.0 ** -24
    M = (rng.standard_normal((n, n)) / np.sqrt(n)).astype(dtype)
    M[np.arange(n), np.arange(n)] = (1.0 + rng.random(n)).astype(dtype)
    buf = torch.zeros((n, n + pad), dtype=torch.from_numpy(M).dtype, device="cuda")
    dM = buf.t()[:n]
    dM.copy_(torch.from_numpy(M))
    for uplo in (0, 1):
        for orient in (0, 1):
            for diag in (0, 1):
                print("[case]", n, nrhs, pad, dtype.__name__, uplo, orient, diag, flush=True)
                T = np.tril(M) if uplo == 0 else np.triu(M)
                if diag == 1:
                    T = T - np.diag(np.diag(T)) + np.eye(n, dtype=dtype)
                T = (T if orient == 0 else T.T).astype(np.float64)
                B = rng.standard_normal((n, nrhs)).astype(dtype)
                dB = dev.to_device(B)
                dev.trsm(0, uplo, orient, diag, 1.0, dM, dB)
                assert residual_ok(T, dev.to_host(dB).astype(np.float64), B.astype(np.float64), u)


def test_diagonal_out_of_the_quick_division_range(dev):
    """Diagonal entries near the ends of the exponent range are divided by as they are."""
    n = 200
    rng = np.random.default_rng(1)
    d = 2.0 ** rng.integers(-1000, 1000, n)
    B = rng.standard_normal((n, 2))
    dB = dev.to_device(B)
    dev.trsm(0, 0, 0, 0, 1.0, dev.to_device(np.diag(d)), dB)
    assert np.array_equal(dev.to_host(dB), B / d[:, None])


def test_captured_solves_replay(dev):
    """A captured lu::SolveAfter is replayed with new right-hand sides, eager solves between the
    replays: every replay matches the eager result bit for bit."""
    n = 700
    rng = np.random.default_rng(2)
    dA = dev.to_device(rng.standard_normal((n, n)))
    d, info = dev.getrf(dA)
    assert int(info.item()) == 0
    dB = dev.to_device(rng.standard_normal((n, 3)))
    dev.getrs(dA, d, dB)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        dev.getrs(dA, d, dB)
    for _ in range(4):
        B = rng.standard_normal((n, 3))
        eager = dev.to_device(B)
        dev.getrs(dA, d, eager)
        dB.copy_(torch.from_numpy(B))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(dB, eager)


def test_capture_that_would_have_to_allocate(dev):
    """A first solve of its size, under capture: it runs without the hand-off area's growth and
    replays to the eager result bit for bit."""
    n, r = 4400, 128
    rng = np.random.default_rng(3)
    dT = dev.to_device(np.tril(rng.standard_normal((n, n)) / n) + np.eye(n))
    B = torch.from_numpy(rng.standard_normal((n, r)))
    dB = dev.to_device(np.zeros((n, r)))
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        dev.trsm(0, 0, 0, 0, 1.0, dT, dB)
    for _ in range(3):
        dB.copy_(B)
        g.replay()
        eager = dev.to_device(B.numpy())
        torch.cuda.synchronize()
        dev.trsm(0, 0, 0, 0, 1.0, dT, eager)
        torch.cuda.synchronize()
        assert torch.equal(dB, eager)


def test_two_streams(dev):
    """Solves queued on two streams without any wait between them."""
    n = 1500
    rng = np.random.default_rng(4)
    dT = dev.to_device(np.tril(rng.standard_normal((n, n)) / n) + np.eye(n))
    B = rng.standard_normal((n, 2))
    want = dev.to_device(B)
    dev.trsm(0, 0, 0, 0, 1.0, dT, want)
    got = [dev.to_device(B) for _ in range(16)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for q, dB in enumerate(got):
        with torch.cuda.stream(streams[q % 2]):
            dev.trsm(0, 0, 0, 0, 1.0, dT, dB)
    torch.cuda.synchronize()
    for dB in got:
        assert torch.equal(dB, want)


def test_captured_branches_and_eager_solves_overlap(dev):
    """Two forked branches of one capture, replayed while eager solves run on another stream."""
    n = 1500
    rng = np.random.default_rng(5)
    dT = dev.to_device(np.tril(rng.standard_normal((n, n)) / n) + np.eye(n))
    B = torch.from_numpy(rng.standard_normal((n, 2))).cuda()
    want = dev.to_device(B.cpu().numpy())
    dev.trsm(0, 0, 0, 0, 1.0, dT, want)
    a, b = dev.colmajor_empty(n, 2), dev.colmajor_empty(n, 2)
    eager = [dev.colmajor_empty(n, 2) for _ in range(6)]
    side, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        cur = torch.cuda.current_stream()
        side.wait_stream(cur)
        dev.trsm(0, 0, 0, 0, 1.0, dT, a)
        with torch.cuda.stream(side):
            dev.trsm(0, 0, 0, 0, 1.0, dT, b)
        cur.wait_stream(side)
    for _ in range(4):
        for t in [a, b] + eager:
            t.copy_(B)
        torch.cuda.synchronize()
        g.replay()
        with torch.cuda.stream(other):
            for t in eager:
                dev.trsm(0, 0, 0, 0, 1.0, dT, t)
        torch.cuda.synchronize()
        for t in [a, b] + eager:
            assert torch.equal(t, want)


def test_eager_solve_beside_a_capture(dev):
    """An eager solve, the first of its size, on another stream while a capture is under way: the
    capture stays valid and both solve."""
    n, r = 12000, 128
    dT = dev.colmajor_empty(n, n)
    dT.copy_(torch.tril(torch.randn(n, n, dtype=torch.float64, device="cuda")) / n)
    dT.diagonal().fill_(1.0)
    small = dT[:700, :700]
    B = torch.randn(n, r, dtype=torch.float64, device="cuda")
    got, want, cap = dev.colmajor_empty(n, r), dev.colmajor_empty(n, r), dev.colmajor_empty(700, 2)
    got.copy_(B)
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        dev.trsm(0, 0, 0, 0, 1.0, small, cap)
        with torch.cuda.stream(other):
            dev.trsm(0, 0, 0, 0, 1.0, dT, got)
        dev.trsm(0, 0, 1, 0, 1.0, small, cap)
    torch.cuda.synchronize()
    want.copy_(B)
    dev.trsm(0, 0, 0, 0, 1.0, dT, want)
    assert torch.equal(got, want)
    ref = dev.to_device(B[:700, :2].cpu().numpy())
    dev.trsm(0, 0, 0, 0, 1.0, small, ref)
    dev.trsm(0, 0, 1, 0, 1.0, small, ref)
    for _ in range(3):
        cap.copy_(B[:700, :2])
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(cap, ref)


def test_a_wait_that_runs_out_is_reported(dev, monkeypatch):
    """With no poll allowed the blocks give up on each other: gesv and posv say so in their info word,
    and the next solves are whole again."""
    n = 2000
    rng = np.random.default_rng(6)
    A = rng.standard_normal((n, n))
    H = A @ A.T / n + np.eye(n)
    B = rng.standard_normal((n, 3))

    def solve():
        x, y = dev.to_device(B), dev.to_device(B)
        infos = [dev.gesv(dev.to_device(A), x), dev.posv(dev.to_device(H), y)]
        return [int(i.item()) for i in infos], x, y

    first, x0, y0 = solve()
    assert first == [0, 0]
    monkeypatch.setenv("ELX_SOLVE_SPIN_LIMIT", "0")
    lost, x, y = solve()
    assert lost == [-1, -1]
    assert bool(torch.isnan(x).any()) and bool(torch.isnan(y).any())
    monkeypatch.delenv("ELX_SOLVE_SPIN_LIMIT")
    again, x, y = solve()
    assert again == [0, 0] and torch.equal(x, x0) and torch.equal(y, y0)


@pytest.mark.parametrize("n,nrhs", [(128 * 256 + 1, 1), (128 * 40, 128)])
def test_more_blocks_than_workgroups(dev, n, nrhs):
    """Workgroups that take several blocks each, against a solve of the same system block by block
    (more than 128 columns): bit for bit."""
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    dT = dev.colmajor_empty(n, n, torch.float32)
    dT.copy_(torch.randn(n, n, dtype=torch.float32, device="cuda", generator=g) / n)
    dT.diagonal().add_(1.0)
    B = torch.randn(n, nrhs, dtype=torch.float32, device="cuda", generator=g)
    for uplo in (0, 1):
        wide, got = dev.colmajor_empty(n, 130, torch.float32), dev.colmajor_empty(n, nrhs, torch.float32)
        wide.zero_()
        wide[:, :nrhs] = B
        got.copy_(B)
        dev.trsm(0, uplo, 0, 0, 1.0, dT, wide)
        dev.trsm(0, uplo, 0, 0, 1.0, dT, got)
        assert torch.equal(got, wide[:, :nrhs])


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_divisions_at_the_ends_of_the_range(dev, dtype):
    """Right-hand sides near underflow and overflow, signed zeros and infinities, and divisors far from 1:
    the chained solve divides as the block by block one (more than 128 columns) does, bit for bit."""
    n = 300
    rng = np.random.default_rng(7)
    tiny, top = (-1060, 1020) if dtype == np.float64 else (-140, 125)
    exps = [tiny, tiny + 15, tiny + 30, tiny // 2, 0, top // 2, top - 20, top]
    B = np.stack([np.ldexp(rng.standard_normal(n), e) for e in exps] +
                 [np.zeros(n), -np.zeros(n), np.ldexp(rng.standard_normal(n), rng.integers(tiny, top, n))],
                 axis=1).astype(dtype)
    B[:, 10][rng.integers(0, n, 20)] = -0.0
    B = np.concatenate([B, B[:, 4:6]], axis=1)
    B[200, 11] = np.inf
    for spread in (0, 55, tiny // -2):
        T = np.tril(rng.standard_normal((n, n)) / n)
        T[np.arange(n), np.arange(n)] = np.ldexp(1.0 + rng.random(n), rng.integers(-spread, spread + 1, n))
        T[np.arange(0, n, 3), np.arange(0, n, 3)] *= -1
        dT = dev.to_device(T.astype(dtype))
        wide = np.zeros((n, 130), dtype)
        wide[:, :B.shape[1]] = B
        for orient in (0, 1):
            for cols in (3, B.shape[1]):
                dB, dW = dev.to_device(np.ascontiguousarray(B[:, :cols])), dev.to_device(wide)
                dev.trsm(0, 0, orient, 0, 1.0, dT, dB)
                dev.trsm(0, 0, orient, 0, 1.0, dT, dW)
                x, y = dev.to_host(dB), dev.to_host(dW)[:, :cols]
                bits = np.int64 if dtype == np.float64 else np.int32
                same = (x.view(bits) == y.view(bits)) | (np.isnan(x) & np.isnan(y))
                print("[case]", dtype.__name__, spread, orient, cols, int((~same).sum()), flush=True)
                assert same.all()


def test_many_columns_of_a_large_order(dev):
    """128 columns of an order past the chained solve's range are solved block by block, to the bits of
    the chained solve of 16 of them."""
    n = 24576
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    dT = dev.colmajor_empty(n, n)
    torch.randn(n, n, dtype=torch.float64, device="cuda", generator=g, out=dT.t())
    dT.mul_(1.0 / n)
    dT.diagonal().add_(1.0)
    B = torch.randn(n, 128, dtype=torch.float64, device="cuda", generator=g)
    for uplo in (0, 1):
        wide, part = dev.colmajor_empty(n, 128), dev.colmajor_empty(n, 16)
        wide.copy_(B)
        part.copy_(B[:, 64:80])
        dev.trsm(0, uplo, 0, 0, 1.0, dT, wide)
        dev.trsm(0, uplo, 0, 0, 1.0, dT, part)
        assert torch.equal(wide[:, 64:80], part)
