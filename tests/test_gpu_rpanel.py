"""The register-resident LU panel at the sizes where it can go wrong: 32-column blocks (partial
last block, 8-column chunks), 1024 rows per workgroup (one workgroup, its remainder, several),
exact ties, and exactly zero pivots in any block. A single panel is lu::Panel alone, so factors,
pivots and the state left at a zero pivot equal the oracle's bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("m,w,pad", [(1, 1, 0), (8, 8, 1), (33, 33, 0), (64, 9, 3), (200, 128, 1),
                                     (1023, 31, 0), (1024, 128, 0), (1025, 97, 2), (1055, 64, 1),
                                     (2049, 128, 5)])
def test_panel_edges(dev, orc, m, w, pad, dtype):
    rng = np.random.default_rng(m * 131 + w)
    for kind in ("gaussian", "ties", "zero first", "zero inside", "zero last"):
        print("[case]", m, w, pad, dtype.__name__, kind, flush=True)
        A = rng.standard_normal((m, w)).astype(dtype)
        if kind == "ties":
            A = rng.integers(-1, 2, size=(m, w)).astype(dtype)
        if kind.startswith("zero"):
            A[:, {"zero first": 0, "zero inside": w // 2, "zero last": w - 1}[kind]] = 0
        F_ref, d_ref, info_ref = orc.lu(A, bsize=128)
        buf = torch.full((w, m + pad), 7.0, dtype=torch.from_numpy(A).dtype, device="cuda")
        dA = buf.t()[:m]
        dA.copy_(torch.from_numpy(A))
        d, info = dev.getrf(dA, nb=128)
        assert int(info.item()) == info_ref
        k = w if info_ref == 0 else info_ref
        assert np.array_equal(d.cpu().numpy()[:k], d_ref[:k])
        assert np.array_equal(dev.to_host(dA), F_ref)
        assert bool((buf[:, m:] == 7.0).all())
