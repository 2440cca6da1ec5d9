"""lpvip products of several chains per lane against the oracle: additions whose
exact branch few, most or all lanes need at once, zeros, ends of groups, one and
four chains a lane, rows that fill the LDS (one chain) or lie in scratch (eight)."""
import numpy as np
import pytest

import oracle_lib as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ln():
    import lnship
    assert torch.cuda.is_available(), "GPU tests need a visible GPU"
    lnship.init()
    return lnship


def operands(kind, K, M, N):
    rng = np.random.default_rng(K + M + N)
    w = (rng.standard_normal((1, 1, M, K)) * 0.02).astype(np.float32)
    x = rng.standard_normal((1, 1, N, K)).astype(np.float32)
    if kind == "near":        # sums and terms within a binade of each other, of either sign
        w = (np.where(rng.random(w.shape) < 0.5, -1, 1) * rng.uniform(0.6, 1.4, w.shape)).astype(np.float32)
        x = np.ones_like(x)
        x[..., 1::2] = -1
    elif kind == "cancel":    # exact cancellation, of either sign before it
        w = np.where(rng.random(w.shape) < 0.5, -0.5, 0.5).astype(np.float32)
        x = np.ones_like(x)
    elif kind == "zeros":
        w[rng.random(w.shape) < 0.3] = 0
        x[..., : K // 2] = 0
        x[..., N - 1, :] = 0
    elif kind == "wide":      # logs at both ends of the field
        w *= np.float32(1e18) ** rng.integers(-2, 3, w.shape).astype(np.float32)
    return w, x


@pytest.mark.parametrize("kind", ["plain", "near", "cancel", "zeros", "wide"])
@pytest.mark.parametrize("K,M,N", [(9, 70, 3), (41, 300, 1200), (24, 520, 900), (130, 256, 1030), (16, 3000, 160)])
def test_products(ln, kind, K, M, N):
    print(f"\n[lpvip] {kind} K={K} M={M} N={N}", flush=True)
    w, x = operands(kind, K, M, N)
    want = O.mul_mat16_f32w(O.LPVIP, w, x)
    got = ln.mul_mat16(O.LPVIP, ln.pack16(torch.from_numpy(w).cuda()), torch.from_numpy(x).cuda(), K, M).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), np.ascontiguousarray(want).view(np.uint32))


@pytest.mark.parametrize("K,M,N", [(9400, 260, 2100), (12000, 260, 2100)])
def test_long_rows(ln, K, M, N):
    print(f"\n[lpvip] long rows K={K} M={M} N={N}", flush=True)
    w, x = operands("plain", K, M, N)
    got = ln.mul_mat16(O.LPVIP, ln.pack16(torch.from_numpy(w).cuda()), torch.from_numpy(x).cuda(), K, M).cpu().numpy()[0, 0]
    for m, n in [(0, 0), (M - 1, N - 1), (100, 1000), (255, 7)]:
        want = O.x2f16(np.array([O.vec_dot16(O.LPVIP, O.f2x16(w[0, 0, m]), O.f2x16(x[0, 0, n]))], np.uint16))
        assert got[n, m].view(np.uint32) == want[0].view(np.uint32)
