"""The rms_norm before a base or Monte product in its launch, whose sum of squares
runs over the product's own table: squares that pass the log field at the first
term, inside a block and at the last, rows of zeros and of tiny values, and rows
so long that the tables are the narrow ones, against the nodes run apart."""
import ctypes

import numpy as np
import pytest

import oracle_lib as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

EPS = 1e-5


@pytest.fixture(scope="module")
def ln():
    import lnship
    assert torch.cuda.is_available(), "GPU tests need a visible GPU"
    lnship.init()
    return lnship


@pytest.mark.parametrize("mode", ["base", "monte"])
@pytest.mark.parametrize("K,M,N", [(5, 40, 6), (8, 40, 6), (9, 40, 6), (41, 70, 6), (577, 40, 6), (40, 2000, 200), (66001, 20, 1),
                                   (77003, 20, 1)])
def test_rms_prologue(ln, mode, K, M, N):
    print(f"\n[norm prologue] {mode} K={K} M={M} N={N}", flush=True)
    if mode == "monte" and K > 70000:
        pytest.skip("longer than the rows that Monte's launches stage")
    m, L = O.MODES[mode], ln.lib()
    rng = np.random.default_rng(K)
    x = rng.standard_normal((N, K)).astype(np.float32)
    if N > 4:
        x[0] *= np.float32(1e19)
        x[1, K // 2:] *= np.float32(1.8e19)
        x[2, K - 1] = 1.84e19
        x[2, : K - 1] *= np.float32(1e18)
        x[3] = 0
        x[4] *= np.float32(1e-25)
    wn = (rng.standard_normal(K) * 0.5 + 1).astype(np.float32)
    w = (rng.standard_normal((M, K)) * 0.02).astype(np.float32)
    dx, dwn, wp = torch.from_numpy(x).cuda(), torch.from_numpy(wn).cuda(), ln.pack16(torch.from_numpy(w).cuda())
    s0 = 3001
    s1 = L.lnship_lfsr_jump(s0, L.lnship16_rms_norm_draws(m, K, N))
    out = torch.full((N, M), float("nan"), device="cuda")
    a = ln.MulMatArgs(wp.data_ptr(), dx.data_ptr(), out.data_ptr(), K, M, N, 1, 1, 1, 1, 0, 0, s1, 0, 0, 0, 0, None, 0, None)
    a.rms_norm_w, a.rms_eps, a.rms_seed = dwn.data_ptr(), EPS, s0
    ln.check(L.lnship16_mul_mat(m, ctypes.byref(a), ln._stream()))
    p = lambda t: ctypes.c_void_p(t.data_ptr())   # noqa: E731
    h, ref = torch.empty(N, K, device="cuda"), torch.empty(N, M, device="cuda")
    ln.check(L.lnship16_rms_norm_mul(m, p(dx), p(dwn), p(h), K, N, ctypes.c_float(EPS), s0, None, 0, ln._stream()))
    ln.mul_mat16_raw(m, wp.data_ptr(), h.data_ptr(), ref.data_ptr(), K, M, N, seed=s1)
    assert np.array_equal(out.cpu().numpy().view(np.uint32), ref.cpu().numpy().view(np.uint32))
    if N > 4 and K < 1000:   # and the nodes apart against the oracle
        O.monte_set(s0)
        want = O.rms_norm16(m, x, EPS)
        got = ln.rms_norm16(m, dx, EPS, seed=s0).cpu().numpy()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
