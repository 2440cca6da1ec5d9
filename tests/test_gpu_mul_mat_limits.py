"""Products of so many columns that a launch of fewer columns a workgroup than the
shape chosen would pass a grid's limits: accepted, and every column block formed,
against the oracle at the ends of the launches."""
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


def check_columns(ln, mode, K, M, N, columns):
    print(f"\n[limits] {mode} K={K} M={M} N={N}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(K)
    w = torch.randn(M, K, generator=g, device="cuda") * 0.02
    x = torch.randn(1, 1, N, K, generator=g, device="cuda")
    y = torch.full((1, 1, N, M), float("nan"), device="cuda")
    ln.mul_mat16(O.MODES[mode], ln.pack16(w), x, K, M, seed=19, out=y)
    assert not bool(torch.isnan(y).any())
    L = O.lib()
    for n in columns:
        xc, wc = O.f2x16(x[0, 0, n].cpu().numpy()), w.cpu().numpy()
        for m in {0, M // 2, M - 1}:
            st = L.lno_lfsr_jump(19, (m * N + n) * (K - 1)) if mode == "monte" else None
            want = O.x2f16(np.array([O.vec_dot16(O.MODES[mode], O.f2x16(wc[m]), xc, st)], np.uint16))
            got = y[0, 0, n, m].cpu().numpy().reshape(1)
            assert got.view(np.uint32)[0] == want.view(np.uint32)[0], (n, m)


@pytest.mark.parametrize("mode,K", [("base", 9704), ("monte", 8192), ("lpvip", 9400)])
def test_fewer_columns_a_workgroup(ln, mode, K):
    # eight rows of codes fill the LDS beside what eight columns a lane take:
    # one column a workgroup, and those past 65535 in a launch of their own
    N = 2 * 65535 + 61
    check_columns(ln, mode, K, 8, N, [0, 65534, 65535, 2 * 65535, N - 1])


@pytest.mark.parametrize("M", [64, 70])
def test_64_row_groups_past_the_grid(ln, M):
    # 64-row groups of up to sixteen columns would take more than 65535 blocks
    N = 16 * 65535 + 5
    check_columns(ln, "sum32", 8, M, N, [0, 16 * 65535 - 1, 16 * 65535, N - 1])
