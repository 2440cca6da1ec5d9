"""soft_max rows against the oracle at the edges of the kernel's lane groups and
batches, with masks that hold finite values beside 0 and -inf, and rows so long
that the Gaussian logs stay in global memory."""
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


def check(ln, mode, H, T, n, masked):
    print(f"\n[soft_max rows] {mode} {H} x {T} x {n} masked={masked}", flush=True)
    rng = np.random.default_rng(n + T)
    x = (rng.standard_normal((1, H, T, n)) * 3).astype(np.float32)
    x[0, 0, 0] *= 40
    mask = None
    if masked:
        mask = np.zeros((1, 1, T, n), np.float32)
        mask[rng.random(mask.shape) < 0.3] = -np.inf
        mask[..., 0] = 0
        some = rng.random(mask.shape) < 0.1
        mask[some] = rng.standard_normal(np.count_nonzero(some)).astype(np.float32)
        mask[0, 0, T - 1, n // 2:] = -1e30
    O.monte_set(77)
    want = O.soft_max16(O.MODES[mode], x, mask, 0.3)
    dm = torch.from_numpy(mask).cuda() if masked else None
    got = ln.soft_max16(O.MODES[mode], torch.from_numpy(x).cuda(), dm, 0.3, seed=77).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("mode", ["base", "monte", "lpvip", "sum32"])
@pytest.mark.parametrize("H,T,n", [(1, 1, 1), (3, 5, 7), (2, 9, 8), (5, 70, 9), (3, 40, 33), (7, 33, 64), (2, 17, 65), (4, 30, 257),
                                   (1, 3, 2049), (9, 300, 20)])
def test_soft_max_rows(ln, mode, H, T, n):
    check(ln, mode, H, T, n, True)
    check(ln, mode, H, T, n, False)


@pytest.mark.parametrize("mode", ["base", "monte", "lpvip", "sum32"])
def test_longest_rows(ln, mode):
    check(ln, mode, 1, 1, ln.lib().lnship_max_row(1, O.MODES[mode]), True)
