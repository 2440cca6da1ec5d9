"""soft_max of few rows, each on several waves of its workgroup, and of many short
rows, each on a few lanes, against the oracle: ends of a row off the waves'
batches, the maximum and the last nonzero exp in any wave, rows wholly masked
but for one cell."""
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


@pytest.mark.parametrize("mode", ["base", "monte", "lpvip", "sum32"])
@pytest.mark.parametrize("T,n", [(1, 511), (1, 512), (1, 900), (2, 1025), (3, 2049), (7, 1000), (1, 4097), (2, 8200),
                                 (300, 640), (5000, 33), (4500, 9), (4200, 5), (4100, 3), (4099, 17)])
def test_rows(ln, mode, T, n):
    print(f"\n[soft_max wide] {mode} {T} x {n}", flush=True)
    rng = np.random.default_rng(n + T)
    x = (rng.standard_normal((1, 1, T, n)) * 3).astype(np.float32)
    x[0, 0, 0, n - 1] = 200          # the maximum last: every other exp underflows
    mask = np.zeros((1, 1, T, n), np.float32)
    for t in range(1, min(T, 40)):   # one live cell, anywhere
        mask[0, 0, t] = -np.inf
        mask[0, 0, t, rng.integers(0, n)] = 0
    if T > 2:
        mask[0, 0, 2] = np.where(rng.random(n) < 0.5, -np.inf, rng.standard_normal(n).astype(np.float32))
        mask[0, 0, 2, 0] = 0
    for m in (None, mask):
        O.monte_set(77)
        want = O.soft_max16(O.MODES[mode], x, m, 0.3)
        dm = torch.from_numpy(m).cuda() if m is not None else None
        got = ln.soft_max16(O.MODES[mode], torch.from_numpy(x).cuda(), dm, 0.3, seed=77).cpu().numpy()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
