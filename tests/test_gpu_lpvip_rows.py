"""lpvip's sums of positive terms (rms_norm's squares, soft_max's exps) against the
oracle: terms far below and above the sum, equal ones, sums past the log field,
rows that end at any place of a group."""
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


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 65, 577, 2001])
def test_row_sums(ln, n):
    print(f"\n[lpvip rows] n={n}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.standard_normal((8, n)).astype(np.float32)
    x[1] = 0
    x[2] *= np.float32(1e19) ** rng.integers(-1, 2, n).astype(np.float32)   # any distance
    x[3] *= np.float32(1e19)                                                # past the field
    x[4] = 1
    x[5, : n // 2] = 0
    x[6] *= np.float32(2.0) ** rng.integers(-14, 15, n).astype(np.float32)  # about the essential zero
    want = O.rms_norm16(O.LPVIP, x, 1e-5)
    got = ln.rms_norm16(O.LPVIP, torch.from_numpy(x).cuda(), 1e-5).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    s = (rng.standard_normal((1, 1, 6, n)) * 8).astype(np.float32)
    want = O.soft_max16(O.LPVIP, s, None, 0.7)
    got = ln.soft_max16(O.LPVIP, torch.from_numpy(s).cuda(), None, 0.7).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
