"""sum32 and xlns32 products whose launches take column groups of one wave's rows
(few rows, or rows that a 256-row group covers badly), and three that stay with
256-row groups beside them, against the oracle: rows and columns off the tiles,
broadcast weight slices, K off the group of eight, activation rows in LDS (sum32)
and in scratch (xlns32)."""
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


@pytest.mark.parametrize("fmt", ["sum32", "lns32"])
@pytest.mark.parametrize("K,M,N,ne02,ne12", [(44, 64, 203, 3, 9), (40, 64, 96, 1, 2), (37, 70, 33, 3, 3), (40, 577, 201, 1, 1),
                                             (16, 40, 16, 2, 30), (24, 64, 1000, 1, 4), (20, 100, 60, 4, 20), (9, 1, 500, 1, 8),
                                             (1100, 64, 130, 1, 9)])
def test_row_groups(ln, fmt, K, M, N, ne02, ne12):
    print(f"\n[row groups] {fmt} K={K} M={M} N={N} slices {ne02} of {ne12}", flush=True)
    rng = np.random.default_rng(K + M + N)
    w = (rng.standard_normal((1, ne02, M, K)) * 0.1).astype(np.float32)
    x = rng.standard_normal((1, ne12, N, K)).astype(np.float32)
    dw, dx = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()
    if fmt == "lns32":
        want, got = O.mul_mat32(w, x, ne02, 1), ln.mul_mat32(ln.pack32(dw), dx, K, M, ne02, 1)
    else:
        want, got = O.mul_mat16_f32w(O.SUM32, w, x, ne02, 1), ln.mul_mat16(O.SUM32, ln.pack16(dw), dx, K, M, ne02, 1)
    assert np.array_equal(got.cpu().numpy().view(np.uint32), np.ascontiguousarray(want).view(np.uint32))
