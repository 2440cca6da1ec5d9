"""The base and Monte products whose sums leave the fast form's range, against the
oracle, over chains long enough to stay exact, to come back and to leave again:
runs of zero activations and weights at every offset, columns and rows of zeros
beside ordinary ones, sparse activations, sums that overflow and cancel, every
number of chains a lane, rows whose LDS leaves no room for all the tables."""
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
    rng = np.random.default_rng(K + 3 * M + 7 * N)
    w = (rng.standard_normal((1, 1, M, K)) * 0.02).astype(np.float32)
    x = rng.standard_normal((1, 1, N, K)).astype(np.float32)
    if kind == "relu":
        x = np.maximum(x, 0)
    elif kind == "runs":            # runs of zeros that cancel sums first
        for n in range(N):
            a = int(rng.integers(0, K))
            x[0, 0, n, a:a + int(rng.integers(1, 200))] = 0
        w[..., 1::2] = -w[..., 0:K - K % 2:2]
        x[..., 1::2] = x[..., 0:K - K % 2:2]
    elif kind == "columns":
        x[..., ::3, :] = 0
    elif kind == "rows":
        w[..., ::2, :] = 0
    elif kind == "late":            # ordinary, then nothing, then ordinary
        x[..., K // 4: K // 2] = 0
        w[..., K // 4 - 8: K // 4] = -w[..., K // 4 - 16: K // 4 - 8][..., ::-1]
    elif kind == "over":            # sums at the upper clamp, both signs
        w *= np.float32(1e18)
        x *= np.float32(1e18)
    return w, x


KINDS = ["relu", "runs", "columns", "rows", "late", "over"]


@pytest.mark.parametrize("mode", ["base", "monte"])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("K,M,N", [(64, 70, 3), (577, 40, 2), (1600, 33, 3), (71, 300, 300), (330, 64, 500), (200, 520, 500),
                                   (1100, 70, 900)])
def test_products(ln, mode, kind, K, M, N):
    print(f"\n[exact sums] {mode} {kind} K={K} M={M} N={N}", flush=True)
    w, x = operands(kind, K, M, N)
    y = ln.mul_mat16(O.MODES[mode], ln.pack16(torch.from_numpy(w).cuda()), torch.from_numpy(x).cuda(), K, M, seed=23)
    y = y.cpu().numpy()[0, 0]
    if M * N * K < 1 << 23:
        O.monte_set(23)
        want = O.mul_mat16_f32w(O.MODES[mode], w, x)[0, 0]
        assert np.array_equal(y.view(np.uint32), np.ascontiguousarray(want).view(np.uint32))
        return
    rng = np.random.default_rng(1)
    for m in {0, 1, M - 1, *rng.integers(0, M, 8).tolist()}:
        for n in {0, 1, N - 1, *rng.integers(0, N, 8).tolist()}:
            st = O.lib().lno_lfsr_jump(23, (m * N + n) * (K - 1)) if mode == "monte" else None
            want = O.x2f16(np.array([O.vec_dot16(O.MODES[mode], O.f2x16(w[0, 0, m]), O.f2x16(x[0, 0, n]), st)], np.uint16))
            assert y[n, m].view(np.uint32) == want[0].view(np.uint32), (m, n)


@pytest.mark.parametrize("mode,K", [("base", 77003), ("monte", 66001)])
@pytest.mark.parametrize("kind", ["plain", "relu", "late"])
def test_narrow_tables(ln, mode, K, kind):
    M = 21
    print(f"\n[exact sums] {mode} {kind} K={K}", flush=True)
    w, x = operands(kind, K, M, 1)
    y = ln.mul_mat16(O.MODES[mode], ln.pack16(torch.from_numpy(w).cuda()), torch.from_numpy(x).cuda(), K, M, seed=23)
    y = y.cpu().numpy()[0, 0, 0]
    for m in (0, 11, M - 1):
        st = O.lib().lno_lfsr_jump(23, m * (K - 1)) if mode == "monte" else None
        want = O.x2f16(np.array([O.vec_dot16(O.MODES[mode], O.f2x16(w[0, 0, m]), O.f2x16(x[0, 0, 0]), st)], np.uint16))
        assert y[m].view(np.uint32) == want[0].view(np.uint32), m


@pytest.mark.parametrize("mode", ["base", "monte"])
@pytest.mark.parametrize("n", [5, 17, 40, 333])
def test_row_sums_past_the_field(ln, mode, n):
    # squares whose sum passes the log field at any block, and ends past it
    rng = np.random.default_rng(n)
    x = (rng.standard_normal((8, n)) * np.float32(1e19)).astype(np.float32)
    x[1, n // 2:] *= np.float32(1e-19)
    x[2, : n // 2] *= np.float32(1e-25)
    O.monte_set(33)
    want = O.rms_norm16(O.MODES[mode], x, 1e-5)
    got = ln.rms_norm16(O.MODES[mode], torch.from_numpy(x).cuda(), 1e-5, seed=33).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
