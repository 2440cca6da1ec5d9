"""The base and Monte products and row sums against the oracle, bit for bit, where
their block-wise fast form can go wrong: ends of groups and blocks, operands that
leave the fast form's range (zeros, cancellation, underflow, overflow) at any
place of a chain, several workgroup shapes, rows that leave Monte's tables no
room in LDS."""
import numpy as np
import pytest

import oracle_lib as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

MODES = ["base", "monte"]


@pytest.fixture(scope="module")
def ln():
    import lnship
    assert torch.cuda.is_available(), "GPU tests need a visible GPU"
    lnship.init()
    return lnship


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def same_bits(got, want, what):
    g, w = np.ascontiguousarray(got).view(np.uint32), np.ascontiguousarray(want).view(np.uint32)
    assert g.shape == w.shape, (what, g.shape, w.shape)
    assert np.array_equal(g, w), f"{what}: {np.count_nonzero(g != w)}/{g.size} differ"


def operands(kind, K, M, N, seed):
    rng = np.random.default_rng(seed)
    w = (rng.standard_normal((1, 1, M, K)) * 0.02).astype(np.float32)
    x = rng.standard_normal((1, 1, N, K)).astype(np.float32)
    if kind == "zeros":          # leading, scattered and trailing zeros, a zero row and a zero column
        w[rng.random(w.shape) < 0.25] = 0
        x[..., : K // 3] = 0
        x[..., K - K // 5:] = 0
        w[..., 0, :] = 0
        x[..., N - 1, :] = 0
    elif kind == "cancel":       # sums that return to exactly zero, of either sign before it
        w[...] = np.where(rng.random(w.shape) < 0.5, 0.5, 1.0)
        x[...] = np.where(np.arange(K) % 2 == 0, 1.0, -1.0)
        w[..., 1::2] = w[..., 0:K - K % 2:2][..., : w[..., 1::2].shape[-1]]
        x[..., 1, :] *= -1 if N > 1 else 1
    elif kind == "tiny":         # products below the smallest code, then ordinary ones in places
        w *= np.float32(1e-30)
        x[rng.random(x.shape) < 0.9] *= np.float32(1e-12)
        w[..., K // 2] = 0.5
    elif kind == "huge":         # products and sums past the largest code
        w *= np.float32(1e30)
        x *= np.float32(1e10)
        w[..., ::7] *= np.float32(1e-25)
    return w, x


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("kind", ["plain", "zeros", "cancel", "tiny", "huge"])
@pytest.mark.parametrize("K,M,N", [(7, 5, 2), (8, 65, 2), (9, 3, 3), (71, 70, 2), (72, 33, 5), (73, 16, 2), (137, 40, 9),
                                   (520, 20, 4), (64, 300, 1200), (40, 520, 800)])
def test_products(ln, mode, kind, K, M, N):
    print(f"\n[products] {mode} {kind} K={K} M={M} N={N}", flush=True)
    w, x = operands(kind, K, M, N, K + M)
    O.monte_set(91)
    want = O.mul_mat16_f32w(O.MODES[mode], w, x)
    same_bits(host(ln.mul_mat16(O.MODES[mode], ln.pack16(dev(w)), dev(x), K, M, seed=91)), want, f"{mode} {kind} {K}x{M}x{N}")


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("K,M,N", [(2048, 2048, 512),    # two row groups share long word rows
                                   (1200, 1030, 530),    # four columns a lane, ragged rows
                                   (5000, 300, 2100),    # word rows do not fit: code rows
                                   (9704, 260, 2100),    # base: nor do eight code rows (one column); Monte: in scratch
                                   (30011, 40, 1),       # one column as logs and signs
                                   (40007, 40, 1),       # as codes: too long for both
                                   (66000, 3, 1)])       # Monte: no room for all the tables
def test_workgroup_shapes(ln, mode, K, M, N):
    print(f"\n[shapes] {mode} K={K} M={M} N={N}", flush=True)
    w, x = operands("plain", K, M, N, 5)
    w[0, 0, M // 2, : K // 2] = 0
    got = host(ln.mul_mat16(O.MODES[mode], ln.pack16(dev(w)), dev(x), K, M, seed=19))[0, 0]
    rng = np.random.default_rng(8)
    L = O.lib()
    for m in {0, M - 1, M // 2, *rng.integers(0, M, 6).tolist()}:
        for n in {0, N - 1, *rng.integers(0, N, 4).tolist()}:
            st = L.lno_lfsr_jump(19, (m * N + n) * (K - 1)) if mode == "monte" else None
            want = O.x2f16(np.array([O.vec_dot16(O.MODES[mode], O.f2x16(w[0, 0, m]), O.f2x16(x[0, 0, n]), st)], np.uint16))
            same_bits(got[n, m:m + 1], want, f"{mode} output ({m}, {n})")


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n", [1, 8, 9, 41, 72, 200])
def test_row_sums(ln, mode, n):
    # rms_norm's squares and soft_max's exps: rows of zeros, of tiny values, of
    # values whose squares overflow, and masked first cells
    print(f"\n[row sums] {mode} n={n}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.standard_normal((6, n)).astype(np.float32)
    x[1] = 0
    x[2] *= np.float32(1e-25)
    x[3] *= np.float32(1e25)
    x[4, : n - 1] = 0
    O.monte_set(33)
    want = O.rms_norm16(O.MODES[mode], x, 1e-5)
    same_bits(host(ln.rms_norm16(O.MODES[mode], dev(x), 1e-5, seed=33)), want, f"rms_norm {mode} {n}")
    s = (rng.standard_normal((1, 1, 6, n)) * 3).astype(np.float32)
    s[0, 0, 2] *= 30
    mask = np.zeros((1, 1, 6, n), np.float32)
    mask[0, 0, 3, : n // 2] = -np.inf
    mask[0, 0, 4, n // 2 + 1:] = -np.inf
    O.monte_set(35)
    want = O.soft_max16(O.MODES[mode], s, mask, 0.5)
    same_bits(host(ln.soft_max16(O.MODES[mode], dev(s), dev(mask), 0.5, seed=35)), want, f"soft_max {mode} {n}")
