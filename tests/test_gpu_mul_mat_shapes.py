"""Products in every shape a launch takes on a device of 256 CUs (columns a lane,
column groups, rows of a group and of a wave, activation rows in LDS as codes or
at four bytes or in scratch, row groups that share them, narrow tables): each case
states its shape and is checked to take it, then against the oracle at sampled
outputs, rows and columns off the tiles among them."""
import ctypes

import numpy as np
import pytest

import oracle_lib as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# mode, K, M, N, activation slices (one weight slice), and the shape:
# (columns a lane, column groups, rows of a group, rows in LDS, rows of a wave,
#  four bytes a value, row groups, narrow tables)
CASES = [
    ("base", 40007, 3, 1, 1, (1, 1, 256, 1, 16, 0, 1, 0)),
    ("base", 77003, 3, 1, 1, (1, 1, 256, 1, 16, 0, 1, 1)),
    ("base", 71, 3, 1, 1, (1, 1, 256, 1, 16, 1, 1, 0)),
    ("base", 40007, 167, 99, 1, (1, 1, 256, 1, 32, 0, 1, 0)),
    ("base", 77003, 530, 31, 1, (1, 1, 256, 1, 32, 0, 1, 1)),
    ("base", 71, 1094, 15, 1, (1, 1, 256, 1, 32, 1, 1, 0)),
    ("base", 9704, 3, 517, 2, (1, 1, 256, 1, 64, 0, 1, 0)),
    ("base", 77003, 1366, 8, 3, (1, 1, 256, 1, 64, 0, 1, 1)),
    ("base", 71, 3643, 1, 9, (1, 1, 256, 1, 64, 1, 1, 0)),
    ("base", 40007, 78, 258, 1, (4, 1, 256, 0, 64, 0, 1, 0)),
    ("base", 9800, 78, 271, 3, (4, 1, 256, 1, 64, 0, 1, 0)),
    ("base", 71, 74, 413, 2, (4, 1, 256, 1, 64, 1, 1, 0)),
    ("base", 3000, 522, 67, 9, (4, 1, 256, 1, 64, 1, 2, 0)),
    ("base", 5000, 1029, 263, 2, (4, 1, 256, 1, 64, 1, 4, 0)),
    ("base", 10500, 74, 529, 2, (8, 1, 256, 0, 64, 0, 1, 0)),
    ("base", 6500, 76, 686, 3, (8, 1, 256, 1, 64, 0, 1, 0)),
    ("base", 71, 71, 1630, 2, (8, 1, 256, 1, 64, 1, 1, 0)),
    ("base", 2048, 517, 347, 3, (8, 1, 256, 1, 64, 1, 2, 0)),
    ("base", 3000, 1066, 410, 3, (8, 1, 256, 1, 64, 1, 4, 0)),
    ("monte", 77003, 3, 1, 1, (1, 1, 256, 0, 64, 0, 1, 0)),
    ("monte", 40007, 3, 1, 1, (1, 1, 256, 1, 16, 0, 1, 0)),
    ("monte", 66001, 3, 1, 1, (1, 1, 256, 1, 16, 0, 1, 1)),
    ("monte", 71, 3, 1, 1, (1, 1, 256, 1, 16, 1, 1, 0)),
    ("monte", 40007, 458, 4, 9, (1, 1, 256, 1, 32, 0, 1, 0)),
    ("monte", 66001, 1822, 1, 9, (1, 1, 256, 1, 32, 0, 1, 1)),
    ("monte", 71, 2342, 7, 1, (1, 1, 256, 1, 32, 1, 1, 0)),
    ("monte", 8192, 3, 1035, 1, (1, 1, 256, 1, 64, 0, 1, 0)),
    ("monte", 66001, 1493, 11, 2, (1, 1, 256, 1, 64, 0, 1, 1)),
    ("monte", 71, 866, 38, 1, (1, 1, 256, 1, 64, 1, 1, 0)),
    ("monte", 30011, 87, 133, 2, (4, 1, 256, 0, 64, 0, 1, 0)),
    ("monte", 8400, 72, 258, 3, (4, 1, 256, 1, 64, 0, 1, 0)),
    ("monte", 71, 86, 409, 2, (4, 1, 256, 1, 64, 1, 1, 0)),
    ("monte", 2048, 580, 182, 3, (4, 1, 256, 1, 64, 1, 2, 0)),
    ("monte", 4001, 74, 1021, 1, (4, 1, 256, 1, 64, 1, 4, 0)),
    ("monte", 9400, 70, 1063, 1, (8, 1, 256, 0, 64, 0, 1, 0)),
    ("monte", 8100, 71, 1028, 1, (8, 1, 256, 1, 64, 0, 1, 0)),
    ("monte", 71, 76, 375, 9, (8, 1, 256, 1, 64, 1, 1, 0)),
    ("monte", 1000, 524, 119, 9, (8, 1, 256, 1, 64, 1, 2, 0)),
    ("monte", 2048, 1143, 123, 9, (8, 1, 256, 1, 64, 1, 4, 0)),
    ("lpvip", 71, 3, 1, 1, (1, 1, 256, 1, 4, 0, 1, 0)),
    ("lpvip", 71, 114, 18, 2, (1, 1, 256, 1, 8, 0, 1, 0)),
    ("lpvip", 71, 34, 241, 1, (1, 1, 256, 1, 16, 0, 1, 0)),
    ("lpvip", 71, 38, 216, 2, (1, 1, 256, 1, 32, 0, 1, 0)),
    ("lpvip", 71, 683, 24, 2, (1, 1, 256, 1, 64, 0, 1, 0)),
    ("lpvip", 40007, 70, 95, 3, (4, 1, 256, 0, 64, 0, 1, 0)),
    ("lpvip", 71, 75, 811, 1, (4, 1, 256, 1, 64, 0, 1, 0)),
    ("lpvip", 9800, 73, 1039, 1, (8, 1, 256, 0, 64, 0, 1, 0)),
    ("lpvip", 71, 70, 1572, 2, (8, 1, 256, 1, 64, 0, 1, 0)),
    ("sum32", 16000, 3, 1, 1, (1, 1, 256, 0, 64, 0, 1, 0)),
    ("sum32", 71, 3, 1, 1, (1, 1, 256, 1, 16, 0, 1, 0)),
    ("sum32", 71, 5483, 3, 1, (1, 1, 256, 1, 64, 0, 1, 0)),
    ("sum32", 8100, 72, 279, 1, (1, 2, 256, 0, 64, 0, 1, 0)),
    ("sum32", 71, 70, 117, 3, (1, 2, 256, 1, 64, 0, 1, 0)),
    ("sum32", 4001, 1578, 9, 9, (1, 4, 256, 0, 64, 0, 1, 0)),
    ("sum32", 71, 1091, 13, 9, (1, 4, 256, 1, 64, 0, 1, 0)),
    ("sum32", 4001, 76, 267, 2, (1, 8, 64, 0, 64, 0, 1, 0)),
    ("sum32", 71, 74, 549, 1, (1, 8, 64, 1, 64, 0, 1, 0)),
    ("sum32", 4001, 322, 33, 9, (1, 12, 64, 0, 64, 0, 1, 0)),
    ("sum32", 71, 74, 1035, 1, (1, 12, 64, 1, 64, 0, 1, 0)),
    ("sum32", 2048, 71, 203, 9, (1, 16, 64, 0, 64, 0, 1, 0)),
    ("sum32", 71, 72, 1670, 1, (1, 16, 64, 1, 64, 0, 1, 0)),
    ("sum32", 2048, 195, 174, 9, (2, 4, 256, 0, 64, 0, 1, 0)),
    ("sum32", 71, 208, 781, 2, (2, 4, 256, 1, 64, 0, 1, 0)),
    ("sum32", 1000, 194, 1870, 2, (4, 4, 256, 0, 64, 0, 1, 0)),
    ("sum32", 71, 202, 1622, 2, (4, 4, 256, 1, 64, 0, 1, 0)),
    ("sum32", 520, 199, 2661, 3, (8, 4, 256, 0, 64, 0, 1, 0)),
    ("sum32", 71, 193, 798, 9, (8, 4, 256, 1, 64, 0, 1, 0)),
    ("lns32", 8100, 3, 1, 1, (1, 1, 256, 0, 16, 0, 1, 0)),
    ("lns32", 8100, 443, 37, 1, (1, 1, 256, 0, 64, 0, 1, 0)),
    ("lns32", 71, 3, 1, 1, (1, 1, 256, 1, 16, 0, 1, 0)),
    ("lns32", 71, 2054, 8, 1, (1, 1, 256, 1, 64, 0, 1, 0)),
    ("lns32", 71, 91, 135, 2, (1, 2, 256, 0, 64, 0, 1, 0)),
    ("lns32", 71, 2426, 6, 9, (1, 4, 256, 0, 64, 0, 1, 0)),
    ("lns32", 71, 70, 515, 1, (1, 8, 64, 0, 64, 0, 1, 0)),
    ("lns32", 71, 77, 1064, 1, (1, 12, 64, 0, 64, 0, 1, 0)),
    ("lns32", 71, 70, 572, 3, (1, 16, 64, 0, 64, 0, 1, 0)),
    ("lns32", 71, 228, 1590, 1, (2, 4, 256, 0, 64, 0, 1, 0)),
    ("lns32", 71, 209, 1043, 3, (4, 4, 256, 0, 64, 0, 1, 0)),
]


@pytest.fixture(scope="module")
def ln():
    import lnship
    assert torch.cuda.is_available(), "GPU tests need a visible GPU"
    lnship.init()
    return lnship


def shape(ln, mode, K, M, N, ns):
    out = (ctypes.c_int * 8)()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    ln.check(ln.lib().lnship_test_mul_mat_shape(4 if mode == "lns32" else O.MODES[mode], K, M, N, ns, cus, out))
    return tuple(out)


def operands(kind, K, M, N, ns):
    g = torch.Generator(device="cuda")
    g.manual_seed(K + M + N)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")   # noqa: E731
    w, x = rn(M, K) * 0.02, rn(1, ns, N, K)
    if kind == "near":       # sums and terms within a binade of each other, of either sign
        w = torch.sign(w) * (0.6 + 0.8 * torch.rand(M, K, generator=g, device="cuda"))
        x = torch.sign(x)
    elif kind == "cancel":   # exact cancellation, of either sign before it
        w, x = torch.sign(w) * 0.5, torch.ones_like(x)
    elif kind == "zeros":
        w[torch.rand(M, K, generator=g, device="cuda") < 0.3] = 0
        x[..., : K // 2] = 0
        x[..., N - 1, :] = 0
    return w, x


def check(ln, mode, K, M, N, ns, kind):
    w, x = operands(kind, K, M, N, ns)
    if mode == "lns32":
        y = ln.mul_mat32(ln.pack32(w), x, K, M)
    else:
        y = ln.mul_mat16(O.MODES[mode], ln.pack16(w), x, K, M, seed=19)
    assert not bool(torch.isnan(y).any()) or kind != "plain"
    rng = np.random.default_rng(K)
    L = O.lib()
    samples = 4 if K > 20000 else 24
    ms = [0, M - 1, M // 2, 63 % M, 64 % M] + rng.integers(0, M, samples).tolist()
    ns_ = [0, N - 1, N // 2] + rng.integers(0, N, samples).tolist()
    for i in range(samples + 3):
        m, n, z = ms[i % len(ms)], ns_[i % len(ns_)], int(rng.integers(0, ns))
        wr, xr = w[m].cpu().numpy(), x[0, z, n].cpu().numpy()
        got = y[0, z, n, m].cpu().numpy().reshape(1)
        if mode == "lns32":
            want = O.mul_mat32(wr.reshape(1, 1, 1, K), xr.reshape(1, 1, 1, K)).reshape(1)
        else:
            st = L.lno_lfsr_jump(19, ((z * M + m) * N + n) * (K - 1)) if mode == "monte" else None
            want = O.x2f16(np.array([O.vec_dot16(O.MODES[mode], O.f2x16(wr), O.f2x16(xr), st)], np.uint16))
        assert got.view(np.uint32)[0] == np.ascontiguousarray(want).view(np.uint32)[0], (m, n, z)


@pytest.mark.parametrize("mode,K,M,N,ns,want", CASES)
def test_shape(ln, mode, K, M, N, ns, want):
    print(f"\n[shapes] {mode} K={K} M={M} N={N} slices={ns}", flush=True)
    assert shape(ln, mode, K, M, N, ns) == want
    check(ln, mode, K, M, N, ns, "plain")
    if K < 20000:
        check(ln, mode, K, M, N, ns, "zeros")


# lpvip's exchange of near distances, with eight and four chains a lane and
# the activation rows in LDS beside its slots
@pytest.mark.parametrize("kind", ["near", "cancel", "zeros"])
@pytest.mark.parametrize("K,M,N,want", [(130, 1030, 2050, (8, 1, 256, 1, 64, 0, 1, 0)),
                                        (2048, 300, 3081, (8, 1, 256, 1, 64, 0, 1, 0)),
                                        (331, 577, 901, (4, 1, 256, 1, 64, 0, 1, 0))])
def test_lpvip_chains(ln, kind, K, M, N, want):
    print(f"\n[shapes] lpvip {kind} K={K} M={M} N={N}", flush=True)
    assert shape(ln, "lpvip", K, M, N, 1) == want
    check(ln, "lpvip", K, M, N, 1, kind)
