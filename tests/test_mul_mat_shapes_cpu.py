"""The shape of a product's launch (no GPU): within a launch's limits wherever
another shape is, and bad arguments refused."""
import ctypes

import pytest

import lnship as ln

MODES = range(5)   # the four xlns16 modes, and 4: xlns32


def shape(mode, K, M, N, ns=1, cus=256):
    out = (ctypes.c_int * 8)()
    assert ln.lib().lnship_test_mul_mat_shape(mode, K, M, N, ns, cus, out) == 0
    return dict(zip(["nc", "cg", "rb", "xl", "w", "x32", "rg", "tight"], out))


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("M", [1, 64, 65, 300, 577])
def test_columns_within_a_grid(mode, M):
    # up to the columns that the widest group takes
    widest = {3: 32, 4: 16}.get(mode, 8)
    for n in (1, 100, 65535, 65536, 500000, 16 * 65535 - 3, 16 * 65535 + 1, 32 * 65535):
        s = shape(mode, 40, M, n)
        if n <= 65535 * widest:
            assert -(-n // (s["nc"] * s["cg"])) <= 65535, (n, s)


@pytest.mark.parametrize("mode", [3, 4])
def test_threads_within_a_launch(mode):
    for M in (1 << 20, (1 << 28) - 1, (1 << 28) + 1, (1 << 29) + 65):
        s = shape(mode, 8, M, 64)
        assert -(-M // s["rb"]) * s["cg"] * s["rb"] < 1 << 32 or s["rb"] == 256, (M, s)


def test_refusals():
    out = (ctypes.c_int * 8)()
    fn = ln.lib().lnship_test_mul_mat_shape
    for args in [(5, 8, 1, 1, 1, 256, out), (-1, 8, 1, 1, 1, 256, out), (0, -1, 1, 1, 1, 256, out), (0, 8, 0, 1, 1, 256, out),
                 (0, 8, 1, 0, 1, 256, out), (0, 8, 1, 1, 0, 256, out), (0, 8, 1, 1, 1, 0, out), (0, 8, 1, 1, 1, 256, None)]:
        assert fn(*args) == -1, args[:6]
