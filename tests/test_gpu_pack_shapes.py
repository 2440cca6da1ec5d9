"""The weight-cache fill in every workgroup shape it takes (runs of one, four and
eight columns, one and four runs a thread, rows of fewer runs than a tile has
lanes, matrices of fewer rows than a tile), against the device's plain
conversions in its layout, and a matrix of more tiles than one launch takes."""
import ctypes

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ln():
    import lnship
    assert torch.cuda.is_available(), "GPU tests need a visible GPU"
    lnship.init()
    return lnship


@pytest.mark.parametrize("width,half", [(16, False), (16, True), (32, False), (32, True)])
@pytest.mark.parametrize("K,M", [(8, 5000), (9, 70), (24, 3000), (40, 1111), (72, 257), (100, 999), (104, 1), (1001, 1),
                                 (2041, 1), (20000, 3), (3000, 17), (5000, 31), (256, 256), (576, 200), (2048, 2048),
                                 (577, 30000), (2049, 2100)])
def test_shapes(ln, width, half, K, M):
    print(f"\n[pack shapes] {width} half={half} K={K} M={M}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(K + M)
    w = torch.randn(M, K, generator=g, device="cuda")
    w[torch.rand(M, K, generator=g, device="cuda") < 0.02] = 0
    if half:
        w = w.half()
    kp = ln.kp(K)
    codes = (ln.from_f32_16 if width == 16 else ln.from_f32_32)(w.float())
    want = torch.zeros(M, kp, dtype=codes.dtype, device="cuda")
    want[:, :K] = codes
    got = (ln.pack16 if width == 16 else ln.pack32)(w)
    assert torch.equal(got.view(kp // 8, M, 8), want.view(M, kp // 8, 8).transpose(0, 1))


def test_more_tiles_than_one_launch(ln):
    # one column: eight codes of output a row, 256 rows a tile, 2^23 tiles a launch
    M = (1 << 31) + 300
    print(f"\n[pack shapes] codes K=1 M={M}", flush=True)
    src = torch.randint(-32768, 32767, (M,), dtype=torch.int16, device="cuda")
    out = torch.full((M, 8), 77, dtype=torch.int16, device="cuda")
    ln.check(ln.lib().lnship16_pack(ctypes.c_void_p(src.data_ptr()), 2, 1, M, ctypes.c_void_p(out.data_ptr()), 1, M, 1,
                                    ln._stream()))
    step = 1 << 28
    for r in range(0, M, step):
        part = out[r:r + step]
        assert torch.equal(part[:, 0], src[r:r + step])
        assert not bool(part[:, 1:].any())
