"""The weight-cache fill against the oracle's conversions in its layout: tiles cut
by rows and columns, K off the group of eight, strided and misaligned sources,
every conversion bucket."""
import ctypes

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


def layout(codes):
    """[slices, M, K] codes -> [slices, Kp / 8, M, 8]"""
    ns, M, K = codes.shape
    out = np.zeros((ns, M, (K + 7) & ~7), codes.dtype)
    out[..., :K] = codes
    return out.reshape(ns, M, -1, 8).transpose(0, 2, 1, 3)


@pytest.mark.parametrize("width,src", [(16, "f32"), (16, "f16"), (16, "codes"), (32, "f32"), (32, "f16")])
@pytest.mark.parametrize("K,M,ns,ld,off", [(8, 1, 1, 8, 0), (5, 3, 2, 5, 0), (256, 33, 1, 256, 0), (264, 32, 2, 272, 0),
                                           (257, 70, 1, 264, 0), (255, 31, 3, 260, 1), (64, 40, 1, 64, 1), (600, 65, 1, 607, 0)])
def test_pack(ln, width, src, K, M, ns, ld, off):
    print(f"\n[pack] {width} {src} K={K} M={M} slices={ns} ld={ld} off={off}", flush=True)
    rng = np.random.default_rng(K + M)
    slice_ = M * ld + 3 * (ld % 8)
    n = off + ns * slice_
    if src == "codes":
        flat = rng.integers(0, 65536, n).astype(np.uint16)
    else:
        flat = rng.standard_normal(n).astype(np.float16 if src == "f16" else np.float32)
        flat[rng.random(n) < 0.05] = 0
        flat[rng.random(n) < 0.02] = np.inf
        flat[rng.random(n) < 0.02] *= flat.dtype.type(1e-5)
    t = torch.from_numpy(flat.view(np.int16) if src == "codes" else flat).cuda()
    kp = (K + 7) & ~7
    out = torch.full((ns * kp * M + 16,), 77, dtype=torch.int16 if width == 16 else torch.int32, device="cuda")
    fn = ln.lib().lnship16_pack if width == 16 else ln.lib().lnship32_pack
    ln.check(fn(ctypes.c_void_p(t.data_ptr() + off * t.element_size()), {"f32": 0, "f16": 1, "codes": 2}[src], ld, slice_,
                ctypes.c_void_p(out.data_ptr()), K, M, ns, ln._stream()))
    torch.cuda.synchronize()
    rows = np.stack([flat[off + z * slice_:][: M * ld].reshape(M, ld)[:, :K] for z in range(ns)])
    if src == "codes":
        codes = rows
    else:
        v = rows.astype(np.float32)
        codes = O.f2x16(v).reshape(v.shape) if width == 16 else O.f2x32(v).reshape(v.shape)
    got = out.cpu().numpy().view(codes.dtype)
    assert np.array_equal(got[: ns * kp * M].reshape(ns, kp // 8, M, 8), layout(codes))
    assert np.all(got[ns * kp * M:] == 77), "nothing past the cache is written"


def test_pack_every_bucket(ln):
    # each of the 2^17 buckets of the float -> xlns16 table, and every half
    x = (np.arange(1 << 17, dtype=np.uint32) << 15 | 0x5a5).view(np.float32).reshape(256, 512)
    want = layout(O.f2x16(x).reshape(1, 256, 512))
    assert np.array_equal(ln.pack16(torch.from_numpy(x).cuda()).cpu().numpy().view(np.uint16).reshape(want.shape), want)
    # (of the halves' NaNs, whose conversions to float keep or quiet the payload, one)
    h = np.arange(1 << 16, dtype=np.uint16).view(np.float16)
    h = np.where(np.isnan(h), np.float16(np.nan), h).reshape(128, 512)
    want = layout(O.f2x16(h.astype(np.float32)).reshape(1, 128, 512))
    assert np.array_equal(ln.pack16(torch.from_numpy(h).cuda()).cpu().numpy().view(np.uint16).reshape(want.shape), want)
