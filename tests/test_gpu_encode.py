"""lsg_lightmap_encode on the GPU: every per-texel buffer format, scaled and linear targets,
lightmap and bent-normal layers, equal byte for byte to the reference's buffer interface
(tests/golden/encode_formats.npz, pinned in test_encode_cpu.py; float formats compare NaN
as NaN, whatever its sign), including the tail of a
batch that is not a multiple of 4 texels; and the lightmaps of a filtered bake encoded to sRGB bytes
equal to the closed form applied to its downloaded RGBA."""
import ctypes
import os

import numpy as np
import pytest

from test_encode_cpu import FORMATS, GOLDEN, model

pytestmark = pytest.mark.gpu


def _encode(rgba, fmt, scaled, bent, bg):
    from lightsprintsdk_amd import native as N
    from lightsprintsdk_amd.collider import DeviceBuffer
    L = N.lib()
    n = len(rgba)
    nb = int(L.lsg_format_bytes(fmt)) * n
    d_in = DeviceBuffer.from_array(np.ascontiguousarray(rgba, np.float32))
    d_out = DeviceBuffer(max(nb, 4))
    b = np.ascontiguousarray(bg, np.float32)
    N.check(L.lsg_lightmap_encode(d_in.ptr, n, fmt, scaled, 0.45, 0.0 if bent else 0.45, b.ctypes.data_as(ctypes.c_void_p),
                                  d_out.ptr, None), "encode")
    N.check(L.lsg_synchronize(), "sync")
    return d_out.download(np.uint8, (nb,))


def test_gpu_encode_equals_reference_buffers(gpu):
    z = np.load(GOLDEN)
    rgba, bg = z["rgba"], z["background"]
    for fmt in FORMATS:
        for scaled in (0, 1):
            for bent in (0, 1):
                for n in (len(rgba), len(rgba) - 3):        # tails of 3 and 0 texels
                    got = _encode(rgba[:n], fmt, scaled, bent, bg)
                    want = z[f"f{fmt}_s{scaled}_b{bent}"][:len(got)]
                    assert len(got) == len(want)
                    if fmt in (3, 4, 10):       # floats: a NaN's sign and payload are not compared
                        assert np.array_equal(got.view(np.float32), want.view(np.float32), equal_nan=True), (fmt, scaled, bent, n)
                    else:
                        np.testing.assert_array_equal(got, want, err_msg=f"format {fmt} scaled {scaled} bent {bent} n {n}")


def test_gpu_encode_bake(gpu):
    from lightsprintsdk_amd import bake as B, scenes as S
    sc = S.box_room(seed=9, n_boxes=6, target_tris=8000, lightmap_size=128)
    plan = B.BakePlan(sc, B.GatherParams(quality=64, ray_length_min=S.minimal_safe_distance(sc.verts), seed=2))
    plan.run(first=True, graph=False)
    bg = np.float32([0.1, 0.2, 0.3, 1.0])
    for k in (0, len(sc.objects) - 1):
        rgba = plan.lightmap_layer_rgba(k, 0).reshape(-1, 4)
        got = _encode(rgba, 0, 1, 0, bg)
        np.testing.assert_array_equal(got, model(rgba, bg, 0, 1, 0))
        assert got.max() > 0
    plan.close()


@pytest.mark.parametrize("fmt", [0, 2])
def test_gpu_encode_bytes_at_their_borders(gpu, fmt):
    """sRGB bytes where the binary32 power alone cannot tell the byte: every value whose
    power is within a few units in the last place of k / 256, values a little further, and
    0, 1, negatives, huge values, infinities and NaN; against the closed form in binary64."""
    k = np.arange(1, 257) / 256.0
    mid = (k ** (1.0 / np.float64(np.float32(0.45)))).astype(np.float32)
    vals = [mid]
    for _ in range(4):
        vals.append(np.nextafter(vals[-1], np.float32(9)))
    lo = mid
    for _ in range(4):
        lo = np.nextafter(lo, np.float32(-1))
        vals.append(lo)
    for r in (2.0 ** -10, 2.0 ** -9, 2.0 ** -8):
        vals += [mid * np.float32(1 + r / 4), mid * np.float32(1 - r / 4), mid * np.float32(1 + r), mid * np.float32(1 - r)]
    rng = np.random.default_rng(6)
    vals.append(np.float32(10) ** rng.uniform(-9, 1, 20000).astype(np.float32))
    vals.append(np.float32([0, -0.0, 1, -1, -1e-3, 1e-45, 1e-38, 1e9, 3e38, -3e38, np.inf, -np.inf, np.nan]))
    x = np.concatenate(vals).astype(np.float32)
    x = x[:len(x) // 3 * 3].reshape(-1, 3)
    rgba = np.ones((len(x), 4), np.float32)
    rgba[:, :3] = x
    bg = np.zeros(4, np.float32)
    with np.errstate(all="ignore"):
        want = model(rgba, bg, fmt, 1, 0)
    np.testing.assert_array_equal(_encode(rgba, fmt, 1, 0, bg), want)
