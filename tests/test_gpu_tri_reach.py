"""The raster and the window on cells whose triangles use the whole reach of
smoothed cells (-48 to 106 of 64), and on some that go beyond it (as far as the
next cell, since those around a sample are its candidates; on a frame of 2x2
cells any distance), from the smallest scale to the largest, against the oracle."""
import ctypes

import numpy as np
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]

CS = 45


def diagram(rng, W, H, beyond):
    d, n = np.zeros((W * H, CS, 2), dtype=np.float32), rng.integers(2, 17, size=W * H).astype(np.int32)
    v = rng.integers(-48, 107, size=(W * H, CS, 2))
    edge = rng.random(v.shape) < 0.3
    v[edge] = rng.choice([-48, 106], size=int(edge.sum()))
    if beyond:  # in every ninth cell, every other one of a small frame
        far = rng.choice([-49, 107, -63, 127] if W > 2 else [-49, 107, 200, -255, -256, -257, 255, 256, 4000, -4000],
                         size=v.shape)
        far[rng.random(v.shape) < 0.7] = 20
        every = 9 if W > 2 else 2
        v[::every] = far[::every]
    k = np.arange(W * H)
    d[..., 0] = v[..., 0] / 64.0 + (k % W)[:, None]
    d[..., 1] = v[..., 1] / 64.0 + (k // W)[:, None]
    # (small triangles too: the reach alone covers the frame)
    small = rng.random((W * H, CS // 3)) < 0.6
    t = d.reshape(W * H, CS // 3, 3, 2)
    t[small, 1:] = t[small, :1] + rng.integers(-20, 21, size=(int(small.sum()), 2, 2)) / 64.0
    if not beyond or W > 2:
        lo, least, most = np.stack([k % W, k // W], axis=1)[:, None, None], *((-63, 127) if beyond else (-48, 106))
        t[:] = np.clip(t, lo + least / 64.0, lo + most / 64.0)
    return d, n


@pytest.mark.parametrize("beyond", [False, True])
@pytest.mark.parametrize("scale", [25, 50, 97, 99, 100, 101, 130, 250, 800, 3200])
@pytest.mark.parametrize("aa", [0, 1])
def test_windows(gpu, D, O, scale, beyond, aa):
    torch, W, H, ww, wh = gpu, 23, 19, 130, 75
    rng = np.random.default_rng(scale + beyond)
    img = np.ascontiguousarray(rng.integers(0, 256, (H, 3 * W)).astype(np.uint8))
    d, n = diagram(rng, W, H, beyond)
    d_img, diag, ec = (torch.from_numpy(a).cuda() for a in (img, d.reshape(-1), n))
    for tx, ty in ((1, 1), (-7 * scale // 100, -300)):
        out = torch.zeros(4 * ww * wh, dtype=torch.uint8, device="cuda")
        view = D.View(0, scale, tx, ty, ww, wh, aa, 0)
        D.check(D.lib.dpx_stage_present(d_img.data_ptr(), W, H, 3 * W, 3, 0, diag.data_ptr(), ec.data_ptr(),
                                        ctypes.byref(view), out.data_ptr(), 4 * ww, torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        want = O.present(img, W, H, d.reshape(-1, 2), n, mode=0, scale_x100=scale, tx=tx, ty=ty, width=ww, height=wh,
                         view_flags=aa)
        np.testing.assert_array_equal(out.cpu().numpy().reshape(wh, ww, 4), want)


@pytest.mark.parametrize("beyond", [False, True])
@pytest.mark.parametrize("scale", [1, 2, 3, 8, 32])
def test_rasters(gpu, D, O, scale, beyond):
    torch, rng = gpu, np.random.default_rng(scale)
    raster(torch, D, O, rng, 23, 19, scale, beyond)
    for _ in range(20 if beyond else 0):
        raster(torch, D, O, rng, 2, 2, scale, beyond)


def raster(torch, D, O, rng, W, H, scale, beyond):
    img = np.ascontiguousarray(rng.integers(0, 256, (H, 3 * W)).astype(np.uint8))
    d, n = diagram(rng, W, H, beyond)
    d_img, diag, ec = (torch.from_numpy(a).cuda() for a in (img, d.reshape(-1), n))
    out = torch.zeros(4 * W * scale * H * scale, dtype=torch.uint8, device="cuda")
    D.check(D.lib.dpx_stage_rasterize(d_img.data_ptr(), W, H, 3 * W, 3, 0, diag.data_ptr(), ec.data_ptr(), scale,
                                      out.data_ptr(), 4 * W * scale, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    want = O.rasterize(img, W, H, d.reshape(-1, 2), n, scale)
    np.testing.assert_array_equal(out.cpu().numpy().reshape(-1), np.asarray(want).reshape(-1))
