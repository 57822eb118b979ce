"""The raster and the window on a caller's diagram whose vertex counts are no
polygon's: such cells cover nothing, whatever the count."""
import ctypes

import numpy as np
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


@pytest.mark.parametrize("count", [-(1 << 31), -(1 << 31) + 1, -3, -1, 1, 2])
def test_counts_below_a_triangle(gpu, D, O, count):
    torch, W, H, S, ww, wh = gpu, 21, 17, 4, 90, 70
    img = np.ascontiguousarray(D.synth_frame(2, 9, W, H, 3))
    ref = O.depixelize(img, W, H, scale=1, subdivide=True, want_diagram=True)
    n = np.array(ref["edge_count"], dtype=np.int32).reshape(-1)
    d_img, diag = torch.from_numpy(img).cuda(), torch.from_numpy(np.array(ref["diagram"], dtype=np.float32).reshape(-1)).cuda()
    s = torch.cuda.current_stream().cuda_stream

    def images(value):
        m = n.copy()
        m[::5] = value
        ec, res = torch.from_numpy(m).cuda(), []
        out = torch.zeros(4 * S * W * S * H, dtype=torch.uint8, device="cuda")
        D.check(D.lib.dpx_stage_rasterize(d_img.data_ptr(), W, H, img.shape[1], 3, 0, diag.data_ptr(), ec.data_ptr(), S,
                                          out.data_ptr(), 4 * S * W, s))
        res.append(out)
        for scale in (50, 100, 800):  # no tiles, low tiles, tall tiles
            out = torch.zeros(4 * ww * wh, dtype=torch.uint8, device="cuda")
            view = D.View(0, scale, 1, 1, ww, wh, 1, 0)
            D.check(D.lib.dpx_stage_present(d_img.data_ptr(), W, H, img.shape[1], 3, 0, diag.data_ptr(), ec.data_ptr(),
                                            ctypes.byref(view), out.data_ptr(), 4 * ww, s))
            res.append(out)
        torch.cuda.synchronize()
        return [r.cpu().numpy() for r in res]

    for got, want in zip(images(count), images(0)):
        np.testing.assert_array_equal(got, want)
