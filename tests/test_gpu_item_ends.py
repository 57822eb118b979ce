"""Frames that end with the last byte of their own device allocation, whole
pages: the pixel loads of the graph and raster kernels stay inside, and the
last pixel's colour and class are right.  Against the oracle."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flags", [0, 1, 2, 3])  # RGB, top-down
@pytest.mark.parametrize("W,H,S,sub", [(1, 1, 2, 0), (5, 7, 4, 0), (64, 64, 4, 0), (64, 64, 3, 1), (63, 130, 6, 0),
                                       (61, 59, 8, 1)])
def test_frames_at_the_end_of_an_allocation(gpu, D, O, W, H, S, sub, flags):
    torch = gpu
    img = np.ascontiguousarray(D.synth_frame(2, 60 + W, W, H, 3))
    hip = ctypes.CDLL("libamdhip64.so")
    size = (img.size + 4095) // 4096 * 4096
    p = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) == 0
    try:
        at = size - img.size
        assert hip.hipMemcpy(ctypes.c_void_p(p.value + at), ctypes.c_void_p(img.ctypes.data), ctypes.c_size_t(img.size), 1) == 0
        d_out = torch.zeros(4 * S * W * S * H, dtype=torch.uint8, device="cuda")
        items = D.items_array([D.Item(at, 0, W, H, img.shape[1], 3, S, sub, flags, 4 * S * W, 0)])
        ctx = D.Context(0)
        D.check(D.lib.dpx_batch_run(ctx.h, p.value, d_out.data_ptr(), items, 1, torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        got = d_out.cpu().numpy().reshape(S * H, S * W, 4)
        ctx.close()
    finally:
        torch.cuda.synchronize()
        hip.hipFree(p)
    want = O.depixelize(img, W, H, scale=S, subdivide=bool(sub), flags=flags)["rgba"]
    np.testing.assert_array_equal(got, want)
