"""kf_graph on a frame of all 2^24 colours, laid out so that neighbours lie
around the thresholds (one step right mostly differs in V, by 5 to 7, one up in
luma, by 5 or 6), in both byte orders and with a fourth byte, against the
oracle's graph."""
import ctypes

import numpy as np
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


@pytest.mark.parametrize("channels,flags", [(3, 0), (3, 1), (4, 0)])
def test_graph_of_every_colour(gpu, D, O, channels, flags):
    torch = gpu
    N = 4096
    x, y = np.arange(N, dtype=np.int64)[None, :], np.arange(N, dtype=np.int64)[:, None]
    i, j, k = x & 255, (y & 15) | (x >> 8) << 4, y >> 4
    img = np.zeros((N, N, channels), np.uint8)
    # (modulo 256 a bijection: the steps' determinant is odd)
    for c, (right, up, far) in enumerate(((7, 5, 0), (-4, 5, 0), (1, 6, 1))):
        img[..., 2 - c if flags & D.RGB else c] = (right * i + up * j + far * k) & 255
    if channels == 4:
        img[..., 3] = (x * 31 + y * 17) & 255  # no alpha test: not looked at
    assert np.unique(img[..., 0].astype(np.uint32) | img[..., 1].astype(np.uint32) << 8 |
                     img[..., 2].astype(np.uint32) << 16).size == 1 << 24
    img = img.reshape(N, N * channels)
    want = O.heuristic_cross(O.trivial_cross(O.similarity_graph(img, N, N, channels=channels, flags=flags)))
    d_in = torch.from_numpy(img.reshape(-1)).cuda()
    d_out = torch.zeros(4 * N * N, dtype=torch.uint8, device="cuda")
    ctx = D.Context(0)
    ctx.keep_graph(True)
    ctx.run(d_in, d_out, [D.Item(0, 0, N, N, N * channels, channels, 1, 0, flags, 4 * N)])
    torch.cuda.synchronize()
    gptr, goffs = ctx.graph(1)
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    got = np.zeros((N, N), np.uint8)
    assert hip.hipMemcpy(got.ctypes.data, gptr + goffs[0], got.size, 2) == 0
    ctx.close()
    for e in range(8):  # every direction has links and gaps
        assert 0.02 < ((want >> e) & 1).mean() < 0.98, e
    np.testing.assert_array_equal(got, np.asarray(want).reshape(N, N))
