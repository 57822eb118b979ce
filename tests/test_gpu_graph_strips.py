"""kf_graph's strips: widths around the 62 columns a strip yields, heights
around its row blocks, the low blocks of small launches and the tall ones of
large ones, every pixel format, against the oracle."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (width, height): one column, one row, a strip's edges, several strips, a
# strip holding several whole row blocks (narrow frames)
SIZES = [(1, 1), (1, 67), (3, 130), (8, 8), (61, 5), (62, 59), (63, 60), (64, 1), (65, 61), (124, 3), (131, 121)]
# channels, flags (1 RGB, 2 top-down, 4 alpha), row padding, synthetic kind
FORMATS = [(3, 0, 0, 0), (3, 3, 1, 2), (3, 2, 0, 4), (4, 4, 0, 1), (4, 7, 4, 1), (1, 0, 0, 5), (1, 2, 3, 5)]


def frames(D, ch, flags, pad, kind):
    out = []
    for k, (W, H) in enumerate(SIZES):
        if ch == 1:
            idx, pal = D.stream_frame(300 + k, 1, W, H)
            rows = np.zeros((H, W + pad), np.uint8)
            rows[:, :W] = np.asarray(idx).reshape(H, -1)[:, :W]
            src = np.asarray(pal, np.uint8).reshape(256, 4)[rows[:, :W]].reshape(H, 4 * W)
            out.append((rows, np.asarray(pal, np.uint8).reshape(-1), np.ascontiguousarray(src), 4, W, H))
        else:
            img = np.asarray(D.synth_frame(kind, 300 + k, W, H, ch)).reshape(H, -1)[:, :W * ch]
            if ch == 3:  # greys: multiples of 1000 in the luma sum, where doubles decide
                g = (np.arange(W * H, dtype=np.uint32).reshape(H, W) * 37 % 256).astype(np.uint8)
                m = np.arange(W * H).reshape(H, W) % 5 == 0
                px = img.reshape(H, W, 3).copy()
                px[m] = g[m][:, None]
                img = px.reshape(H, 3 * W)
            rows = np.zeros((H, W * ch + pad), np.uint8)
            rows[:, :W * ch] = img
            out.append((rows, None, np.ascontiguousarray(img), ch, W, H))
    return out


def graphs(torch, D, fr, ch, flags, copies):
    blobs, items, in_off, out_off = [], [], 0, 0
    for rows, pal, _, _, W, H in fr:
        off = in_off
        for a in ([rows] if pal is None else [rows, pal]):
            a = a.reshape(-1)
            blobs += [a, np.zeros(-a.size % 4, np.uint8)]
            in_off += a.size + -a.size % 4
        pal_off = 0 if pal is None else in_off - pal.size
        for _ in range(copies):
            items.append(D.Item(off, out_off, W, H, rows.shape[1], ch, 1, 0, flags, 4 * W, pal_off))
            out_off += 4 * W * H
    d_in = torch.from_numpy(np.concatenate(blobs)).cuda()
    d_out = torch.zeros(out_off, dtype=torch.uint8, device="cuda")
    ctx = D.Context(0)
    ctx.keep_graph(True)
    ctx.run(d_in, d_out, items)
    torch.cuda.synchronize()
    gptr, goffs = ctx.graph(len(items))
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    res = []
    for it, go in zip(items, goffs):
        g = np.zeros((it.height, it.width), np.uint8)
        assert hip.hipMemcpy(g.ctypes.data, gptr + go, g.size, 2) == 0
        res.append(g)
    ctx.close()
    return res


# copies: a launch of 2-row blocks, one of middling blocks, one of the tallest
@pytest.mark.parametrize("copies", [1, 40, 600])
@pytest.mark.parametrize("ch,flags,pad,kind", FORMATS)
def test_strips_match_the_oracle(gpu, D, O, ch, flags, pad, kind, copies):
    fr = frames(D, ch, flags, pad, kind)
    ref = [O.depixelize(src, W, H, scale=1, channels=sch, flags=flags)["graph"].reshape(H, W)
           for _, _, src, sch, W, H in fr]
    got = graphs(gpu, D, fr, ch, flags | (D.INDEXED if ch == 1 else 0), copies)
    for k, (r, f) in enumerate(zip(ref, fr)):
        for c in (0, copies // 2, copies - 1):
            np.testing.assert_array_equal(got[k * copies + c], r, err_msg=f"{f[4]}x{f[5]} copy {c}")
