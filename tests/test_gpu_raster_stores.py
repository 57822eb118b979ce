"""kf_raster's searched cells and its stores at every scale: tiles that keep
colours and tiles that keep winners, chunks across cells and inside one, odd
output alignments and strides, partial tiles, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (kind, width, height): a dithered frame (most cells searched), a game frame
# (few), a sprite narrower than a tile, one cell
FRAMES = [(4, 37, 19), (0, 70, 18), (1, 9, 24), (0, 1, 1)]
# bytes before the first output row, bytes after each
LAYOUTS = [(0, 0), (16, 16), (8, 8), (4, 12)]


@pytest.mark.parametrize("sub", [0, 1])
@pytest.mark.parametrize("S", range(1, 16))
def test_searched_cells_and_stores(gpu, D, O, S, sub):
    torch = gpu
    blobs, items, refs, in_off, out_off = [], [], [], 0, 0
    for k, (kind, W, H) in enumerate(FRAMES):
        ch = 4 if kind == 1 else 3
        flags = (D.ALPHA if kind == 1 else 0) | (D.FLIP_OUT if k == 1 else 0)
        img = D.synth_frame(kind, 40 + k, W, H, ch)
        # (the oracle knows no DPX_FLIP_OUT: its rows, reversed)
        rgba = O.depixelize(img, W, H, scale=S, subdivide=bool(sub), channels=ch, flags=flags & ~D.FLIP_OUT)["rgba"]
        rows = np.asarray(rgba).reshape(S * H, 4 * S * W)[::-1 if flags & D.FLIP_OUT else 1]
        for lead, gap in LAYOUTS:
            pitch = 4 * S * W + gap
            out_off = (out_off + 15) // 16 * 16 + lead
            items.append(D.Item(in_off, out_off, W, H, img.shape[1], ch, S, sub, flags, pitch, 0))
            refs.append(rows)
            out_off += pitch * S * H
        blob = np.asarray(img, np.uint8).reshape(-1)
        blobs += [blob, np.zeros(-blob.size % 4, np.uint8)]
        in_off += blob.size + -blob.size % 4
    d_in = torch.from_numpy(np.concatenate(blobs)).cuda()
    d_out = torch.full((out_off,), 0xA5, dtype=torch.uint8, device="cuda")
    ctx = D.Context(0)
    ctx.run(d_in, d_out, items)
    torch.cuda.synchronize()
    out = d_out.cpu().numpy()
    ctx.close()
    used = np.zeros(out.size, bool)
    for it, ref in zip(items, refs):
        rows = np.lib.stride_tricks.as_strided(out[it.out_offset:], ref.shape, (it.out_stride, 1))
        np.testing.assert_array_equal(rows, ref, err_msg=f"{it.width}x{it.height} at {it.out_offset} + {it.out_stride}")
        for r in range(ref.shape[0]):
            o = it.out_offset + r * it.out_stride
            used[o:o + ref.shape[1]] = True
    assert (out[~used] == 0xA5).all(), "bytes outside the rows were written"
