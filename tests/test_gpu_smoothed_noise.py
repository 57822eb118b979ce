"""Smoothed batches of dithers of nearly similar colours, where cut points blend
with hulls that do not hold the corner and cells reach up to three quarters of a
cell beyond their square, at every scale, against the oracle."""
import numpy as np
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


def noise(rng, kind, W, H, ch):
    if kind == 0:  # around one colour, some pairs similar and some not
        a = rng.integers(0, 256, ch) + rng.integers(-9, 10, (H, W, ch))
    elif kind == 1:  # greys around one
        a = rng.integers(10, 240) + rng.integers(-6, 7, (H, W, 1)) + np.zeros(ch, int)
    else:  # a few colours
        pal = rng.integers(0, 256, (int(rng.integers(2, 6)), ch))
        a = pal[rng.integers(0, len(pal), (H, W))]
    return np.ascontiguousarray((a & 255).astype(np.uint8).reshape(H, W * ch))


@pytest.mark.parametrize("S", range(1, 16))
def test_noise(gpu, D, O, S):
    torch, rng = gpu, np.random.default_rng(S)
    blobs, items, refs, in_off, out_off = [], [], [], 0, 0
    for k in range(9):
        W, H, ch, flags = int(rng.integers(30, 80)), int(rng.integers(20, 60)), 3 + k % 2, k % 4  # RGB, top-down
        img = noise(rng, k % 3, W, H, ch)
        items.append(D.Item(in_off, out_off, W, H, img.shape[1], ch, S, 1, flags, 4 * S * W))
        refs.append(O.depixelize(img, W, H, scale=S, subdivide=True, channels=ch, flags=flags)["rgba"])
        blobs += [img.reshape(-1), np.zeros(-img.size % 4, np.uint8)]
        in_off += img.size + -img.size % 4
        out_off += 4 * S * W * S * H
    d_in = torch.from_numpy(np.concatenate(blobs)).cuda()
    d_out = torch.zeros(out_off, dtype=torch.uint8, device="cuda")
    ctx = D.Context(0)
    ctx.run(d_in, d_out, items)
    torch.cuda.synchronize()
    out = d_out.cpu().numpy()
    ctx.close()
    for k, (it, ref) in enumerate(zip(items, refs)):
        got = out[it.out_offset:it.out_offset + it.out_stride * it.height * S].reshape(it.height * S, it.width * S, 4)
        bad = (got != ref).any(-1).sum()
        assert bad == 0, f"item {k}, {it.width}x{it.height}: {bad} pixels"
