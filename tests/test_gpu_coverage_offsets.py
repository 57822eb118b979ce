"""Smoothed batches whose cell coverage passes 2^32 words: a frame behind that
mark takes its own coverage, not another frame's."""
import numpy as np
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


def test_coverage_beyond_32_bits_of_words(gpu, D, O):
    torch = gpu
    N, W, H, fill = 16384, 64, 48, 4  # 4 x 16384 x 16384 cells of 5 words at 1x: 5.4 G words, 21.5 GB
    img = np.asarray(D.synth_frame(0, 77, W, H, 3), np.uint8)
    # the fillers are one black frame, read and written over each other
    items = [D.Item(0, 0, N, N, N, 1, 1, 1, D.INDEXED, 4 * N, N * N) for _ in range(fill)]
    items.append(D.Item(N * N + 1024, 4 * N * N, W, H, img.shape[1], 3, 1, 1, 0, 4 * W))
    d_in = torch.zeros(N * N + 1024 + img.size, dtype=torch.uint8, device="cuda")
    d_in[N * N + 1024:] = torch.from_numpy(img.reshape(-1)).cuda()
    d_out = torch.zeros(4 * N * N + 4 * W * H, dtype=torch.uint8, device="cuda")
    ctx = D.Context(0)
    ctx.run(d_in, d_out, items)
    torch.cuda.synchronize()
    got = d_out[4 * N * N:].cpu().numpy().reshape(H, W, 4)
    ctx.close()
    del d_in, d_out
    torch.cuda.empty_cache()
    np.testing.assert_array_equal(got, O.depixelize(img, W, H, scale=1, subdivide=True)["rgba"])
