"""A reserved context takes batches without waiting for the device: while
another stream's kernel still runs, dpx_batch_run returns."""
import numpy as np
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


def batch(D, torch, sizes, S):
    blobs, items, refs, in_off, out_off = [], [], [], 0, 0
    for k, (W, H) in enumerate(sizes):
        img = np.asarray(D.synth_frame(0, 500 + k, W, H, 3), np.uint8)
        items.append(D.Item(in_off, out_off, W, H, img.shape[1], 3, S, 0, 0, 4 * S * W))
        blobs.append(img.reshape(-1))
        refs.append(img)
        in_off += img.size
        out_off += 4 * S * W * S * H
    return (torch.from_numpy(np.concatenate(blobs)).cuda(), torch.zeros(out_off, dtype=torch.uint8, device="cuda"), items,
            refs)


# the raster tile grid is the same for a batch's items, the number of strips is not
@pytest.mark.parametrize("sizes", [[(640, 480)] * 4 + [(639, 480)], [(60 - k % 9, 31) for k in range(3000)],
                                   [(64, 860)] + [(49, 860)] * 39])  # (the last needs a map of 13,900 strips)
def test_reserved_context_does_not_wait(gpu, D, O, sizes):
    torch = gpu
    S = 2
    d_in, d_out, items, imgs = batch(D, torch, sizes, S)
    warm = D.Context(0)  # (loads the kernels)
    warm.run(d_in, d_out, items, torch.cuda.current_stream())
    torch.cuda.synchronize()
    warm.close()
    d_out.zero_()
    ctx = D.Context(0)
    ctx.reserve(len(sizes), max(w * h for w, h in sizes), S)
    arr = D.items_array(items)
    t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t0.record()
    torch.cuda._sleep(1 << 20)
    t1.record()
    torch.cuda.synchronize()
    cycles = int((1 << 20) * 400.0 / t0.elapsed_time(t1))  # 400 ms
    side, busy = torch.cuda.Stream(), torch.cuda.Event()
    with torch.cuda.stream(side):
        torch.cuda._sleep(cycles)
        busy.record(side)
    ctx.run(d_in, d_out, arr, torch.cuda.current_stream())
    waited = busy.query()
    torch.cuda.synchronize()
    assert not waited, "dpx_batch_run waited for the device"
    out = d_out.cpu().numpy()
    for k in (0, len(items) - 1):
        it = items[k]
        got = out[it.out_offset:it.out_offset + it.out_stride * it.height * S].reshape(it.height * S, it.width * S, 4)
        np.testing.assert_array_equal(got, O.depixelize(imgs[k], it.width, it.height, scale=S)["rgba"])
    ctx.close()
