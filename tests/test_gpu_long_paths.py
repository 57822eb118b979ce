"""Border chains of faces beyond the 8192 positions that a block's LDS holds:
the minima over them (64 positions an entry up to 524288, 128 from there), walks
that wrap around the face's end, and the time a walk takes, which does not grow
with the face.  Against the oracle's sequential scan, node for node."""
import numpy as np
import pytest

from test_gpu_chains import check

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


def path_into_90(n, teeth=0):
    # an internal node (90, its four links symmetric) with a line of n nodes: one path of 2 n - 1 positions
    g = np.zeros((3, n + 2), dtype=np.uint8)
    g[1, 1] = 90
    g[1, 0], g[0, 1], g[2, 1] = 1 << 4, 1 << 1, 1 << 6
    g[1, 2:] |= 1 << 3
    g[1, 2:-1] |= 1 << 4
    if teeth:
        g[1, 5:-1:teeth] |= 1 << 1
        g[2, 5:-1:teeth] |= 1 << 6
        g[1, 7:-1:teeth] |= 1 << 6
        g[0, 7:-1:teeth] |= 1 << 1
    return g


def ring(W, spots, length, teeth):
    # a ring around rows 0 and 6, listed by the chain around it, and lines of `length` nodes in row 3 inside it, each
    # on a stub from the ring: the walks of their nodes run on the inner face, a cycle of some 2 W positions, and are
    # abandoned at the ring or at each other's marks
    g = np.zeros((7, W), dtype=np.uint8)

    def link(a, b):  # b is right of a or above it
        up = b[0] > a[0]
        g[a] |= 1 << (1 if up else 4)
        g[b] |= 1 << (6 if up else 3)

    for r in (0, 6):
        g[r, :-1] |= 1 << 4
        g[r, 1:] |= 1 << 3
    for c in (0, W - 1):
        for r in range(6):
            link((r, c), (r + 1, c))
    for x in spots:
        for r in range(3):
            link((r, x), (r + 1, x))
        for k in range(length):
            link((3, x + k), (3, x + k + 1))
            if teeth and k % teeth == 2:
                link((3, x + k), (4, x + k))
            if teeth and k % teeth == 4:
                link((2, x + k), (3, x + k))
    return g


# (walks, times their lengths, are the sequential oracle's time: paths of up to 12,000 nodes, and in the rings, whose
# faces pass 524288 positions between 255,000 and 275,000 columns, lines of up to 1,500)
@pytest.mark.parametrize("n,teeth", [(4097, 0), (4160, 9), (10000, 0), (12000, 5)])
def test_paths(gpu, D, O, n, teeth):
    check(gpu, D, O, path_into_90(n, teeth), f"path of {n} nodes, teeth every {teeth}")


@pytest.mark.parametrize("flip", [False, True])
@pytest.mark.parametrize("W,spots,length,teeth", [(4200, (3, 900, 2500), 600, 0), (20000, (5, 3000, 17000), 1500, 7),
                                                  (255000, (1, 100000, 253000), 1500, 9),
                                                  (275000, (1, 64000, 140000, 273000), 1500, 11)])
def test_cycles(gpu, D, O, W, spots, length, teeth, flip):
    g = ring(W, spots, length, teeth)
    if flip:  # rows upside down: up and down links change places
        g = np.ascontiguousarray(((g & 0x18) | ((g >> 5) & 0x02) | ((g << 5) & 0x40))[::-1])
    check(gpu, D, O, g, f"ring of {W} columns, lines at {spots}, flipped {flip}")


@pytest.mark.parametrize("kind,seed", [(0, 2 * 4096), (0, 3 * 4096), (4, 1 * 4096)])
def test_large_frames(gpu, D, O, kind, seed):
    # game frames of 1280x960 with faces of some 20,000 positions, and a dithered one
    g = O.depixelize(D.synth_frame(kind, seed, 1280, 960, 3), 1280, 960, scale=1)["graph"]
    check(gpu, D, O, np.ascontiguousarray(g.reshape(960, 1280)), f"frame {kind} {seed}")


def test_a_walk_takes_as_long_on_a_longer_path(gpu, D):
    torch = gpu

    def ms(n):
        g = torch.from_numpy(path_into_90(n)).cuda()
        H, W = g.shape
        size = W * H
        scratch = torch.zeros(size, dtype=torch.uint8, device="cuda")
        nodes = torch.zeros(8 * size, dtype=torch.int32, device="cuda")
        sizes, counts = torch.zeros(size, dtype=torch.int32, device="cuda"), torch.zeros(3, dtype=torch.int32, device="cuda")
        t = []
        for _ in range(3):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            D.check(D.lib.dpx_stage_border_chains(g.data_ptr(), W, H, scratch.data_ptr(), nodes.data_ptr(), 8 * size,
                                                  sizes.data_ptr(), size, counts.data_ptr(),
                                                  torch.cuda.current_stream().cuda_stream))
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b))
        return min(t)

    short, long = ms(10000), ms(40000)
    # four times the walks on four times the positions: 4 times as long where a walk's time is its own, 16 times
    # where it reads the positions ahead of it; the line between them is their geometric mean
    assert long < 8 * short, (short, long)
