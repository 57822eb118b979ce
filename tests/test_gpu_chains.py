"""Border chains at the sizes where the kernels change: faces around the
lengths that a wave, a block's LDS and global memory hold (64, 512 and 8192
positions), faces that thousands of walks run on, and outputs that hold only
the first chains.  Against the oracle's sequential scan, node for node."""
import numpy as np
import pytest

from test_gpu_parity import gpu_border_chains

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]

DX, DY = [-1, 0, 1, -1, 1, -1, 0, 1], [1, 1, 1, 0, 0, -1, -1, -1]


def random_graph(seed, W, H, p, diagonal):
    """Links between neighbours at random; no crossing diagonals."""
    rng = np.random.default_rng(seed)
    g = np.zeros((H, W), dtype=np.uint8)
    right, up = rng.random((H, W - 1)) < p, rng.random((H - 1, W)) < p
    g[:, :-1] |= right.astype(np.uint8) << 4
    g[:, 1:] |= right.astype(np.uint8) << 3
    g[:-1] |= up.astype(np.uint8) << 1
    g[1:] |= up.astype(np.uint8) << 6
    slash = rng.random((H - 1, W - 1)) < diagonal
    back = (rng.random((H - 1, W - 1)) < diagonal) & ~slash
    g[:-1, :-1] |= slash.astype(np.uint8) << 2
    g[1:, 1:] |= slash.astype(np.uint8) << 5
    g[:-1, 1:] |= back.astype(np.uint8) << 0
    g[1:, :-1] |= back.astype(np.uint8) << 7
    return g


def check(gpu, D, O, g, what):
    chains, _, status = gpu_border_chains(gpu, D, g)
    assert status == 0, what
    assert chains == O.border_chains(g), what


@pytest.mark.parametrize("n", [2, 32, 33, 34, 256, 257, 258, 4096, 4097, 4098, 9000])
def test_lines_of_every_path_class(gpu, D, O, n):
    # a line of n nodes is one face of 2 (n - 1) positions; a second, joined
    # to it at one end, is walked on the same face
    g = np.zeros((3, n), dtype=np.uint8)
    g[::2, :-1] |= 1 << 4
    g[::2, 1:] |= 1 << 3
    check(gpu, D, O, g, f"two lines of {n}")
    g[0, 0] |= 1 << 1
    g[1, 0] |= (1 << 1) | (1 << 6)
    g[2, 0] |= 1 << 6
    check(gpu, D, O, g, f"two joined lines of {n}")


# (0.3 with diagonals: faces of up to 1,000 positions on which 5,000 walks are abandoned)
@pytest.mark.parametrize("case", [(1, 61, 47, 0.35, 0.2), (2, 200, 150, 0.45, 0.1), (3, 160, 130, 0.5, 0.05),
                                  (8, 300, 200, 0.3, 0.2), (5, 640, 480, 0.25, 0.2), (6, 511, 97, 0.6, 0.0)],
                         ids=lambda c: f"{c[1]}x{c[2]}p{c[3]}d{c[4]}")
def test_random_faces(gpu, D, O, case):
    seed, W, H, p, diagonal = case
    check(gpu, D, O, random_graph(seed, W, H, p, diagonal), f"random graph {case}")


@pytest.mark.parametrize("n", [30, 32, 33, 256, 257, 4094, 4097, 4099])
@pytest.mark.parametrize("teeth", [0, 7])
def test_paths_of_abandoned_walks(gpu, D, O, n, teeth):
    # a line of n nodes that begins at an internal node (90, its four links
    # symmetric): one path of 2 n - 1 positions into it, from which every walk
    # is abandoned, each at a node further along
    g = np.zeros((3, n + 2), dtype=np.uint8)
    g[1, 1] = 90
    g[1, 0], g[0, 1], g[2, 1] = 1 << 4, 1 << 1, 1 << 6
    g[1, 2:] |= 1 << 3
    g[1, 2:-1] |= 1 << 4
    if teeth:  # nodes beside the line, walked before it or after it
        g[1, 5:-1:teeth] |= 1 << 1
        g[2, 5:-1:teeth] |= 1 << 6
        g[1, 7:-1:teeth] |= 1 << 6
        g[0, 7:-1:teeth] |= 1 << 1
    check(gpu, D, O, g, f"line of {n} from an internal node, teeth every {teeth}")
    check(gpu, D, O, np.ascontiguousarray(((g & 0x18) | ((g >> 5) & 0x02) | ((g << 5) & 0x40))[::-1]),
          "the same upside down")


@pytest.mark.parametrize("seed", [5 * 4096, 15 * 4096])
def test_faces_of_thousands_of_walks(gpu, D, O, seed):
    # dithered 640x480 frames with a face of 4,700-6,500 positions that an
    # earlier chain touches: 2,300 and 3,200 walks on it are abandoned in turn
    img = D.synth_frame(4, seed, 640, 480, 3)
    g = O.depixelize(img, 640, 480, scale=1)["graph"]
    check(gpu, D, O, np.ascontiguousarray(g), f"frame {seed}")


@pytest.mark.parametrize("k", [0, 1, 7, -1])
def test_outputs_that_hold_the_first_chains(gpu, D, O, k):
    g = random_graph(9, 120, 90, 0.4, 0.1)
    want = O.border_chains(g)
    k = k % len(want)
    nodes = sum(len(c) for c in want[:k])
    # as many chains, and as many nodes, as the first k need (one node short of the next)
    for max_nodes, max_chains in ((8 * g.size, k), (nodes + len(want[k]) - 1, g.size)):
        chains, nn, status = gpu_border_chains(gpu, D, g, max_nodes=max_nodes, max_chains=max_chains)
        assert status == D.ENOMEM and chains == want[:k] and nn == nodes
