"""Border chains when the rounds are used up: no chains and a status, not the
chains of a state that has not settled."""
import ctypes

import numpy as np
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


def test_unsettled_walks_are_reported(gpu, D, O):
    torch = gpu
    W, H = 640, 480
    g = O.depixelize(D.synth_frame(4, 5 * 4096, W, H, 3), W, H, scale=1)["graph"]  # waits after the launched rounds
    d_g = torch.from_numpy(np.ascontiguousarray(g).reshape(-1)).cuda()
    scratch = torch.zeros(W * H, dtype=torch.uint8, device="cuda")
    nodes = torch.full((8 * W * H,), -1, dtype=torch.int32, device="cuda")
    sizes, counts = torch.zeros(W * H, dtype=torch.int32, device="cuda"), torch.zeros(3, dtype=torch.int32, device="cuda")
    run = D.lib.dpx_internal_border_chains
    run.restype = ctypes.c_int
    run.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int,
                    ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_uint32]

    def chains(rounds):
        D.check(run(d_g.data_ptr(), W, H, scratch.data_ptr(), nodes.data_ptr(), 8 * W * H, sizes.data_ptr(), W * H,
                    counts.data_ptr(), torch.cuda.current_stream().cuda_stream, rounds))
        torch.cuda.synchronize()
        return counts.cpu().tolist()

    want = O.border_chains(g.reshape(H, W))
    for rounds in (0, 1):
        assert chains(rounds) == [0, 0, D.EHIP]
        assert int(nodes.max()) == -1 and int(sizes.max()) == 0
    assert chains(2 * W * H + 1) == [len(want), sum(map(len, want)), 0]
