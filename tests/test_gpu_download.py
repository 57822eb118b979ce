"""Large results to host memory (launch_kernel, the plain frame path): the
diagram's 360 bytes a pixel around the 4 MiB from which they go through pinned
slots, ragged last chunks, and several threads at once."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(D, O, W, H, sub, seed):
    img = D.synth_frame(0, seed, W, H, 3, W * 3)
    ref = O.depixelize(img, W, H, scale=1, subdivide=sub, want_diagram=True)
    diag, ec, graph = D.launch_kernel(img, W, H, sub)
    np.testing.assert_array_equal(graph.reshape(H, W), ref["graph"].reshape(H, W))
    np.testing.assert_array_equal(ec.reshape(H, W), ref["edge_count"].reshape(H, W))
    np.testing.assert_array_equal(diag.view(np.int32).reshape(-1), ref["diagram"].view(np.int32).reshape(-1))
    diag[0] = 0  # the caller's to write
    *_, diag2 = D.frame(img, W, H, 3, scale=1, subdivide=sub, want_diagram=True)
    np.testing.assert_array_equal(diag2.view(np.int32).reshape(-1), ref["diagram"].view(np.int32).reshape(-1))


# below 4 MiB, just above, one whole chunk and a bit, three chunks and a part
@pytest.mark.parametrize("W,H,sub", [(107, 108, False), (108, 108, True), (151, 97, False), (199, 187, True)])
def test_large_results(gpu, D, O, W, H, sub):
    check(D, O, W, H, sub, 7)


def test_large_results_from_threads(gpu, D, O):
    bad = []

    def run(k):
        try:
            for rep in range(3):
                check(D, O, 120 + 11 * k, 108 + rep, k % 2 == 1, 10 * k + rep)
        except Exception as e:  # noqa: BLE001
            bad.append(f"thread {k}: {e}")

    threads = [threading.Thread(target=run, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
