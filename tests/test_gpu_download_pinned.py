"""Large results to pinned memory go to it directly: equal to those in
pageable memory, which pass through the library's slots and its threads."""
import ctypes
import os
import threading

import numpy as np
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]


def test_pinned_destinations_are_written_directly(gpu, D):
    W, H, S = 640, 480, 8
    img = D.synth_frame(0, 3, W, H, 3)
    p = D.Params(S, 0, 0, 0)
    outs = {"pageable": np.zeros((S * H, 4 * S * W), np.uint8), "pinned": D.pinned_empty((S * H, 4 * S * W))}

    def frame(out):
        D.check(D.lib.dpx_frame(img.ctypes.data, W, H, img.shape[1], 3, ctypes.byref(p), out.ctypes.data, 4 * S * W,
                                None, None, None))

    def threads_seen(out):
        """The process's threads beyond those before the calls, at most, while they run."""
        frame(out)  # (the runtime's own threads start)
        most, stop, ready = [0], threading.Event(), threading.Event()

        def watch():
            base = len(os.listdir("/proc/self/task"))
            ready.set()
            while not stop.is_set():
                most[0] = max(most[0], len(os.listdir("/proc/self/task")) - base)

        t = threading.Thread(target=watch)
        t.start()
        ready.wait()
        for _ in range(10):
            frame(out)
        stop.set()
        t.join()
        return most[0]

    seen = {k: threads_seen(o) for k, o in outs.items()}
    np.testing.assert_array_equal(outs["pinned"], outs["pageable"])
    assert seen["pageable"] > 0 and seen["pinned"] == 0, seen
