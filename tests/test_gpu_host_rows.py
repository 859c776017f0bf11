"""Rows from host memory while the device is behind: what a call that waits for it does to the rest of the program."""
import threading
import time

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def keep_busy(ms):
    """Queues about `ms` milliseconds of work on the current stream (all of it host-side launches: a fraction of that)."""
    a = torch.randn(4096, 4096, device="cuda")
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    for timed in (False, True):  # the first product also sets the library up
        if timed:
            start.record()
        b = a @ a
    end.record()
    end.synchronize()
    for _ in range(int(ms / start.elapsed_time(end)) + 1):
        torch.mm(a, a, out=b)


@pytest.mark.parametrize("form", ["numpy", "cpu"])
def test_other_threads_run_while_an_insert_waits_for_the_device(form):
    """A call that comes around to staging memory which queued work has yet to read waits for it, without the
    interpreter's lock: a thread that wants to run every millisecond does so meanwhile."""
    from mindrl_amd.core import UniformReplayBuffer
    rows = 16
    b = UniformReplayBuffer(4, 64, [(28224,)], [torch.uint8])  # 451,584 bytes a call: a segment of the staging memory each
    frames = np.ones((rows, 28224), np.uint8)
    given = [frames if form == "numpy" else torch.from_numpy(frames)]
    for _ in range(8):
        b.insert(given)
    torch.cuda.synchronize()
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.is_set():
            ticks.append(time.perf_counter())
            time.sleep(0.001)

    thread = threading.Thread(target=tick)
    thread.start()
    try:
        keep_busy(400)
        began = time.perf_counter()
        for _ in range(5):  # the fifth finds the first one's segment, still to be read
            b.insert(given)
        ended = time.perf_counter()
    finally:
        stop.set()
        thread.join()
    assert ended - began > 0.1, "the inserts waited for no queued work: the test shows nothing"
    inside = [began] + [t for t in ticks if began < t < ended] + [ended]
    assert max(np.diff(inside)) < 0.5 * (ended - began)
    torch.cuda.synchronize()
    assert bool((b.buffer[0] == 1).all())
    b.destroy()
