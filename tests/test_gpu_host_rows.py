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


@pytest.mark.parametrize("form", ["pinned", "numpy view", "converted", "pageable"])
@pytest.mark.parametrize("kind", ["uniform", "priority", "reservoir"])
def test_rows_that_queued_work_is_still_filling(kind, form):
    """A non-blocking copy from the device into host memory, then the insert, in the order of one stream and with no wait
    between: the rows are those of the copy, as when the insert itself was a copy on that stream."""
    from mindrl_amd.core import PriorityReplayBuffer, ReservoirReplayBuffer, UniformReplayBuffer
    n, shapes, types = 8, [(100,), (1,)], [torch.float32, torch.int64]
    b = (UniformReplayBuffer(4, n, shapes, types) if kind == "uniform" else
         PriorityReplayBuffer(0.6, n, 4, shapes, types, seed0=1) if kind == "priority" else
         ReservoirReplayBuffer(n, 4, shapes, types, seed0=1))
    ids = torch.arange(n)[:, None]
    host = torch.zeros((n, 100), dtype=torch.float64 if form == "converted" else torch.float32)
    if form != "pageable":
        host = host.pin_memory()
    rows = [host.numpy() if form == "numpy view" else host, ids]
    b.insert(rows)  # the staging memory is there: nothing but the rows themselves is waited for below
    torch.cuda.synchronize()
    keep_busy(100)
    host.copy_(torch.ones((n, 100), dtype=host.dtype, device="cuda"), non_blocking=True)
    b.insert(rows)
    views = b.buffer if kind == "uniform" else b.storage()
    stored = views[0].cpu()
    if kind == "reservoir":  # the second eight rows replace some of the first
        assert set(stored.sum(1).tolist()) <= {0.0, 100.0} and bool((stored.sum(1) == 100).any())
    else:
        assert bool((stored == 1).all())
    b.destroy()
