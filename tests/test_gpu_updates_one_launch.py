"""Updates of up to 4096 entries, and the push that follows one of up to 1024 in the same call, in one launch: on both sides of the lines of
their rules (tree levels, entries, how many runs of leaves the tree is divided into), against the oracle bit for bit. Forms:
duplicates, entries that name no leaf and invalid priorities, everything in one tile, consecutive slots; pushes of one row to
more than a launch takes, across a run's end and around the ring's, over slots the entries name, with a new running max in the
same call, with and without (some invalid) priorities of their own. Recorded launches are replayed."""
import numpy as np
import pytest
import torch

from gpu_util import assert_tree_equal, t2n, to_dev

pytestmark = pytest.mark.gpu


def pair(cap, fill, seed=3):
    from mindrl_amd.core import PriorityReplayBuffer
    from oracle import orc
    g = PriorityReplayBuffer(0.7, cap, 8, [(1,)], [torch.int32], seed0=seed)
    c = orc.OraclePER(0.7, cap, [(1,)], [np.int32], seed=seed)
    rng = np.random.default_rng(cap)
    for at in range(0, fill, 200_000):
        n = min(200_000, fill - at)
        rows, pr = np.arange(at, at + n, dtype=np.int32)[:, None], (np.abs(rng.normal(size=n)) + 1e-3).astype(np.float32)
        g.insert(torch.from_numpy(rows).cuda(), priorities=torch.from_numpy(pr).cuda())
        c.push([rows], n, pr)
    return g, c, rng


def entries(rng, cap, n, form):
    idx, pr = rng.integers(0, cap, n), (rng.pareto(1.5, n) + 1e-6).astype(np.float32)
    if form == 1:
        idx[: n // 2] = idx[0]  # duplicates: the last entry wins
    if form == 2:
        idx = (rng.integers(0, cap) + np.arange(n)) % cap
    if form == 3:
        idx = np.minimum(idx[0] // 256 * 256 + rng.integers(0, 256, n), cap - 1)
    if form == 4:
        bad = rng.integers(0, n, 6)
        idx[bad[:3]] = [-1, cap, 1 << 40]
        pr[bad[3:]] = [-1.0, np.inf, np.nan]
    return idx, pr, (idx >= 0) & (idx < cap) & (pr >= 0) & (pr <= 3e38)


def flags(buf):
    from mindrl_amd import _lib
    import ctypes
    f = ctypes.c_uint32(0)
    assert _lib.lib().mrb_per_check(buf._h, ctypes.byref(f), None) == 0
    return f.value & 3


def same(g, c, what):
    assert_tree_equal(g, c, what)
    assert np.float32(g.max_priority) == np.float32(c.max_priority), what


@pytest.mark.parametrize("cap", [129, 257, 1000, 1025, 2048, 4095, 4097, 16_384, 16_385, 65_536, 100_000, 131_073, 300_007, (1 << 20) + 1,
                                 (1 << 22) - 3])
def test_updates(cap):
    g, c, rng = pair(cap, cap if cap < 200_000 else 150_000)
    flags(g)
    for n in (1, 2, 64, 96, 97, 192, 193, 255, 256, 257, 512, 513, 1024, 1025, 2049, 4096, 4097):
        for form in range(5):
            idx, pr, ok = entries(rng, cap, n, form)
            g.update_priorities(*to_dev([idx, pr]))
            c.update(idx[ok], pr[ok])
            what = "cap %d n %d form %d" % (cap, n, form)
            same(g, c, what)
            bad_index, bad_priority = ((idx < 0) | (idx >= cap)).any(), not ((pr >= 0) & (pr <= 3e38)).all()
            assert flags(g) == (1 if bad_index else 0) + (2 if bad_priority else 0), what
    g.destroy()


@pytest.mark.parametrize("cap", [130, 1000, 2050, 5000, 16_384, 30_000, 70_000, 300_007, (1 << 20) + 1, (1 << 22) - 3])
def test_updates_with_a_push(cap):
    g, c, rng = pair(cap, min(cap - 3, 180_000))
    serial = 0
    # (512 rows are the most a launch takes; the ring's end is met again and again where the capacity is small)
    for step, (n, nrows) in enumerate([(64, 1), (1, 1), (512, 4), (65, 5), (1024, 300), (256, 512), (257, 513), (100, 1), (1024, 1), (512, 129),
                                       (33, 512), (700, 2)]):
        nrows = min(nrows, cap)
        for ipr_form in range(3):
            idx, pr, ok = entries(rng, cap, n, step % 5 if n >= 6 else 0)
            head = c.head
            if step % 2:  # slots the push overwrites: the push's value must win
                idx[-1], ok[-1] = (head + nrows - 1) % cap, (pr[-1] >= 0) & (pr[-1] <= 3e38)
                idx[0], ok[0] = head, (pr[0] >= 0) & (pr[0] <= 3e38)
            if ipr_form == 0 and step % 3 == 0:
                pr[n // 2] = np.float32(1e3 * (step + 2))  # a new running max that the pushed rows take
                ok[n // 2] = 0 <= idx[n // 2] < cap
            ipr = None
            if ipr_form:
                ipr = (np.abs(rng.normal(size=nrows)) + 1e-6).astype(np.float32)
                if ipr_form == 2:
                    ipr[0] = -1.0 if nrows > 1 else np.nan  # takes the running max, as a row without a priority
            rows = [np.arange(serial, serial + nrows, dtype=np.int32)[:, None]]
            serial += nrows
            g.update_priorities_and_insert(*to_dev([idx, pr]), *to_dev(rows), insert_priorities=None if ipr is None else torch.from_numpy(ipr).cuda())
            c.update(idx[ok], pr[ok])
            c.push(rows, nrows)
            if ipr is not None:
                given = (ipr >= 0) & (ipr <= 3e38)
                c.update(((head + np.arange(nrows)) % cap)[given], ipr[given])
            what = "cap %d step %d (%d entries, %d rows, %d)" % (cap, step, n, nrows, ipr_form)
            same(g, c, what)
            assert g.size() == c.size and g._state()[1] == c.head, what
            want = (0 if ok.all() and ((idx >= 0) & (idx < cap)).all() else (1 if ((idx < 0) | (idx >= cap)).any() else 0)) | \
                (2 if not ((pr >= 0) & (pr <= 3e38)).all() or ipr_form == 2 else 0)
            assert flags(g) == want, what
    assert np.array_equal(t2n(g.storage()[0]), c.field(0).reshape(g.storage()[0].shape))
    g.destroy()


def test_recorded_updates_count_their_launches_on_the_device():
    """The number that tells one launch's roots from the next one's lives on the device: a recorded launch, replayed with
    other entries each time and the program's own updates between the replays, leaves the trees of the eager twin."""
    cap, n = 200_000, 700
    g, c, rng = pair(cap, cap)
    idx, pr = torch.zeros(n, dtype=torch.int64, device="cuda"), torch.ones(n, device="cuda")
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        g.update_priorities(idx, pr)
        g.update_priorities(idx, pr)
    for step in range(6):
        i, p, ok = entries(rng, cap, n, step % 4)
        idx.copy_(torch.from_numpy(i)), pr.copy_(torch.from_numpy(p))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        c.update(i, p), c.update(i, p)
        same(g, c, "replay %d" % step)
        i, p, ok = entries(rng, cap, 300, 0)
        g.update_priorities(*to_dev([i, p]))
        c.update(i, p)
        same(g, c, "after replay %d" % step)
    g.destroy()


def test_two_buffers_on_two_streams():
    cap, n = 100_000, 512
    pairs = [pair(cap, cap, seed) for seed in (1, 2)]
    streams = [torch.cuda.Stream() for _ in pairs]
    data = [[entries(rng, cap, n, k % 4) for k in range(20)] for _, _, rng in pairs]
    dev = [[to_dev(d[:2]) for d in ds] for ds in data]
    torch.cuda.synchronize()
    for k in range(20):
        for (g, _, _), s, d in zip(pairs, streams, dev):
            with torch.cuda.stream(s):
                g.update_priorities(*d[k])
    torch.cuda.synchronize()
    for (g, c, _), ds in zip(pairs, data):
        for i, p, _ in ds:
            c.update(i, p)
        same(g, c, "two streams")
        g.destroy()
