"""Pushes of a run of slots as one launch (a wave per leaf tile, up to 16, and the tiles above them): runs that start and
end on and beside tile edges, that cross the end of a tile eight or sixteen levels up, that wrap around the ring, on trees
whose last tile has 1 to 8 levels; plain and with priorities (invalid ones among them). Both trees, the running max and the
stored rows against the oracle after every push."""
import numpy as np
import pytest
import torch

from gpu_util import assert_tree_equal, random_rows, t2n, to_dev, torch_types

pytestmark = pytest.mark.gpu

SHAPES, DTYPES = [(3,), (1,)], [np.float32, np.int32]

# (capacity, first slots of the runs): 13 to 26 levels; 17 and 25 levels leave one level to the last tile, 18 and 26 two
CASES = [(5000, [0, 250, 4600, 4990]),
         (70_000, [0, 255, 65_000, 69_900]),
         (140_003, [65_300, 131_060, 139_990]),
         (1_000_000, [65_535, 65_530]),
         ((1 << 24) + 9, [65_400, 131_071]),
         ((1 << 25) + 1, [65_280])]


@pytest.mark.parametrize("device_counters", [0, 1])
@pytest.mark.parametrize("cap,starts", CASES)
def test_push_runs(cap, starts, device_counters):
    from mindrl_amd.core import PriorityReplayBuffer
    from oracle import orc
    rng = np.random.default_rng(cap)
    for start in starts:
        g = PriorityReplayBuffer(0.6, cap, 8, SHAPES, torch_types(DTYPES), seed0=3)
        c = orc.OraclePER(0.6, cap, SHAPES, DTYPES, seed=3)
        if start:
            rows = random_rows(rng, start, SHAPES, DTYPES)
            pr = (np.abs(rng.normal(size=start)) + 1e-3).astype(np.float32)
            g.insert(*to_dev(rows), priorities=torch.from_numpy(pr).cuda())
            c.push(rows, start, pr)
        g.set_option("device_counters", device_counters)
        for step, n in enumerate((2, 6, 255, 256, 257, 900, 3800, 4096)):
            if n > cap:
                continue
            rows = random_rows(rng, n, SHAPES, DTYPES)
            pr = None
            if step % 2:
                pr = (np.abs(rng.normal(size=n)) + 1e-3).astype(np.float32) * np.float32(1 + step)
                pr[n // 2] = -1.0  # keeps the running max as a plain push would
            g.insert(*to_dev(rows), priorities=None if pr is None else torch.from_numpy(pr).cuda())
            head = c.head
            c.push(rows, n)
            if pr is not None:  # a push with priorities is a push and then the update of its slots
                valid = np.arange(n) != n // 2
                c.update(((head + np.arange(n)) % cap)[valid], pr[valid])
            assert_tree_equal(g, c, "cap %d start %d n %d" % (cap, start, n))
            assert np.float32(g.max_priority) == np.float32(c.max_priority), (cap, start, n)
        for f, view in enumerate(g.storage()):
            assert np.array_equal(t2n(view[: c.size]).view(np.uint8), c.field(f)[: c.size].view(np.uint8))
        with pytest.raises(ValueError, match="priority"):
            g.check()
        g.destroy()


@pytest.mark.parametrize("device_counters", [0, 1])
@pytest.mark.parametrize("cap", [3000, 20_000, 70_000, 600_000])
def test_running_max_comes_from_the_pushed_priorities_alone(cap, device_counters):
    """A loaded state may hold leaves above its running max. A push with priorities raises the running max to the largest of
    its OWN powers, whatever lies beside its slots: one workgroup's pushes, runs of tiles, more tiles than a run takes, and
    pushes that follow an update in one call."""
    from mindrl_amd.core import PriorityReplayBuffer
    from oracle import orc
    rng = np.random.default_rng(cap)
    g = PriorityReplayBuffer(0.6, cap, 8, SHAPES, torch_types(DTYPES), seed0=3)
    c = orc.OraclePER(0.6, cap, SHAPES, DTYPES, seed=3)
    rows = random_rows(rng, cap, SHAPES, DTYPES)
    g.insert(*to_dev(rows), priorities=torch.full((cap,), 20.0, device="cuda"))
    c.push(rows, cap, np.full(cap, 20.0, np.float32))
    state = dict(g.state_dict(), max_priority=1e-3)  # far below the leaves, 20 ** 0.6
    g.load_state_dict(state)
    c.load_state_dict({**c.state_dict(), "max_priority": 1e-3})
    g.set_option("device_counters", device_counters)
    assert np.float32(g.max_priority) == np.float32(c.max_priority)
    largest = np.float32(1e-3)
    for step, n in enumerate((1, 3, 255, 900, 1500, 1, 5, 300, 5000)):
        if n > cap:
            continue
        largest *= np.float32(1.5)
        rows = random_rows(rng, n, SHAPES, DTYPES)
        pr = (largest * rng.random(n)).astype(np.float32)
        pr[n // 3] = largest
        slots = (c.head + np.arange(n)) % cap
        if step < 5:
            g.insert(*to_dev(rows), priorities=torch.from_numpy(pr).cuda())
        else:
            idx, low = rng.integers(0, cap, 100), np.full(100, 1e-6, np.float32)
            g.update_priorities_and_insert(torch.from_numpy(idx).cuda(), torch.from_numpy(low).cuda(), *to_dev(rows),
                                           insert_priorities=torch.from_numpy(pr).cuda())
            c.update(idx, low)
        c.push(rows, n)
        c.update(slots, pr)
        assert np.float32(g.max_priority) == np.float32(c.max_priority) < np.float32(1.0), (cap, n)
        assert_tree_equal(g, c, "cap %d n %d" % (cap, n))
    g.destroy()


# 8 levels, which one workgroup rebuilds whole, and 9 to 12: one to four levels above the leaf tiles
@pytest.mark.parametrize("device_counters", [0, 1])
@pytest.mark.parametrize("cap,starts", [(256, [0, 200]), (257, [0, 250]), (510, [255, 500]), (512, [0, 511]), (1000, [0, 513, 990]),
                                        (2048, [255, 2040]), (2049, [1, 2000]), (4096, [0, 300, 4000])])
def test_push_runs_on_small_trees(cap, starts, device_counters):
    test_push_runs(cap, starts, device_counters)


@pytest.mark.parametrize("cap", [257, 1000, 4096])
def test_saved_small_trees(cap):
    """A state that is loaded takes the way of a push of all slots."""
    from mindrl_amd.core import PriorityReplayBuffer
    rng = np.random.default_rng(cap)
    a = PriorityReplayBuffer(0.6, cap, 8, SHAPES, torch_types(DTYPES), seed0=3)
    b = PriorityReplayBuffer(0.6, cap, 8, SHAPES, torch_types(DTYPES), seed0=4)
    for n in (2, cap // 2, cap):
        a.insert(*to_dev(random_rows(rng, n, SHAPES, DTYPES)), priorities=torch.from_numpy(rng.pareto(1.5, n).astype(np.float32)).cuda())
        b.load_state_dict(a.state_dict())
        assert all(np.array_equal(x[1:], y[1:]) for x, y in zip(a.export_tree(), b.export_tree())) and a.max_priority == b.max_priority
        a.check(), b.check()
    a.destroy()
    b.destroy()
