"""Updates driven by their entries on very large trees, at every depth at which the plan changes: groups of four, eight and
sixteen lanes per entry, runs of 4, 8 and 16 tiles, and the round of tiles in between from 27 levels on. Every node above
a written leaf is compared with sums and minima taken level by level in numpy (the exponent is 1, so a leaf is its
priority), and a few thousand others with what they were."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def levels_above(capacity, idx, pr):
    """(nodes, sums, minima) per level, from the leaves up, of the nodes above the written leaves of an empty buffer."""
    depth = max(1, (capacity - 1).bit_length())
    last = dict(zip(idx.tolist(), range(len(idx))))  # the last entry aimed at a leaf wins
    nodes = np.array(sorted(last), np.int64)
    sums = pr[[last[i] for i in nodes.tolist()]]
    mins = sums.copy()
    nodes += 1 << depth
    yield nodes, sums, mins
    for _ in range(depth):
        parents, at = np.unique(nodes >> 1, return_inverse=True)
        pair_s = np.zeros((len(parents), 2), np.float32)
        pair_m = np.full((len(parents), 2), np.finfo(np.float32).max, np.float32)
        pair_s[at, nodes & 1] = sums
        pair_m[at, nodes & 1] = mins
        nodes, sums, mins = parents, pair_s[:, 0] + pair_s[:, 1], pair_m.min(1)
        yield nodes, sums, mins


@pytest.mark.parametrize("capacity,n", [((1 << 22) - 1, 8193), ((1 << 22) - 1, 16384), ((1 << 22) + 1, 1025), (1 << 23, 32768),
                                        (1 << 24, 65536), ((1 << 24) + 5, 20011), ((1 << 26) - 3, 4097), ((1 << 26) + 3, 30000)])
def test_every_node_above_the_entries(capacity, n):
    from mindrl_amd.core import PriorityReplayBuffer
    g = PriorityReplayBuffer(1.0, capacity, 4, [(1,)], [torch.uint8], seed0=1)
    rng = np.random.default_rng(n)
    idx = np.sort(rng.integers(0, capacity, n))
    idx[n // 2:] = rng.permutation(idx[n // 2:])
    idx[:200] = capacity - 1 - np.arange(200) // 2  # the last tiles, twice each
    idx[200:300] = 77  # one leaf, many times
    pr = (rng.pareto(1.5, n) + 1e-6).astype(np.float32)
    for _ in range(2):  # an update on the nodes that an update left
        pr = pr[::-1].copy()
        g.update_priorities(torch.from_numpy(idx).cuda(), torch.from_numpy(pr).cuda())
    sums, mins = g.export_tree()
    touched = []
    for nodes, want_s, want_m in levels_above(capacity, idx, pr):
        assert np.array_equal(sums[nodes], want_s) and np.array_equal(mins[nodes], want_m), int(nodes[0]).bit_length() - 1
        touched.append(nodes)
    others = np.setdiff1d(rng.integers(1, len(sums), 4096), np.concatenate(touched))
    assert not sums[others].any() and (mins[others] == np.finfo(np.float32).max).all()
    assert g.check() == 0
    g.destroy()


# (21 levels' own lines: fewer entries go by runs of leaves, more by tiles; and the most entries of 22 to 24 levels)
@pytest.mark.parametrize("capacity,n", [((1 << 21) - 7, 3072), ((1 << 21) - 7, 3073), ((1 << 20) + 1, 20_000), (1 << 21, 32_768), (1 << 21, 32_769),
                                        ((1 << 22) - 1, 3072), ((1 << 22) - 1, 3073), (1 << 22, 131_072), (1 << 22, 131_073),
                                        ((1 << 23) - 1, 262_144), ((1 << 24) - 1, 262_144)])
def test_where_the_entries_take_over(capacity, n):
    test_every_node_above_the_entries(capacity, n)


# entries of a wave bid for their leaf among themselves first: many of them on one leaf, on leaves that lie together, entries that
# count for nothing behind those that do
@pytest.mark.parametrize("capacity,n", [((1 << 14) - 1, 20_000), (1 << 20, 20_000), ((1 << 21) - 7, 3073), (1 << 21, 16_385), ((1 << 22) - 1, 8193), (1 << 24, 65_537)])
def test_many_entries_on_few_leaves(capacity, n):
    from mindrl_amd.core import PriorityReplayBuffer
    rng = np.random.default_rng(n)
    wild = rng.integers(0, capacity, n)
    for idx in (np.full(n, capacity // 3), np.where(rng.random(n) < 0.5, capacity // 3, wild), np.sort(rng.integers(0, 100, n)) * (capacity // 100),
                5 + np.arange(n) // 7 % capacity, 3 + rng.integers(0, 5, n) * 128 % capacity):
        g = PriorityReplayBuffer(1.0, capacity, 4, [(1,)], [torch.uint8], seed0=1)
        pr = (rng.pareto(1.5, n) + 1e-6).astype(np.float32)
        bad = rng.random(n) < 0.3
        bad[-3:] = True
        given, at = np.where(bad & (np.arange(n) % 2 == 0), np.float32(-1), pr), np.where(bad & (np.arange(n) % 2 == 1), -1 - idx, idx)
        g.update_priorities(torch.from_numpy(at).cuda(), torch.from_numpy(given).cuda())
        sums, mins = g.export_tree()
        for nodes, want_s, want_m in levels_above(capacity, idx[~bad], pr[~bad]):
            assert np.array_equal(sums[nodes], want_s) and np.array_equal(mins[nodes], want_m), int(nodes[0]).bit_length() - 1
        assert np.float32(g.max_priority) == max(pr[~bad].max(), np.float32(1.0))
        with pytest.raises((IndexError, ValueError)):
            g.check()
        g.destroy()


@pytest.mark.parametrize("capacity,n", [(1 << 20, 65_536), (1 << 21, 16_384), (1 << 22, 8192), (1 << 24, 65_536)])
def test_many_entries_on_one_leaf_take_no_longer(capacity, n):
    """One after the other their bids would take 11 ns each: 8 to 70 times as long as an update of as many leaves."""
    from mindrl_amd.core import PriorityReplayBuffer
    g = PriorityReplayBuffer(0.6, capacity, 4, [(1,)], [torch.uint8], seed0=1)
    pr, took = torch.rand(n, device="cuda") + 0.01, []
    for idx in (torch.randint(0, capacity, (n,), device="cuda"), torch.full((n,), capacity // 3, device="cuda")):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        best = []
        for _ in range(5):
            start.record()
            for _ in range(20):
                g.update_priorities(idx, pr)
            end.record()
            torch.cuda.synchronize()
            best.append(start.elapsed_time(end))
        took.append(min(best))
    assert took[1] < 2.5 * took[0], took
    g.destroy()
