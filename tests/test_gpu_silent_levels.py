"""The three levels above the leaves are not kept up on trees of 15 levels and more (kSilentLevels, mrb_tree.h): whatever reads or
rebuilds such a tree must do without them. Updates of every size class, pushes of one row and of several, both as one call, and samples by
every kernel, one after the other on one buffer without an export in between (which writes the levels), against the oracle; then
both trees, node by node."""
import numpy as np
import pytest
import torch

from gpu_util import assert_sample_equal, assert_tree_equal, random_rows, to_dev, torch_types

pytestmark = pytest.mark.gpu

SHAPES, TYPES = [(5,), (1,)], [np.float32, np.int32]


@pytest.mark.parametrize("capacity", [(1 << 14) + 1, 1 << 15, (1 << 16) - 3, (1 << 17) + 9, (1 << 19) - 1, 1 << 20, (1 << 21) - 5, (1 << 22) - 300])
@pytest.mark.parametrize("options", [{}, {"device_counters": 1}, {"fused_rebuild": 0}])
def test_nothing_needs_them(capacity, options):
    run(capacity, options, sizes=(1, 5, 64, 70, 500, 1024, 1025, 3000, 5000, 20_000), batches=(64, 1500, 4096, 20_000))


# 23 to 26 levels: paths of a wave, groups of four, eight and sixteen lanes
@pytest.mark.parametrize("capacity", [(1 << 23) - 1, (1 << 24) - 11, (1 << 25) - 7, (1 << 26) - 1])
def test_nothing_needs_them_on_very_large_trees(capacity):
    run(capacity, {}, sizes=(3, 64, 700, 5000, 40_000), batches=(64, 2048, 20_000))


def run(capacity, options, sizes, batches):
    from mindrl_amd.core import PriorityReplayBuffer
    from oracle import orc
    rng = np.random.default_rng(capacity % 1000 + len(options))
    shapes, types = (SHAPES, TYPES) if capacity < 1 << 23 else ([(1,)], [np.uint8])
    g = PriorityReplayBuffer(0.6, capacity, 64, shapes, torch_types(types), seed0=3)
    c = orc.OraclePER(0.6, capacity, shapes, types, seed=3)
    for name, value in options.items():
        g.set_option(name, value)

    def push(n, with_priorities):
        rows = random_rows(rng, n, shapes, types)
        pr = (rng.pareto(1.5, n) + 1e-3).astype(np.float32) if with_priorities else None
        g.insert(*to_dev(rows), priorities=None if pr is None else torch.from_numpy(pr).cuda())
        c.push(rows, n, pr)

    def entries(n):
        idx = rng.integers(0, capacity, n)
        idx[::7] = idx[0]
        if rng.random() < 0.5:
            idx.sort()
        return idx, (rng.pareto(1.5, n) + 1e-3).astype(np.float32)

    def sample():
        for path in (0, 1, 2):
            g.set_option("sample_path", path)
            for levels in (0, 12) if path == 2 else (0,):
                g.set_option("lds_levels", levels)
                for batch in batches:
                    g._sample_size = batch
                    u = rng.random(batch).astype(np.float32)
                    assert_sample_equal(g.sample(0.4, uniforms=torch.from_numpy(u).cuda()), c.sample(batch, 0.4, u), "%d by %d" % (batch, path))
        g.set_option("sample_path", 0)

    push(capacity, True)
    push(777, False)  # (the ring's position)
    for n in sizes:
        if n > 1024 and options.get("device_counters"):
            continue
        idx, pr = entries(n)
        g.update_priorities(torch.from_numpy(idx).cuda(), torch.from_numpy(pr).cuda())
        c.update(idx, pr)
        for rows, with_priorities in ((1, False), (1, True), (4, False), (300, True)):
            push(rows, with_priorities)
        m = min(n, 64)
        idx, pr = entries(m)
        rows = random_rows(rng, 1, shapes, types)
        g.update_priorities_and_insert(torch.from_numpy(idx).cuda(), torch.from_numpy(pr).cuda(), *to_dev(rows))
        c.update(idx, pr)
        c.push(rows, 1)
    push(6000, False)
    push(1, True)
    sample()
    idx, pr = entries(64)
    g.update_priorities(torch.from_numpy(idx).cuda(), torch.from_numpy(pr).cuda())
    c.update(idx, pr)
    assert_tree_equal(g, c, "capacity %d" % capacity)
    assert np.float32(g.max_priority) == np.float32(c.max_priority)
    push(1, False)
    assert_tree_equal(g, c, "capacity %d, after an export" % capacity)
    g.destroy()
