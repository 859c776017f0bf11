"""update_priorities by runs of leaves: on both sides of every line of its rule (entries and tree levels), with duplicates,
entries that name no leaf, invalid priorities, all entries in one tile and in one leaf, consecutive slots, and a capacity
that fills its last run only partly. Both trees and the running max against the oracle after every call, and the flags."""
import numpy as np
import pytest
import torch

from gpu_util import assert_tree_equal

pytestmark = pytest.mark.gpu


def flags_of(buf):
    try:
        buf.check()
        return ""
    except IndexError:
        return "index"
    except ValueError:
        return "priority"


@pytest.mark.parametrize("cap,sizes", [
    (513, (385, 2048)), (1000, (384, 385, 2048, 2049)), (4096, (385, 1024, 4097, 8192, 8193)), (5000, (384, 385, 1025, 4096)),
    (16_384, (385, 1024, 16_384, 16_385)), (16_385, (64, 65, 2047, 4097)), (65_536, (65, 129, 4096)), (100_000, (65, 512, 16_384)),
    (1_000_000, (65, 1024, 1025, 8191)), ((1 << 21) - 5, (65, 2048, 12_289, 16_385)), ((1 << 22) - 3, (65, 8192, 8193)),
    ((1 << 22) + 1, (65, 1025))])
def test_updates_by_runs_of_leaves(cap, sizes):
    from mindrl_amd.core import PriorityReplayBuffer
    from oracle import orc
    rng = np.random.default_rng(cap)
    g = PriorityReplayBuffer(0.7, cap, 8, [(1,)], [torch.int32], seed0=3)
    c = orc.OraclePER(0.7, cap, [(1,)], [np.int32], seed=3)
    fill = cap if cap < 200_000 else 150_000
    rows = np.zeros((fill, 1), np.int32)
    pr = (np.abs(rng.normal(size=fill)) + 1e-3).astype(np.float32)
    g.insert(torch.from_numpy(rows).cuda(), priorities=torch.from_numpy(pr).cuda())
    c.push([rows], fill, pr)
    flags_of(g)
    for n in sizes:
        for form in range(5):
            idx = rng.integers(0, cap, n)
            pr = (rng.pareto(1.5, n) + 1e-6).astype(np.float32)
            if form == 1:  # many duplicates, some of one leaf
                idx[: n // 2] = rng.integers(0, cap, max(1, n // 20)).repeat(20)[: n // 2][: idx[: n // 2].size] if n >= 40 else idx[0]
                idx[-n // 4:] = cap - 1
            if form == 2:  # one tile's worth of neighbours, in consecutive slots
                idx = (rng.integers(0, cap) + np.arange(n)) % cap
            if form == 3:  # everything aimed at one tile
                idx = np.minimum(idx[0] // 256 * 256 + rng.integers(0, 256, n), cap - 1)
            valid = np.ones(n, bool)
            if form == 4:  # entries to skip: no such slot, no such priority
                bad = rng.integers(0, n, 6)
                idx[bad[:3]] = [-1, cap, 1 << 40]
                pr[bad[3:]] = [-1.0, np.inf, np.nan]
                valid = (idx >= 0) & (idx < cap) & (pr >= 0) & (pr <= 3e38)
            g.update_priorities(torch.from_numpy(idx).cuda(), torch.from_numpy(pr).cuda())
            c.update(idx[valid], pr[valid])
            assert_tree_equal(g, c, "cap %d n %d form %d" % (cap, n, form))
            assert np.float32(g.max_priority) == np.float32(c.max_priority), (cap, n, form)
            assert flags_of(g) == ("index" if form == 4 and ((idx < 0) | (idx >= cap)).any() else
                                   "priority" if form == 4 else ""), (cap, n, form)
    g.destroy()
