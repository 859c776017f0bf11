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
