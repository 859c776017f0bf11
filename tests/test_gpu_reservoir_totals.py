"""Reservoir pushes around the 2^32nd row, up to which the later rows' slots are drawn with 32-bit bounds, and of calls whose rows replace
one another at totals just below and above small powers of two: storage against the oracle."""
import numpy as np
import pytest
import torch

from gpu_util import t2n

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("capacity,total,sizes", [(1 << 22, (1 << 32) - 6000, (4096, 1903, 1, 4096)), (1 << 22, (1 << 32) - 4097, (4096, 4096)),
                                                  (700, 700, (700, 699, 2, 700)), (4096, 65_530, (4096, 4000)), (4100, 1 << 20, (4096, 4100))])
def test_around(capacity, total, sizes):
    from mindrl_amd.core import ReservoirReplayBuffer
    from oracle import orc
    rng = np.random.default_rng(total % 1000)
    g = ReservoirReplayBuffer(capacity, 8, [(1,)], [torch.uint8], seed0=5)
    c = orc.OracleReservoir(capacity, [(1,)], [np.uint8], seed=5)
    start = [np.zeros((min(capacity, 5000), 1), np.uint8)]
    g.push(*[torch.from_numpy(r).cuda() for r in start])
    c.push(start, len(start[0]))
    state = g.state_dict()
    state.update(size=capacity, total=total, fields=[torch.zeros(capacity, 1, dtype=torch.uint8)])
    g.load_state_dict(state)
    state["fields"] = [f.numpy() for f in state["fields"]]
    c.load_state_dict(state)
    for n in sizes:
        new = [rng.integers(1, 256, (n, 1)).astype(np.uint8)]
        g.push(*[torch.from_numpy(r).cuda() for r in new])
        c.push(new, n)
        assert (g.size(), g.total()) == (c.size, c.total)
        assert np.array_equal(t2n(g.storage()[0]), c.field(0)), n
    g.destroy()
