"""Reservoir pushes past the capacity in one launch and in two: on both sides of the rule that chooses (rows of the call,
bytes of a row, rows against the capacity), around multiples of a workgroup's rows, with calls most of whose rows replace
one another and calls that begin before the buffer is full. Storage and totals against the oracle after every call."""
import numpy as np
import pytest
import torch

from gpu_util import t2n, torch_types

pytestmark = pytest.mark.gpu

SMALL = ([(17,), (1,), (5,)], [np.float32, np.int32, np.float32])      # 8 granules, 16 rows to a workgroup at 4096
ODD = ([(147,), (1,), (3,), (1,)], [np.uint8, np.int64, np.float16, np.bool_])
LARGE = ([(84, 84, 4), (1,)], [np.uint8, np.int64])                    # a workgroup per row
LARGEST = ([(70_000,)], [np.uint8])                                    # more granules than a workgroup takes


@pytest.mark.parametrize("rows,cap,sizes", [
    (SMALL, 2, (3, 2, 2, 1)), (SMALL, 64, (65, 2, 63, 64)), (SMALL, 1000, (900, 999, 17, 16, 15, 1000, 1001)),
    (SMALL, 5000, (4990, 33, 1025, 4096, 4097, 5000)), (SMALL, 9001, (9001, 4095, 8192, 8193)), (ODD, 700, (650, 511, 700, 2, 129)),
    (ODD, 6000, (6000, 5793, 2049)), (LARGE, 300, (299, 2, 257, 300)), (LARGE, 1500, (1500, 1448, 1449)), (LARGEST, 20, (20, 5, 19))])
@pytest.mark.parametrize("packed", [False, True])
def test_pushes_past_the_capacity(rows, cap, sizes, packed):
    from mindrl_amd.core import ReservoirReplayBuffer
    from oracle import orc
    shapes, dtypes = rows
    if packed and rows in (LARGE, LARGEST):
        pytest.skip("rows too large to pack")
    rng = np.random.default_rng(cap)
    g = ReservoirReplayBuffer(cap, 8, shapes, torch_types(dtypes), seed0=5, packed_rows=4096 if packed else 0)
    c = orc.OracleReservoir(cap, shapes, dtypes, seed=5)
    for n in sizes:
        new = [rng.integers(0, 2 if d == np.bool_ else 100, (n,) + s).astype(d) for s, d in zip(shapes, dtypes)]
        g.push(*[torch.from_numpy(r).cuda() for r in new])
        c.push(new, n)
        assert (g.size(), g.total()) == (c.size, c.total)
        for f, view in enumerate(g.storage()):
            assert np.array_equal(t2n(view).view(np.uint8), c.field(f).view(np.uint8)), (n, f)
    g.destroy()
