"""Rows of every size around the copy granules (16 bytes, 8, 4, 2, 1; the last granule of a row lies over the one before it)
through every kernel that copies rows: ring append and gather, the prioritized sample's kernels (workgroup per row, wave per
row, LDS top), the pushes that carry rows along, the whole-step kernel, the reservoir; array per field and packed rows.
Neighbouring rows are compared too: a granule past its row would show there."""
import numpy as np
import pytest
import torch

from gpu_util import assert_sample_equal, random_rows, t2n, to_dev, torch_types

pytestmark = pytest.mark.gpu

GROUPS = [list(range(1, 17)), list(range(17, 33)), [1, 33, 2, 47, 48, 49, 3, 63, 64, 65, 5, 95, 127, 128, 129, 7],
          [15, 255, 257, 31, 1023, 1025], [4095, 4097, 9], [28_223, 1, 3], [40_001]]


def assert_storage_equal(views, oracle, n, rows):
    for f in range(n):
        assert np.array_equal(t2n(views[f][:rows]), oracle.field(f)[:rows]), f


@pytest.mark.parametrize("packed", [0, 1])
@pytest.mark.parametrize("group", range(len(GROUPS)))
def test_rows_of_odd_sizes(group, packed):
    from mindrl_amd.core import PriorityReplayBuffer, ReservoirReplayBuffer, UniformReplayBuffer
    from oracle import orc
    shapes = [(s,) for s in GROUPS[group]]
    if packed and sum(GROUPS[group]) + 32 > 4096:
        pytest.skip("rows too large to pack")
    packed_rows = 4096 if packed else 0
    dtypes = [np.uint8] * len(shapes)
    types = torch_types(dtypes)
    rng = np.random.default_rng(group)
    cap, batch = 600, 70
    # uniform: append, wrap, draws, given slots, one item
    g = UniformReplayBuffer(batch, cap, shapes, types, seed=4, packed_rows=packed_rows)
    c = orc.OracleUniform(cap, shapes, dtypes, seed=4)
    for n in (1, 333, 300, 65):
        rows = random_rows(rng, n, shapes, dtypes)
        g.insert(to_dev(rows))
        c.append(rows, n)
    assert_storage_equal(g.buffer, c, len(shapes), cap)
    idx, fields = g.sample_with_indices()
    want_idx, want = c.sample(batch)
    assert np.array_equal(t2n(idx), want_idx) and all(np.array_equal(t2n(a), b) for a, b in zip(fields, want))
    assert all(np.array_equal(t2n(a), b) for a, b in zip(g.get_item(7), c.get_item(7)))
    g.destroy()
    # reservoir past its capacity
    g = ReservoirReplayBuffer(cap, batch, shapes, types, seed0=9, packed_rows=packed_rows)
    c = orc.OracleReservoir(cap, shapes, dtypes, seed=9)
    for n in (500, 1, 400):
        rows = random_rows(rng, n, shapes, dtypes)
        g.push(*to_dev(rows))
        c.push(rows, n)
    assert_storage_equal(g.storage(), c, len(shapes), cap)
    g.destroy()
    # prioritized: pushes of one and of many rows, the sample's kernels, the whole step
    g = PriorityReplayBuffer(0.6, cap, batch, shapes, types, seed0=2, packed_rows=packed_rows)
    c = orc.OraclePER(0.6, cap, shapes, dtypes, seed=2)
    for n in (1, 599, 3, 1):
        rows = random_rows(rng, n, shapes, dtypes)
        g.insert(*to_dev(rows))
        c.push(rows, n)
    assert_storage_equal(g.storage(), c, len(shapes), cap)
    for path, wave in ((1, 2), (1, 1), (2, 0)):
        g.set_option("sample_path", path)
        g.set_option("row_wave", wave)
        u = rng.random(batch).astype(np.float32)
        assert_sample_equal(g.sample(0.4, uniforms=torch.from_numpy(u).cuda()), c.sample(batch, 0.4, u), "path %d %d" % (path, wave))
    g.set_option("sample_path", 0)
    for n in (40, 100):
        idx = rng.integers(0, cap, n)
        pr = (np.abs(rng.normal(size=n)) + 1e-3).astype(np.float32)
        row = random_rows(rng, 1, shapes, dtypes)
        u = rng.random(batch).astype(np.float32)
        out = g.update_priorities_insert_and_sample(torch.from_numpy(idx).cuda(), torch.from_numpy(pr).cuda(), *to_dev(row), beta=0.4,
                                                    uniforms=torch.from_numpy(u).cuda())
        c.update(idx, pr)
        c.push(row, 1)
        assert_sample_equal(out, c.sample(batch, 0.4, u), "step")
    assert_storage_equal(g.storage(), c, len(shapes), cap)
    slots = rng.integers(0, cap, 33)
    got = g.gather(torch.from_numpy(slots).cuda())
    assert all(np.array_equal(t2n(a), c.field(f)[slots]) for f, a in enumerate(got))
    g.destroy()


@pytest.mark.parametrize("size", [147, 444, 813])
def test_large_batches_of_odd_rows(size):
    """Batches for which the wave-per-row and the LDS-top sample kernels are taken by size."""
    from mindrl_amd.core import PriorityReplayBuffer
    from oracle import orc
    shapes, dtypes = [(size,), (1,), (size // 3,)], [np.uint8, np.int64, np.float16]
    rng = np.random.default_rng(size)
    cap = 20_011
    for batch in (3001, 8193):
        g = PriorityReplayBuffer(0.6, cap, batch, shapes, torch_types(dtypes), seed0=2)
        c = orc.OraclePER(0.6, cap, shapes, dtypes, seed=2)
        rows = random_rows(rng, cap, shapes, dtypes)
        g.insert(*to_dev(rows))
        c.push(rows, cap)
        assert_sample_equal(g.sample(0.4), c.sample(batch, 0.4), "batch %d" % batch)
        g.destroy()
