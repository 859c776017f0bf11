"""Gathers that number the granules of a field over all rows: on both sides of the number from which on a thread takes four, of
rows that went to other kernels before, in up to eight fields; drawn slots and given ones, some of them no slot of the buffer."""
import numpy as np
import pytest
import torch

from gpu_util import kernels, random_rows, t2n, to_dev, torch_types

pytestmark = pytest.mark.gpu

F, U, L, B, H = np.float32, np.uint8, np.int64, np.bool_, np.float16


CASES = [
    ([(1024,), (1,), (1,), (1,)], [U, L, F, B], (64, 4096, 4097, 5248, 5249, 9000)),  # 64 granules: 1024 workgroups (drawn: 1312), and more
    ([(301,), (9,), (1,), (301,), (1,)], [F, F, F, F, B], (500, 3449, 3450)),      # two large fields, one of three granules
    ([(1,), (2413,), (5,), (45,), (999,), (3, 3), (33,)], [B, U, F, H, U, U, L], (1700, 1737)),  # the first one small, all of odd sizes
    ([(7500,)] + [(1,)] * 7, [U] * 8, (425, 426, 2230, 2236)),                     # eight fields; around those with a workgroup to a row
    ([(28224,), (1,)], [U, L], (113, 114, 594, 595)),
    ([(4096,), (1,)], [U, L], (7031, 7032)),                                       # around those with a wave to a row
    ([(300,), (300,), (5, 51), (1,)], [F, F, U, B], (10_843, 10_844)),
]


def _row(shapes, dtypes):
    return sum(int(np.prod(s)) * np.dtype(d).itemsize for s, d in zip(shapes, dtypes))


# (packed rows have at most 4096 bytes)
@pytest.mark.parametrize("packed,shapes,dtypes,batches", [(0,) + c for c in CASES] + [(4096,) + c for c in CASES if _row(*c[:2]) <= 4096])
def test_flat_gathers(packed, shapes, dtypes, batches):
    from mindrl_amd.core import UniformReplayBuffer
    from oracle import orc
    rng = np.random.default_rng(len(shapes))
    cap = max(batches) + 50
    for batch in batches:
        g = UniformReplayBuffer(batch, cap, shapes, torch_types(dtypes), seed=4, packed_rows=packed)
        c = orc.OracleUniform(cap, shapes, dtypes, seed=4)
        new = random_rows(rng, cap - 30, shapes, dtypes)
        g.insert(to_dev(new))
        c.append(new, cap - 30)
        idx, fields = g.sample_with_indices() if len(shapes) < 8 else (None, g.sample())
        want_idx, want = c.sample(batch)
        assert idx is None or np.array_equal(t2n(idx), want_idx), batch
        assert all(np.array_equal(t2n(a), b) for a, b in zip(fields, want)), batch
        given = rng.integers(0, cap - 30, batch)
        fields = g.sample(torch.from_numpy(given).cuda())
        assert all(np.array_equal(t2n(a), b[given]) for a, b in zip(fields, new)), batch
        g.check()
        given[batch // 2], given[-1] = cap - 30, -1
        fields = g.sample(torch.from_numpy(given).cuda())
        with pytest.raises(IndexError):
            g.check()
        given = np.clip(given, 0, cap - 31)
        assert all(np.array_equal(t2n(a), b[given]) for a, b in zip(fields, new)), batch
        g.destroy()


def _time(call, n=20):
    best = []
    for _ in range(5):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(n):
            call()
        end.record()
        torch.cuda.synchronize()
        best.append(start.elapsed_time(end) / n)
    return min(best)


@pytest.mark.parametrize("shapes,dtypes,n", [([(28224,), (1,)], [U, L], 4096), ([(400,), (1,), (1,), (400,)], [F, F, F, F], 8192)])
def test_rows_outside_are_flagged_once_each(shapes, dtypes, n):
    """Flags go to one word, one atomic after the other, 11 ns each: one for each such row, not one for each of its granules, so a
    batch of nothing but such rows takes the time of its atomics at most on top of its copy."""
    from mindrl_amd.core import UniformReplayBuffer
    rng = np.random.default_rng(3)
    g = UniformReplayBuffer(n, 5000, shapes, torch_types(dtypes))
    g.insert(to_dev(random_rows(rng, 5000, shapes, dtypes)))
    good = torch.from_numpy(rng.integers(0, 5000, n)).cuda()
    took = _time(lambda: g.sample(good))
    g.check()
    bad = _time(lambda: g.sample(good + 5000 * (1 + good % 2)))
    with pytest.raises(IndexError):
        g.check()
    assert bad < took + 0.03 + n * 15e-6, (took, bad)  # (ms; two small kernels work out the slots)
    g.destroy()


@pytest.mark.parametrize("option,kernel", [(0, "k_short_gather"), (1, "k_rows_gather_rows"), (2, "k_rows_gather_wide")])
def test_row_wave(option, kernel):
    """1 asks for a wave to a row, 2 forbids it."""
    from mindrl_amd.core import UniformReplayBuffer
    g = UniformReplayBuffer(2048, 5000, [(1024,), (1,)], torch_types([U, L]))
    g.insert(to_dev([np.zeros((5000, 1024), U), np.zeros((5000, 1), L)]))
    g.set_option("row_wave", option)
    g.sample()
    ran = kernels(lambda: g.sample())
    assert any(kernel in name for name in ran), ran
    g.destroy()
