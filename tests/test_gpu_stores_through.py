"""Batches on both sides of the sizes from which, and up to which, their rows are stored through the caches (store_granule, mrb_rows.h), by each of the
kernels that do so: a workgroup to a row with one and with several large fields, the same with the next observation, a wave to a
row, and granules numbered over all rows. Rows against the buffer's own at the returned slots, byte for byte, also of calls replayed
from a graph into tensors that have been cleared."""
import numpy as np
import pytest
import torch

from gpu_util import random_rows, to_dev, torch_types

pytestmark = pytest.mark.gpu

LINE, GATHERS_LINE, BROKEN_LINE = 20 << 20, 40 << 20, 160 << 20  # samples and gathers from the first and the second on; stores that end within 64 bytes up to the last
ROWS = {  # (the second field: a slot number)
    "frames": ([(84, 84, 4), (1,), (1,)], [np.uint8, np.int64, np.float32]),
    "odd": ([(48, 51, 3), (1,), (307,), (1,), (9,)], [np.uint8, np.int64, np.float32, np.bool_, np.float16]),
    "pair": ([(5008,), (1,), (5003,)], [np.uint8, np.int64, np.uint8]),
    "wave": ([(905,), (1,), (3,)], [np.float32, np.int64, np.uint8]),
    "flat": ([(130,), (1,), (131,)], [np.float32, np.int64, np.float32]),
}


def same_rows(out, stored, slots):
    for o, s in zip(out, stored):
        want = s.reshape(s.shape[0], -1)[slots.reshape(-1).clamp(max=s.shape[0] - 1)].reshape(o.shape)  # (as the rows are: a number past them is no index)
        assert torch.equal(o.contiguous().view(torch.uint8), want.contiguous().view(torch.uint8))


def row_bytes(shapes, dtypes):
    return sum(int(np.prod(s)) * np.dtype(d).itemsize for s, d in zip(shapes, dtypes))


def filled(make, rows, cap, insert):
    shapes, dtypes = ROWS[rows]
    b = make(shapes, torch_types(dtypes))
    new = to_dev(random_rows(np.random.default_rng(7), cap, shapes, dtypes))
    new[1] = torch.randint(0, cap, (cap, 1), device="cuda")
    insert(b, new)
    return b, new


@pytest.mark.parametrize("rows", ["frames", "odd", "pair", "wave", "flat"])
def test_uniform(rows):
    from mindrl_amd.core import UniformReplayBuffer
    size = row_bytes(*ROWS[rows])
    cap = GATHERS_LINE // size * 5 // 4 + 5
    for n in (LINE // size, LINE // size + 1, GATHERS_LINE // size, GATHERS_LINE // size + 1, cap):
        b, new = filled(lambda s, t: UniformReplayBuffer(n, cap, s, t, seed=3), rows, cap, lambda b, new: b.insert(new))
        for _ in range(2):
            slots, out = b.sample_with_indices()
            same_rows(out, new, slots)
        given = torch.randint(0, cap, (n,), device="cuda")
        same_rows(b.sample(indices=given), new, given)
        b.check()
        b.destroy()


@pytest.mark.parametrize("rows", ["frames", "odd", "pair"])
def test_prioritized(rows):
    from mindrl_amd.core import PriorityReplayBuffer
    cap, size = 700, row_bytes(*ROWS[rows])
    b, new = filled(lambda s, t: PriorityReplayBuffer(0.6, cap, 64, s, t, seed0=3), rows, cap, lambda b, new: b.insert(*new))
    b.update_priorities(torch.arange(cap, device="cuda"), torch.rand(cap, device="cuda") + 0.1)
    first = int(np.prod(ROWS[rows][0][0]))
    for n in (LINE // size, LINE // size + 1, LINE // (size + first), LINE // (size + first) + 1):
        b._sample_size = n
        out = b.sample(0.4)
        same_rows(out[2:], new, out[0])
        out = b.sample_with_next(0.4, slot_field=1, row_field=0)
        same_rows(out[2:-1], new, out[0])
        same_rows(out[-1:], new[:1], new[1].reshape(-1)[out[0]])
    b._sample_size = 211
    out = b.sample_many(1 + LINE // (211 * size), 0.4)
    same_rows(out[2:], new, out[0])
    b.check()
    b.destroy()


def test_replayed():
    from mindrl_amd.core import PriorityReplayBuffer
    cap, n = 700, LINE // row_bytes(*ROWS["frames"]) + 9
    b, new = filled(lambda s, t: PriorityReplayBuffer(0.6, cap, n, s, t, seed0=3), "frames", cap, lambda b, new: b.insert(*new))
    b.set_option("device_counters", 1)
    out = b.sample(0.4)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(torch.cuda.Stream()):
        graph.capture_begin()
        b.sample(0.4, out=(out[0], out[1], list(out[2:])))
        graph.capture_end()
    torch.cuda.synchronize()
    seen = []
    for _ in range(4):
        for o in out:
            o.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        same_rows(out[2:], new, out[0])
        seen.append(out[0].clone())
    assert not torch.equal(seen[0], seen[1])
    b.destroy()


@pytest.mark.parametrize("shape", [(192, 8192, 1), (1024, 8192, 1), (1025, 8192, 1), (2049, 4095, 1), (2047, 1365, 3), (1025, 2730, 3), (7, 3, 1)])
def test_returns(shape):
    """Returns and their gradient on both sides of the size up to which they are stored so, bit for bit: the recurrence, an operation
    at a time."""
    from mindrl_amd.utils import DiscountedReturn
    rng = np.random.default_rng(shape[0])
    x, w = [rng.normal(size=shape).astype(np.float32) for _ in range(2)]
    done, value = rng.random(shape[:2]) < 0.03, rng.normal(size=shape[1:]).astype(np.float32)
    c = ((np.float32(1) - done.astype(np.float32)) * np.float32(0.97))[..., None]
    want, last = np.empty_like(x), value
    for t in reversed(range(shape[0])):
        want[t] = last = x[t] + c[t] * last
    grad, last = np.empty_like(x), np.zeros_like(value)
    for t in range(shape[0]):
        grad[t] = last = w[t] + (c[t - 1] * last if t else 0)
    X, V = [torch.from_numpy(a).cuda().requires_grad_(True) for a in (x, value)]
    for _ in range(2):
        out = DiscountedReturn(0.97, need_bprop=True)(X, torch.from_numpy(done).cuda(), V)
        gx, gv = torch.autograd.grad(out, (X, V), torch.from_numpy(w).cuda())
        assert np.array_equal(out.detach().cpu().numpy(), want)
        assert np.array_equal(gx.cpu().numpy(), grad)
        assert np.array_equal(gv.cpu().numpy(), c[-1] * grad[-1])


@pytest.mark.parametrize("rows", ["frames", "odd", "wave", "flat"])
def test_more_than_the_memorys_cache_takes(rows):
    from mindrl_amd.core import PriorityReplayBuffer, UniformReplayBuffer
    cap, size = 700, row_bytes(*ROWS[rows])
    for n in (BROKEN_LINE // size, BROKEN_LINE // size + 9):
        b, new = filled(lambda s, t: UniformReplayBuffer(n, cap, s, t, seed=3), rows, cap, lambda b, new: b.insert(new))
        given = torch.randint(0, cap, (n,), device="cuda")
        same_rows(b.sample(indices=given), new, given)
        b.check()
        b.destroy()
        b, new = filled(lambda s, t: PriorityReplayBuffer(0.6, cap, n, s, t, seed0=3), rows, cap, lambda b, new: b.insert(*new))
        out = b.sample(0.4)
        same_rows(out[2:], new, out[0])
        b.check()
        b.destroy()
