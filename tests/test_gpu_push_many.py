"""Pushes whose tiles several workgroups rebuild, against the oracle (buffers of up to 200,000 slots) and against the kernels that take
the same call where its matrices lie too far apart to be given as distances (more than 2^31 bytes at an odd address): trees, running
max, rows and flags, bit for bit. Runs of 1 to 257
tiles, aligned and not, up to the ring's end and around it, across the boundaries of the tiles 8 and 16 levels up; some priorities
invalid."""
import numpy as np
import pytest
import torch

from gpu_util import assert_tree_equal, bits, t2n

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def big():
    return torch.empty((1 << 31) + (1 << 25), dtype=torch.uint8, device="cuda")


def flags(buf):
    import ctypes

    from mindrl_amd import _lib
    f = ctypes.c_uint32(0)
    assert _lib.lib().mrb_per_check(buf._h, ctypes.byref(f), None) == 0
    return f.value


def trees(buf):
    return [bits(t[1:]) for t in buf.export_tree()] + [bits([buf.max_priority])]


T = 256
CASES = [  # capacity, first slot, rows
    (5000, 0, 2), (5000, 100, 156), (5000, 100, 157), (5000, 255, 2), (5000, 4999, 1), (5000, 4000, 1000), (5000, 4001, 1000),
    (5000, 0, 5000), (4097, 1, 4096), (100_000, 7 * T, 7 * T), (100_000, 7 * T, 8 * T), (100_000, 7 * T + 1, 8 * T),
    (100_000, 7 * T, 11 * T), (100_000, 7 * T, 12 * T), (60_000, 5, 12 * T), (60_000, T, 16 * T), (60_000, T + 1, 16 * T),
    (100_000, 65_536 - T, 2 * T), (100_000, 65_535, 2), (100_000, 60_000, 40_000), (100_000, 3, 160 * T), (100_000, 3, 159 * T),
    (200_000, 5, 256 * T), (200_000, 0, 256 * T), (200_000, 5, 255 * T), (200_000, 65_536 + 9, 97 * T),
    ((1 << 24) + 70_000, (1 << 24) - 300, 2), ((1 << 24) + 70_000, (1 << 24) - 300, 600), ((1 << 24) + 70_000, (1 << 24) - 2000, 65_000),
    ((1 << 24) + 70_000, (1 << 24) + 69_000, 1000),
]


@pytest.mark.parametrize("cap,first,n", CASES)
def test_push(cap, first, n, big):
    from mindrl_amd.core import PriorityReplayBuffer
    from oracle import orc
    a, b = (PriorityReplayBuffer(0.7, cap, 8, [(1,), (3,)], [torch.int32, torch.uint8], seed0=5) for _ in range(2))
    c = orc.OraclePER(0.7, cap, [(1,), (3,)], [np.int32, np.uint8]) if cap <= 200_000 else None
    rng = np.random.default_rng(first + n)
    for how in range(3):
        # up to the slot `first`: the ring's head is a multiple of the capacity away after each round
        lead = (first - (0 if how == 0 else first + n)) % cap
        for buf in (a, b):
            if lead:
                x = torch.arange(lead, device="cuda")
                buf.insert((x % 1000)[:, None].int(), (x[:, None] % torch.tensor([3, 5, 7], device="cuda")).to(torch.uint8),
                           priorities=(x % 97).float() + 0.5)
        if c is not None and lead:
            x = np.arange(lead)
            c.push([(x % 1000)[:, None].astype(np.int32), (x[:, None] % np.array([3, 5, 7])).astype(np.uint8)], lead, (x % 97 + 0.5).astype(np.float32))
        wide = torch.from_numpy(rng.integers(0, 1 << 30, (n, 1), dtype=np.int32)).cuda()
        small = torch.from_numpy(rng.integers(0, 256, (n, 3), dtype=np.uint8)).cuda()
        far0, far1 = big[: 4 * n].view(torch.int32).view(n, 1), big[(1 << 31) + 4099 : (1 << 31) + 4099 + 3 * n].view(n, 3)
        far0.copy_(wide)
        far1.copy_(small)
        pr = None
        if how:
            pr = (rng.pareto(1.5, n) * (100 if how == 2 else 1) + 1e-6).astype(np.float32)
            if how == 2:
                pr[rng.integers(0, n, 1 + n // 100)] = rng.choice(np.array([-1.0, np.inf, np.nan, 0.0], np.float32), 1 + n // 100)
            pr = torch.from_numpy(pr).cuda()
        a.insert(wide, small, priorities=pr)
        b.insert(far0, far1, priorities=pr)
        for x, y in zip(trees(a), trees(b)):
            assert np.array_equal(x, y), how
        for x, y in zip(a.storage(), b.storage()):
            assert np.array_equal(t2n(x), t2n(y)), how
        assert flags(a) == flags(b), how
        if c is not None:
            head, values = c.head, None if pr is None else t2n(pr)
            c.push([t2n(wide), t2n(small)], n)
            if pr is not None:  # (a row whose priority is invalid takes the running max)
                ok = (values >= 0) & (values <= 3e38)
                c.update(((head + np.arange(n)) % cap)[ok], values[ok])
            assert_tree_equal(a, c, how)
            assert np.float32(a.max_priority) == np.float32(c.max_priority), how
            for k, x in enumerate(a.storage()):
                assert np.array_equal(t2n(x), c.field(k).reshape(x.shape)), how


@pytest.mark.parametrize("n", [3, 290, 700, 9000])
def test_large_copies(n):
    """Copies of several granules to a thread, with the tiles' work and ahead of it: the rows lie where they belong."""
    from mindrl_amd.core import PriorityReplayBuffer, UniformReplayBuffer
    cap = 10_000
    shapes, types = [(4099,), (1031,), (1,)], [torch.int32, torch.uint8, torch.int64]
    a, u = PriorityReplayBuffer(0.7, cap, 8, shapes, types), UniformReplayBuffer(8, cap, shapes, types)
    g = torch.Generator(device="cuda").manual_seed(n)
    for first in (0, n):
        rows = [torch.randint(0, 200, (n,) + s, device="cuda", generator=g).to(t) for s, t in zip(shapes, types)]
        a.insert(*rows)
        u.insert(rows)
        for stored in (a.storage(), u.buffer):
            for x, y in zip(stored, rows):
                kept = min(n, cap - first)
                assert torch.equal(x[first : first + kept], y[:kept]) and torch.equal(x[: n - kept], y[kept:]), first
    s, m = a.export_tree()
    assert s[1] == min(2 * n, cap) and m[1] == 1.0


def test_replays():
    """A recorded call is replayed between the program's own."""
    from mindrl_amd.core import PriorityReplayBuffer
    cap, n = 100_000, 5000
    a, b = (PriorityReplayBuffer(0.7, cap, 8, [(1,)], [torch.int32], seed0=5) for _ in range(2))
    rows, pr = torch.zeros((n, 1), dtype=torch.int32, device="cuda"), torch.rand(n, device="cuda")
    for buf in (a, b):
        buf.insert(rows, priorities=pr)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        a.insert(rows, priorities=pr)
    for k in range(4):
        rows.fill_(k)
        pr.copy_(torch.rand(n, device="cuda") + k)
        g.replay()  # (writes the recorded slots)
        torch.cuda.synchronize()
        if k == 0:
            b.insert(rows, priorities=pr)
            for x, y in zip(trees(a), trees(b)):
                assert np.array_equal(x, y)
        a.insert(rows, priorities=pr)
        first = ((2 + k) * n) % cap
        got = [bits(t[1:]) for t in a.export_tree()]
        leaves = 1 << 17
        assert np.array_equal(got[0][leaves - 1 + n : leaves - 1 + 2 * n], got[0][leaves - 1 + first : leaves - 1 + first + n])
        s = got[0].view(np.float32)
        assert np.array_equal(s[: leaves - 1].view(np.int32), (s[1::2] + s[2::2]).astype(np.float32).view(np.int32))
