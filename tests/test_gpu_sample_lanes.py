"""Samples of a thousand rows and more, sixteen lanes to a stratum (k_per_sample_lanes): trees of every number of staged levels and of
trips below them, rows of every form of the copy (sixteen lanes, a wave, several passes of it), last workgroups
of one row, the fewest and the most rows of each form, several batches at once, packed rows and the counters on the device. Indices,
weights and rows against the oracle (on the largest trees: against the kernel with a workgroup to a row)."""
import os
import re
import subprocess

import numpy as np
import pytest
import torch

from gpu_util import assert_sample_equal, kernels, random_rows, to_dev, torch_types

F, U, B, H, L, I = np.float32, np.uint8, np.bool_, np.float16, np.int64, np.int32
ROWS = {
    "narrow": ([(1,), (1,)], [I, F]),                                      # no wide field
    "48": ([(15,), (15,), (15,), (3,), (7, 7, 3)], [U, U, U, U, U]),       # as many narrow bytes as there may be
    "16": ([(17,), (6,), (1,), (17,), (1,)], [F, F, F, F, B]),             # up to 16 granules
    "32": ([(64,), (1,), (60,), (1,)], [F, I, F, B]),                      # up to 32
    "64": ([(777,), (19,), (45,), (1,), (1,)], [U, B, H, L, F]),           # up to 64
    "65": ([(1025,), (1,)], [U, F]),                                       # a wave, two granules to a lane
    "129": ([(1031,), (9,), (1,), (993,), (1,)], [U, F, F, U, B]),         # four
    "470": ([(50, 50, 3), (1,), (1,)], [U, I, F]),                         # eight
    "1280": ([(20463,), (17,), (1,)], [U, U, L]),                          # three passes; the largest rows
}


def _buffers(rows, cap, packed=0):
    from mindrl_amd.core import PriorityReplayBuffer
    from oracle import orc
    shapes, dtypes = ROWS[rows]
    rng = np.random.default_rng(cap)
    g = PriorityReplayBuffer(0.6, cap, 8, shapes, torch_types(dtypes), seed0=2, packed_rows=packed)
    c = orc.OraclePER(0.6, cap, shapes, dtypes, seed=2)
    new = random_rows(rng, cap, shapes, dtypes)
    pr = (np.abs(rng.normal(size=cap)) + 1e-3).astype(np.float32)
    g.insert(*to_dev(new), priorities=torch.from_numpy(pr).cuda())
    c.push(new, cap, pr)
    return g, c, rng


def _compare(g, c, rng, batch, n, what):
    g._sample_size = batch  # (one buffer for all batch sizes)
    if n > 1:
        out = g.sample_many(n, 0.4)
        for i in range(n):
            assert_sample_equal([o[i] for o in out], c.sample(batch, 0.4), "%s number %d" % (what, i))
        return
    assert_sample_equal(g.sample(0.4), c.sample(batch, 0.4), what)
    u = rng.random(batch).astype(np.float32)
    u[0], u[-1] = 0.0, np.float32(1.0) - np.float32(2.0 ** -24)
    assert_sample_equal(g.sample(0.4, uniforms=torch.from_numpy(u).cuda()), c.sample(batch, 0.4, u), what)


@pytest.mark.gpu
@pytest.mark.parametrize("cap", [100, 129, 1024, 2048, 2049, 4096, 4097, 20_000, 40_000, 131_072, 131_073, 300_001, 1_000_000,
                                 (1 << 20) + 1, (1 << 22) - 5])
@pytest.mark.parametrize("device_counters", [0, 1])
def test_trees(cap, device_counters):
    g, c, rng = _buffers("narrow", cap)
    g.set_option("device_counters", device_counters)
    for batch in (1280, 1665):
        _compare(g, c, rng, batch, 1, "%d leaves, batch %d" % (cap, batch))
    g.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,batches", [
    ("48", [(1280, 1), (1281, 1)]), ("16", [(1297, 1), (14_335, 1), (1, 1300), (431, 3)]), ("32", [(1280, 1), (20_479, 1)]),
    ("64", [(1536, 1), (12_287, 1), (7, 221)]), ("65", [(2048, 1), (3073, 1), (8193, 1)]),
    ("129", [(2049, 1), (3073, 1), (4096, 1), (4097, 1), (5633, 1), (700, 3)]), ("470", [(2048, 1), (2051, 1), (4099, 1), (5125, 1)]),
    ("1280", [(2048, 1), (2049, 1), (3601, 1), (4096, 1), (6001, 1), (6145, 1)])])
@pytest.mark.parametrize("packed", [0, 4096])
def test_rows(rows, batches, packed):
    g, c, rng = _buffers(rows, 1500, packed)
    for batch, n in batches:
        _compare(g, c, rng, batch, n, "rows %s, batch %d x %d" % (rows, batch, n))
    g.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("device_counters", [0, 1])
@pytest.mark.parametrize("cap,batch,n", [(20_000, 431, 5), (300_001, 100, 20)])
def test_several_batches(cap, batch, n, device_counters):
    """Each batch draws with a call number of the generator of its own, the host's or the device's."""
    g, c, rng = _buffers("16", cap)
    g.set_option("device_counters", device_counters)
    g._sample_size = batch
    assert any("k_per_sample_lanes" in name for name in kernels(lambda: g.sample_many(n, 0.4)))
    for _ in range(n):
        c.sample(batch, 0.4)
    for step in range(3):
        _compare(g, c, rng, batch, n, "call %d" % step)
    g.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("cap,device_counters", [((1 << 22) + 5, 0), ((1 << 23) + 1, 0), ((1 << 24) + 1, 1), ((1 << 25) + 1, 0), ((1 << 27) + 3, 0),
                                                 ((1 << 28) + 7, 0), ((1 << 29) + 11, 1)])
def test_very_large_trees(cap, device_counters):
    """23 to 25 levels: nine of them staged and two trips of seven or eight below; 26 and 28: twelve and two; 29 and 30: three trips. The
    same slots, weights and rows as the kernel with a workgroup to a row."""
    from mindrl_amd.core import PriorityReplayBuffer
    g = PriorityReplayBuffer(1.0, cap, 2049, [(1,)], [torch.uint8], seed0=2)
    g.insert(torch.arange(50_000, device="cuda").to(torch.uint8)[:, None])
    at = torch.randint(0, cap, (60_000,), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    at[:2] = torch.tensor([cap - 1, 0])
    g.update_priorities(at[:30_000], torch.rand(30_000, device="cuda") + 1e-3)
    g.update_priorities(at[30_000:], torch.rand(30_000, device="cuda") * 1e-3)
    u = torch.rand(2049, device="cuda")
    u[0], u[-1] = 0.0, 1.0 - 2.0 ** -24
    g.set_option("device_counters", device_counters)
    assert any("k_per_sample_lanes" in name for name in kernels(lambda: g.sample(0.4, uniforms=u)))
    seen = []
    for path in (0, 1):
        g.set_option("sample_path", path)
        seen.append(g.sample(0.4, uniforms=u))
    assert all(torch.equal(a, b) for a, b in zip(*seen))
    assert len(set(seen[0][0].tolist())) > 1000
    g.destroy()


@pytest.mark.gpu
def test_trees_that_were_never_filled():
    """Priorities of zero and slots without a row: the same slots and flags as the kernel with a workgroup to a row."""
    from mindrl_amd.core import PriorityReplayBuffer
    g = PriorityReplayBuffer(0.6, 5000, 1500, [(17,)], [torch.float32], seed0=5)
    g.insert(torch.arange(700 * 17, dtype=torch.float32, device="cuda").reshape(700, 17))
    for priorities in (torch.zeros(700), torch.full((700,), 1e-38), torch.cat([torch.zeros(699), torch.ones(1)])):
        g.update_priorities(torch.arange(700, device="cuda"), priorities.cuda())
        u = torch.rand(1500, device="cuda")
        seen = []
        for path in (0, 1):
            g.set_option("sample_path", path)
            out = g.sample(0.4, uniforms=u)
            try:
                g.check()
                flags = ""
            except Exception as e:
                flags = str(e)
            seen.append(([o.view(torch.int32) for o in out], flags))
        assert all(torch.equal(a, b) for a, b in zip(seen[0][0], seen[1][0])) and seen[0][1] == seen[1][1]
    g.destroy()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cap", [(r, c) for r in sorted(ROWS) + ["49"] for c in (100, 20_000, 200_000, 1_000_000, (1 << 20) + 1, (1 << 22) - 5)])
def test_the_benchmark_names_the_kernel_that_runs(rows, cap):
    import bench
    from mindrl_amd.core import PriorityReplayBuffer
    shapes, dtypes = ROWS.get(rows, ([(49,)] + [(1,)] * 4 + [(9,)] * 5, [U] * 10))
    if cap * sum(int(np.prod(s)) for s in shapes) > 1e9:
        cap = 20_000
    g = PriorityReplayBuffer(0.6, cap, 8, shapes, torch_types(dtypes), seed0=2)
    g.insert(*to_dev(random_rows(np.random.default_rng(cap), 5, shapes, dtypes)))
    for batch in (64, 1024, 1300, 1500, 2048, 2500, 4000, 5500, 6500, 13_000, 15_000, 21_000):
        g._sample_size = batch
        want, ran = bench.sample_kernel(g._layout.bytes, cap, batch), kernels(lambda: g.sample(0.4))
        assert any(want in name for name in ran), (batch, want, ran)
    g.destroy()


def test_registers(tmp_path):
    """No scratch memory, and no more registers than leave a compute unit two workgroups of eight waves (one where a lane holds
    eight granules of two rows)."""
    from mindrl_amd import build
    out = tmp_path / "kernels.s"
    flags = [f for f in build.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    res = subprocess.run(["/opt/rocm/bin/hipcc"] + flags + ["--cuda-device-only", "-S", "-o", str(out), os.path.join(build.CSRC, "mrb_sample_lanes.hip")],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout
    kernels = out.read_text().split("  - .agpr_count:")[1:]
    assert kernels
    for block in kernels:
        number = lambda key: int(re.search(r"\.%s:\s+(\d+)" % key, block).group(1))
        name = re.search(r"\.name:\s+(\S+)", block).group(1)
        assert number("private_segment_fixed_size") == 0, name
        assert number("vgpr_count") <= (168 if "ELb1ELi8E" in name else 128), name
