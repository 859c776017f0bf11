"""Samples of many rows with large fields, which the LDS-top kernel copies field by field (large_field, mrb_lds_sample.h): rows on both sides
of its rules - granules of a field, whole and odd ones, bytes of the batch and of the rows held -, last workgroups of few strata, several batches. Slots and
weights against the workgroup-per-row kernel's for the same draws, rows against the buffer's at these slots, byte for byte."""
import numpy as np
import pytest
import torch

from gpu_util import random_rows, to_dev, torch_types

pytestmark = pytest.mark.gpu

U1, F4, I8, B1 = np.uint8, np.float32, np.int64, np.bool_


@pytest.mark.parametrize("shapes,types,cap,sizes", [
    ([(128,), (1,), (128,)], [F4, I8, F4], 3001, [(1, 12_288), (1, 41_003), (5, 16_384), (3, 4099)]),  # 32 granules: from 64 strata to a workgroup on
    ([(128,), (1,), (128,)], [F4, I8, F4], 70_001, [(5, 16_384), (3, 18_001)]),                        # (several batches, from buffers of some MB)
    ([(512,), (512,), (3,)], [F4, F4, U1], 9001, [(1, 12_289), (1, 12_300), (2, 6100), (2000, 7)]),    # 128: from sixteen on; fewer strata than a workgroup has
    ([(2031,), (1,), (5,)], [U1, I8, F4], 3001, [(1, 12_300), (1, 20_481), (1, 50_000), (1, 53_001)]),
    ([(2031,), (1,), (5,)], [U1, I8, F4], 100_003, [(1, 20_480), (1, 20_481), (1, 40_961), (1, 48_865), (1, 48_866)]),  # 127, odd: from 32 on, up to 96 MB
    ([(3069,), (17,), (1,), (100,)], [U1, B1, I8, F4], 60_001, [(1, 12_291), (2, 10_500), (1, 33_000)]),
    ([(1024,), (1,)], [F4, F4], 3001, [(1, 12_301), (1, 20_490)]),
    ([(5909,)], [U1], 36_001, [(1, 12_288)]),
    ([(64,), (1,), (64,)], [F4, I8, F4], 3001, [(1, 98_304), (1, 98_305), (1, 100_100)]),              # 16: from 256 strata on
    ([(32,), (17,)], [F4, U1], 3001, [(1, 98_305), (2, 50_003)]),                                       # 8
    ([(125,), (3,)], [U1, F4], 1_110_001, [(1, 98_305)]),                                               # (odd)
])
def test_rows(shapes, types, cap, sizes):
    from mindrl_amd.core import PriorityReplayBuffer
    rng = np.random.default_rng(len(sizes) + shapes[0][0])
    b = PriorityReplayBuffer(0.6, cap, 64, shapes, torch_types(types), seed0=3)
    new = to_dev(random_rows(rng, cap, shapes, types))
    b.insert(*new)
    b.update_priorities(torch.arange(cap, device="cuda"), torch.rand(cap, device="cuda") + 0.1)
    for nbatch, batch in sizes:
        b._sample_size = batch
        u = torch.rand(nbatch * batch, device="cuda")
        # (not the end of a batch's last stratum: with this many strata u + k rounds up to their number, and the sample may end on a
        # leaf past the rows, whose number is handed out as it is and is no index into them)
        u.reshape(nbatch, batch)[:, -1] = 0.25
        outs = []
        for path in (1, 2):
            b.set_option("sample_path", path)
            outs.append(b.sample(0.4, uniforms=u) if nbatch == 1 else b.sample_many(nbatch, 0.4, uniforms=u))
            b.set_option("sample_path", 0)
        assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1]), (nbatch, batch)
        slots = outs[1][0].reshape(-1)
        assert int(slots.min()) >= 0 and int(slots.max()) < cap, (nbatch, batch)
        for got, stored in zip(outs[1][2:], new):
            want = stored.reshape(cap, -1)[slots]
            assert torch.equal(got.reshape(want.shape).contiguous().view(torch.uint8), want.contiguous().view(torch.uint8)), (nbatch, batch)
    b.check()
    b.destroy()


@pytest.mark.parametrize("words,cap,nbatch,batch,large", [
    (512, 12_000, 1, 12_300, True), (512, 12_000, 2, 10_500, False), (512, 33_000, 2, 10_500, True),  # 23.5 MB of rows, and 65
    (275, 50_000, 5, 12_500, False), (512, 33_000, 1, 12_300, True)])
def test_rows_of_small_buffers_are_looked_up(words, cap, nbatch, batch, large):
    """Rows that come from the caches are copied by the kernel that is faster there."""
    from torch.profiler import ProfilerActivity, profile
    from mindrl_amd.core import PriorityReplayBuffer
    b = PriorityReplayBuffer(0.6, cap, batch, [(words * 4 + (words == 275),), (1,)], [torch.uint8, torch.int64], seed0=3)
    b.insert(torch.zeros(cap, words * 4 + (words == 275), dtype=torch.uint8, device="cuda"), torch.zeros(cap, 1, dtype=torch.int64, device="cuda"))
    call = (lambda: b.sample(0.4)) if nbatch == 1 else (lambda: b.sample_many(nbatch, 0.4))
    call()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        call()
        torch.cuda.synchronize()
    ran = [e.name for e in p.events() if "k_per_sample" in e.name]
    assert ran and all(("k_per_sample_lds_large" in name) == large and "k_per_sample_lds" in name for name in ran), ran
    b.destroy()
