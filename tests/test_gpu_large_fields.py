"""Samples of many rows with large fields, which the LDS-top kernel copies field by field (large_field, mrb_lds_sample.h): rows on both sides
of its rules - granules of a field, whole and odd ones, bytes of the batch -, last workgroups of few strata, several batches. Slots and
weights against the workgroup-per-row kernel's for the same draws, rows against the buffer's at these slots, byte for byte."""
import numpy as np
import pytest
import torch

from gpu_util import random_rows, to_dev, torch_types

pytestmark = pytest.mark.gpu

U1, F4, I8, B1 = np.uint8, np.float32, np.int64, np.bool_


@pytest.mark.parametrize("shapes,types,sizes", [
    ([(128,), (1,), (128,)], [F4, I8, F4], [(1, 12_288), (1, 41_003), (5, 16_384), (3, 4099)]),      # 32 granules: from 64 strata to a workgroup on
    ([(512,), (512,), (3,)], [F4, F4, U1], [(1, 12_289), (1, 12_300), (2, 12_288)]),                  # 128: from sixteen on
    ([(2031,), (1,), (5,)], [U1, I8, F4], [(1, 12_300), (1, 20_481), (1, 50_000), (1, 53_001)]),      # 127, odd: from 32 on, up to 96 MB
    ([(3069,), (17,), (1,), (100,)], [U1, B1, I8, F4], [(1, 12_291), (2, 10_500), (1, 33_000)]),
    ([(1024,), (1,)], [F4, F4], [(1, 12_301), (1, 20_490)]),
    ([(5909,)], [U1], [(1, 12_288)]),
])
def test_rows(shapes, types, sizes):
    from mindrl_amd.core import PriorityReplayBuffer
    cap = 3001
    rng = np.random.default_rng(len(sizes) + shapes[0][0])
    b = PriorityReplayBuffer(0.6, cap, 64, shapes, torch_types(types), seed0=3)
    new = to_dev(random_rows(rng, cap, shapes, types))
    b.insert(*new)
    b.update_priorities(torch.arange(cap, device="cuda"), torch.rand(cap, device="cuda") + 0.1)
    for nbatch, batch in sizes:
        b._sample_size = batch
        u = torch.rand(nbatch * batch, device="cuda")
        outs = []
        for path in (1, 2):
            b.set_option("sample_path", path)
            outs.append(b.sample(0.4, uniforms=u) if nbatch == 1 else b.sample_many(nbatch, 0.4, uniforms=u))
            b.set_option("sample_path", 0)
        assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1]), (nbatch, batch)
        slots = outs[1][0].reshape(-1)
        for got, stored in zip(outs[1][2:], new):
            want = stored.reshape(cap, -1)[slots]
            assert torch.equal(got.reshape(want.shape).contiguous().view(torch.uint8), want.contiguous().view(torch.uint8)), (nbatch, batch)
    b.check()
    b.destroy()
