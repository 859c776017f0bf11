"""The native host side of the buffer classes: rows from host memory through the staging memory (numpy arrays, CPU tensors,
a mix with device tensors, other dtypes, more than the staging memory takes, segments used again while earlier calls are
still queued), and results that are tensors of their own."""
import io

import numpy as np
import pytest
import torch

from gpu_util import random_rows, t2n, to_dev, torch_types

pytestmark = pytest.mark.gpu

SHAPES, DTYPES = [(5,), (3,), (1,), (2,), (1,)], [np.float32, np.uint8, np.int64, np.float16, np.bool_]


def buffers():
    from mindrl_amd.core import PriorityReplayBuffer, ReservoirReplayBuffer, UniformReplayBuffer
    types = torch_types(DTYPES)
    per = PriorityReplayBuffer(0.6, 400, 16, SHAPES, types, seed0=3)
    urb = UniformReplayBuffer(16, 400, SHAPES, types, seed=3)
    res = ReservoirReplayBuffer(400, 16, SHAPES, types, seed0=3)
    return [(per, lambda rows: per.insert(*rows), per.storage()), (urb, urb.insert, urb.buffer), (res, lambda rows: res.push(*rows), res.storage())]


def as_given(rows, form):
    if form == "numpy":
        return rows
    if form == "cpu":
        return [torch.from_numpy(r) for r in rows]
    if form == "mixed":
        return [torch.from_numpy(r).cuda() if i % 2 else r for i, r in enumerate(rows)]
    if form == "negated":  # views whose memory holds the opposite of their values
        return [torch._neg_view(-torch.from_numpy(r)) if r.dtype in (np.float32, np.int64) else r for r in rows]
    if form == "converted":  # dtypes that need converting, not contiguous
        return [rows[0].astype(np.float64), rows[1].astype(np.int32), rows[2].tolist(), torch.from_numpy(rows[3]).float(),
                torch.from_numpy(np.repeat(rows[4], 2, axis=1))[:, ::2]]
    return to_dev(rows)


@pytest.mark.parametrize("form", ["device", "numpy", "cpu", "mixed", "converted", "negated"])
def test_rows_from_host_memory(form):
    rng = np.random.default_rng(5)
    for buf, put, views in buffers():
        at = 0
        for n in (1, 2, 7, 100, 1, 200):
            rows = random_rows(rng, n, SHAPES, DTYPES)
            put(as_given(rows, form))
            for v, r in zip(views, rows):
                assert np.array_equal(t2n(v[at:at + n]).view(np.uint8), r.view(np.uint8)), (type(buf).__name__, form, n)
            at += n
        with pytest.raises(ValueError):
            put(as_given(random_rows(rng, 2, SHAPES, DTYPES), form)[:-1])  # a field missing
        bad = random_rows(rng, 2, SHAPES, DTYPES)
        bad[1] = bad[1][:1]  # fields that disagree on the number of rows
        with pytest.raises(ValueError):
            put(bad)
        buf.destroy()


@pytest.mark.parametrize("per_call", [1, 18, 19, 40])  # 28 KB, just under and just over a segment (512 KiB), over a megabyte
def test_staging_memory_is_used_again_behind_queued_work(per_call):
    """More host rows than the staging memory holds, in calls that nothing waits between, behind work that keeps the
    stream busy: every row arrives as it was when its call was made."""
    from mindrl_amd.core import UniformReplayBuffer
    calls = 200 if per_call == 1 else 12
    b = UniformReplayBuffer(4, calls * per_call, [(84, 84, 4), (1,)], [torch.uint8, torch.int64])
    busy = torch.randn(2048, 2048, device="cuda")
    frames = np.zeros((per_call, 84, 84, 4), np.uint8)
    for k in range(calls):
        if k % 4 == 0:
            busy = (busy @ busy).clamp_(-1, 1)
        frames[:] = k % 251  # the caller's array is its own again when the call returns
        ids = np.arange(k * per_call, (k + 1) * per_call)[:, None]
        b.insert([frames, ids])
    want = torch.arange(calls).repeat_interleave(per_call)
    assert torch.equal(b.buffer[1][:, 0].cpu(), want * 0 + torch.arange(calls * per_call))
    assert torch.equal(b.buffer[0].amin(dim=(1, 2, 3)).cpu().long(), want % 251)
    assert torch.equal(b.buffer[0].amax(dim=(1, 2, 3)).cpu().long(), want % 251)
    b.destroy()


def test_results_are_tensors_of_their_own():
    per, put, _ = buffers()[0]
    put(to_dev(random_rows(np.random.default_rng(1), 300, SHAPES, DTYPES)))
    first = per.sample(0.4)
    kept = [t.clone() for t in first]
    assert all(t.is_contiguous() and t.data_ptr() % 256 == 0 and t.device.index == 0 for t in first)
    second = per.sample(0.4)
    for t in second:
        t.zero_()
    for i, t in enumerate(first):  # neither the next call's results nor the other results of the call change with one
        assert torch.equal(t, kept[i])
        t.fill_(1)
        assert all(torch.equal(u, kept[j]) for j, u in enumerate(first) if j > i)
    weights = per.sample(0.4)[1].requires_grad_(True)
    (weights * 2).sum().backward()
    assert torch.equal(weights.grad, torch.full_like(weights, 2))
    per.destroy()
    with pytest.raises(ValueError):
        per.sample(0.4)


def test_fields_of_many_dimensions():
    from mindrl_amd.core import PriorityReplayBuffer
    shape = (1,) * 20 + (2,) + (1,) * 20 + (3,)
    per = PriorityReplayBuffer(0.6, 8, 4, [shape, (1,)], [torch.float32, torch.int64], seed0=3)
    rows = torch.randn((8,) + shape)
    per.insert(rows.cuda(), torch.arange(8)[:, None].cuda())
    idx, _, got, ids = per.sample(0.4)
    assert got.shape == (4,) + shape and torch.equal(got.cpu(), rows[idx.cpu()]) and torch.equal(ids[:, 0], idx)
    per.destroy()


def test_results_have_storages_of_their_own():
    """A result can be grown in place, given as out= of a larger result, or saved, without the call's other results."""
    from mindrl_amd.core import PriorityReplayBuffer
    per = PriorityReplayBuffer(0.6, 400, 16, SHAPES, torch_types(DTYPES), seed0=3)
    rows = to_dev(random_rows(np.random.default_rng(1), 300, SHAPES, DTYPES))
    per.insert(*rows)
    step = lambda: per.update_priorities_insert_and_sample(torch.arange(4, device="cuda"), torch.ones(4, device="cuda"),
                                                           *[r[:1] for r in rows], beta=0.4)
    for call in (lambda: per.sample(0.4), lambda: per.sample_many(2, 0.4), lambda: per.gather(torch.arange(16, device="cuda")), step):
        results = call()
        kept = [t.clone() for t in results]
        for i, t in enumerate(results):
            assert t.untyped_storage().nbytes() == t.numel() * t.element_size() and t.storage_offset() == 0
            saved = io.BytesIO()
            torch.save(t, saved)
            assert torch.equal(torch.load(io.BytesIO(saved.getvalue()), weights_only=True), kept[i])
            t.resize_(50_000).zero_()
            assert all(torch.equal(u, kept[j]) for j, u in enumerate(results) if j > i)
    per.destroy()


def test_given_outputs_that_do_not_hold_the_batch_are_refused():
    """`out` with indices or weights of too few rows, another dtype or device: refused before anything is written or changed."""
    per, put, _ = buffers()[0]
    rows = to_dev(random_rows(np.random.default_rng(1), 300, SHAPES, DTYPES))
    put(rows)
    good = per.sample(0.4)
    idx, w, fields = good[0], good[1], list(good[2:])
    step = lambda out: per.update_priorities_insert_and_sample(torch.arange(4, device="cuda"), torch.ones(4, device="cuda"),
                                                               *[r[:1] for r in rows], beta=0.4, out=out)
    for call in (lambda out: per.sample(0.4, out=out), step):
        size = per.size()
        for bad in ((idx[:15], w, fields), (idx, w[:15], fields), (idx.int(), w, fields), (idx, w.double(), fields),
                    (idx.cpu(), w, fields), (idx, torch.empty(32, device="cuda")[::2], fields), (idx, w, fields[:-1])):
            with pytest.raises(ValueError):
                call(bad)
        assert per.size() == size
        larger = (torch.empty(20, dtype=torch.int64, device="cuda"), torch.empty(20, device="cuda"), fields)
        assert call(larger)[0] is larger[0]  # more room than needed is fine: the first rows are written
    per.destroy()


def test_calls_follow_the_current_stream():
    from mindrl_amd.core import UniformReplayBuffer
    b = UniformReplayBuffer(64, 64, [(4,)], [torch.float32], seed=2)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        rows = torch.randn(4096, 4096, device="cuda").softmax(1)[:64, :4].contiguous()  # work ahead of the insert on s
        b.insert([rows])
        idx, (out,) = b.sample_with_indices()
    s.synchronize()
    assert torch.equal(out, rows[idx])
    b.destroy()


def test_host_rows_on_streams_that_run_unordered():
    """The staging memory's segments come round while the OTHER stream's work that reads them is still queued: the rows of
    a stream that is far behind are its own all the same."""
    from mindrl_amd.core import UniformReplayBuffer
    per_call, calls, floats = 16, 24, 1500  # 96,000 bytes a call: five to a segment
    b = UniformReplayBuffer(16, per_call * calls, [(floats,)], [torch.float32], seed=2)
    behind, ahead = torch.cuda.Stream(), torch.cuda.Stream()
    busy = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    for k in range(calls):
        late = k % 8 == 0
        with torch.cuda.stream(behind if late else ahead):
            if late:
                for _ in range(4):
                    busy = (busy @ busy).clamp_(-1, 1)
            b.insert([np.full((per_call, floats), k, np.float32)])
    torch.cuda.synchronize()
    want = torch.arange(calls, dtype=torch.float32).repeat_interleave(per_call)
    assert torch.equal(b.buffer[0].cpu(), want[:, None].expand(-1, floats))
    b.destroy()
