"""What a program that trains with these buffers has them do, as cases that can be timed and compared.

Five kinds of pass, all through the public classes of `mindrl_amd.core` and `mindrl_amd.utils`:

  per_step     a learner's step on a PriorityReplayBuffer: the priorities of the batch it has just used, the
               transitions the actors have produced meanwhile, and the batch it uses next
               (`update_priorities`, `insert`, `sample`; or the calls that combine them)
  per_sample   batches drawn from a PriorityReplayBuffer between two updates (`sample`, `sample_with_next`,
               `sample_many`)
  uniform      a step on a UniformReplayBuffer (`insert`, `sample`)
  reservoir    a step on a ReservoirReplayBuffer past its capacity (`push`, `sample`)
  returns      `DiscountedReturn` over a rollout, with or without its gradients

A row is written as text, one entry per field: type:shape, e.g. "f4:17;f4:6;f4:1;f4:17;b1:1".
"""
import math

import numpy as np
import torch

from mindrl_amd.core import PriorityReplayBuffer, ReservoirReplayBuffer, UniformReplayBuffer
from mindrl_amd.utils import DiscountedReturn

_TYPES = {"f4": torch.float32, "f2": torch.float16, "i8": torch.int64, "i4": torch.int32, "u1": torch.uint8, "b1": torch.bool}

_CARTPOLE = "f4:4;i4:1;f4:1;f4:4;b1:1"
_MUJOCO = "f4:17;f4:6;f4:1;f4:17;b1:1"
_ATARI = "u1:84,84,4;i8:1;i4:1;f4:1;b1:1"
_APEX = "f4:64;i4:1;f4:1;f4:64;b1:1"


def listed():
    return [
        # DQN on a small control task. The environment runs on the host, so the new transition is host arrays; the
        # three calls are the reference's loop. Everything here is latency.
        dict(name="dqn_step", kind="per_step", calls=3, capacity=10_000, rows=_CARTPOLE, batch=64, update=0, insert=1,
             with_priorities=False, host_rows=True, priorities="normal", fill=1.0),
        # The same step as the one call that combines the three, with the new transition already on the device.
        dict(name="dqn_one_call", kind="per_step", calls=1, capacity=10_000, rows=_CARTPOLE, batch=64, update=0, insert=1,
             with_priorities=False, host_rows=False, priorities="normal", fill=1.0),
        # DQN on stacked frames: one batch of images out of the full buffer of a million.
        dict(name="atari_sample", kind="per_sample", capacity=1_000_000, rows=_ATARI, batch=512, nbatch=1,
             priorities="lognormal"),
        # The learner's whole step on frames, with the next observation stored as a slot number: update and insert as
        # one call, then the batch together with its next observations.
        dict(name="atari_step", kind="per_step", calls=2, capacity=100_000, rows=_ATARI, batch=512, update=0, insert=4,
             with_priorities=False, host_rows=False, priorities="lognormal", fill=1.0, following=True),
        # A learner that takes several gradient steps between updates: sixteen batches at once. The largest case.
        dict(name="atari_prefetch", kind="per_sample", capacity=250_000, rows=_ATARI, batch=512, nbatch=16,
             priorities="lognormal"),
        # Distributed actors that compute their own initial priorities: 4096 new rows, 2048 updates (some of them of
        # the same slot, heavy-tailed), a batch of 1024.
        dict(name="apex_step", kind="per_step", calls=3, capacity=1 << 21, rows=_APEX, batch=1024, update=2048, insert=4096,
             with_priorities=True, host_rows=False, priorities="normal", fill=1.0),
        # A very deep tree over rows of 8 bytes and very large batches: the descent and the rebuild are everything.
        dict(name="deep_tree_step", kind="per_step", calls=3, capacity=1 << 24, rows="i4:1;f4:1", batch=65_536, update=0,
             insert=64, with_priorities=False, host_rows=False, priorities="mixture", fill=1.0),
        # Prioritized replay of a robot's long state vectors, an odd number of floats each, in a buffer of no round
        # size that is still filling up.
        dict(name="odd_rows_step", kind="per_step", calls=3, capacity=300_007, rows="f4:111;f4:9;f4:1;f4:111;b1:1", batch=250,
             update=0, insert=5, with_priorities=False, host_rows=False, priorities="normal", fill=0.61),
        # SAC: one environment step, one batch.
        dict(name="sac_step", kind="uniform", capacity=1_000_000, rows=_MUJOCO, batch=256, insert=1, host_rows=False, fill=1.0),
        # Many environments side by side with small byte images, action masks and half-precision features: a chunk
        # in, a large batch out; no field is a multiple of 16 bytes.
        dict(name="masked_batch", kind="uniform", capacity=400_003, rows="u1:7,7,3;b1:19;f2:45;i8:1;f4:1", batch=8192,
             insert=1000, host_rows=False, fill=1.0),
        # Average-policy learning: everything ever seen is offered to the reservoir, batches come out of it.
        dict(name="reservoir_step", kind="reservoir", capacity=1_000_000, rows="f4:17;i4:1;f4:5", batch=256, insert=4096),
        # Returns of a long rollout of a few thousand environments that a loss is taken of: forward and backward.
        dict(name="returns_train", kind="returns", timesteps=1000, envs=4096, inner=1, grad=True, gamma=0.99, ends=0.01),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_rows(rng):
    form = rng.randrange(4)
    d = _log_uniform(rng, 3, 400)
    if form == 0:
        return "f4:%d;i4:1;f4:1;f4:%d;b1:1" % (d, d)
    if form == 1:
        return "f4:%d;f4:%d;f4:1;f4:%d;b1:1" % (d, rng.randint(1, 24), d)
    if form == 2:
        return "u1:%d,%d,%d;i8:1;i4:1;f4:1;b1:1" % (rng.randint(7, 96), rng.randint(7, 96), rng.randint(1, 4))
    return "u1:%d;b1:%d;f2:%d;i8:1;f4:1" % (_log_uniform(rng, 20, 2000), rng.randint(2, 40), d)


def _frames(rows):
    """Whether rows are images of whole 16-byte pieces followed by the slot number of the next one (`following`)."""
    fields = _fields(rows)
    return fields[0][0] == "u1" and fields[1][0] == "i8" and int(np.prod(fields[0][1])) % 16 == 0


#: Most bytes of rows a drawn case keeps, and most it moves out of the buffer in a pass.
_KEPT, _MOVED = 3 << 30, 100 << 20


def draw(rng):
    kind = rng.choice(["per_step"] * 4 + ["per_sample"] * 2 + ["uniform"] * 2 + ["reservoir", "returns"])
    if kind == "returns":
        timesteps = _log_uniform(rng, 20, 2000)
        inner = rng.choice([1, 1, 1, 3])
        envs = _log_uniform(rng, 4, max(8, min(30_000, 16_000_000 // (timesteps * inner))))
        return dict(kind=kind, timesteps=timesteps, envs=envs, inner=inner, grad=rng.random() < 0.5,
                    gamma=rng.choice([0.9, 0.99, 0.997]), ends=rng.choice([0.0, 0.005, 0.05]))
    rows = _draw_rows(rng)
    size = _row_bytes(rows)
    capacity = _log_uniform(rng, 3000, max(4000, min(4_000_000, _KEPT // size)))
    batch = _log_uniform(rng, 16, max(32, min(16_384, capacity // 2, _MOVED // size)))
    if kind == "per_sample":
        nbatch = rng.choice([1, 1, 2, 5])
        if nbatch * batch * size > _MOVED:
            nbatch = 1
        return dict(kind=kind, capacity=capacity, rows=rows, batch=batch, nbatch=nbatch,
                    priorities=rng.choice(["normal", "lognormal", "mixture"]),
                    following=nbatch == 1 and _frames(rows) and rng.random() < 0.5)
    if kind == "reservoir":
        return dict(kind=kind, capacity=capacity, rows=rows, batch=batch, insert=_log_uniform(rng, 1, min(5000, capacity)))
    host = rng.random() < 0.25
    if kind == "uniform":
        insert = _log_uniform(rng, 1, 16 if host else min(5000, capacity))
        return dict(kind=kind, capacity=capacity, rows=rows, batch=batch, insert=insert, host_rows=host,
                    fill=rng.choice([1.0, 0.55]))
    calls = rng.choice([3, 3, 2, 1])
    insert = rng.choice([1, 1, _log_uniform(rng, 2, 16 if host else 2000)])
    return dict(kind=kind, calls=calls, capacity=capacity, rows=rows, batch=batch, update=rng.choice([0, 0, 2 * batch]),
                insert=min(insert, capacity // 4), with_priorities=rng.random() < 0.3, host_rows=host,
                priorities=rng.choice(["normal", "lognormal", "mixture"]), fill=rng.choice([1.0, 0.7]),
                following=calls > 1 and _frames(rows) and rng.random() < 0.5)


# ------------------------------------------------------------------- rows and priorities
def _fields(rows):
    out = []
    for entry in rows.split(";"):
        t, shape = entry.split(":")
        out.append((t, tuple(int(v) for v in shape.split(","))))
    return out


def _row_bytes(rows):
    return sum(int(np.prod(s)) * torch.empty((), dtype=_TYPES[t]).element_size() for t, s in _fields(rows))


def _make_rows(rows, n, first, filled, gen):
    """n rows on the device: pixels and masks, normal floats, and slot numbers of the following row among the filled
    ones (i8)."""
    out = []
    for t, shape in _fields(rows):
        shape = (n,) + shape
        if t == "u1":
            out.append(torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=gen))
        elif t == "b1":
            out.append(torch.rand(shape, device="cuda", generator=gen) < 0.05)
        elif t == "i8":
            out.append(((torch.arange(first, first + n, device="cuda") + 1) % filled).reshape(shape))
        elif t == "i4":
            out.append(torch.randint(0, 18, shape, dtype=torch.int32, device="cuda", generator=gen))
        else:
            out.append(torch.randn(shape, device="cuda", generator=gen).to(_TYPES[t]))
    return out


def _make_priorities(form, n, gen):
    if form == "lognormal":
        return torch.randn(n, device="cuda", generator=gen).exp()
    if form == "mixture":  # nearly all tiny, one in a hundred large
        u = torch.rand(n, device="cuda", generator=gen)
        return torch.where(torch.rand(n, device="cuda", generator=gen) < 0.01, 1.0 + 99.0 * u, 1e-6 + 1e-3 * u)
    return torch.randn(n, device="cuda", generator=gen).abs() + 1e-6


def _fill(put, rows, n, gen):
    chunk = max(1, (256 << 20) // _row_bytes(rows))
    for first in range(0, n, chunk):
        put(_make_rows(rows, min(chunk, n - first), first, n, gen))


def _new_rows(case, gen):
    """What the actors hand over: device tensors, or host arrays where the environment runs on the host."""
    rows = _make_rows(case["rows"], case["insert"], 0, case["insert"], gen)
    return [r.cpu().numpy() for r in rows] if case.get("host_rows") else rows


# ------------------------------------------------------------------- the cases' four functions
def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "returns":
        shape = (case["timesteps"], case["envs"]) + ((case["inner"],) if case["inner"] > 1 else ())
        reward = torch.randn(shape, device="cuda", generator=gen)
        done = torch.rand(shape[:2], device="cuda", generator=gen) < case["ends"]
        value = torch.randn(shape[1:], device="cuda", generator=gen)
        state = dict(case=case, returns=DiscountedReturn(case["gamma"], need_bprop=case["grad"]), done=done,
                     reward=reward.requires_grad_(case["grad"]), value=value.requires_grad_(case["grad"]))
        if case["grad"]:
            state["loss_grad"] = torch.randn(shape, device="cuda", generator=gen)
        return state
    capacity, batch, rows = case["capacity"], case["batch"], case["rows"]
    shapes, types = [s for _, s in _fields(rows)], [_TYPES[t] for t, _ in _fields(rows)]
    state = dict(case=case)
    if kind == "uniform":
        buf = UniformReplayBuffer(batch, capacity, shapes, types, seed=seed)
        _fill(buf.insert, rows, int(case["fill"] * capacity), gen)
    elif kind == "reservoir":
        buf = ReservoirReplayBuffer(capacity, batch, shapes, types, seed0=seed + 1)
        _fill(buf.push, rows, capacity + capacity // 3, gen)
    else:
        buf = PriorityReplayBuffer(0.6, capacity, batch, shapes, types, seed0=seed + 1)
        n = int(case.get("fill", 1.0) * capacity)
        _fill(buf.insert, rows, n, gen)
        buf.update_priorities(torch.arange(n, device="cuda"), _make_priorities(case["priorities"], n, gen))
    state["buf"] = buf
    if "insert" in case:
        state["rows"] = _new_rows(case, gen)
        state["rings"] = buf.buffer if kind == "uniform" else buf.storage()
    if kind == "per_step":
        if case["update"]:  # slots of rows used some time ago, one in ten of them named twice
            idx = torch.randint(0, n, (case["update"],), device="cuda", generator=gen)
            idx[::10] = idx[1::10][: idx[::10].numel()] if case["update"] > 10 else idx[::10]
            state["used"] = idx
            state["priorities"] = torch.rand(case["update"], device="cuda", generator=gen).clamp_min(1e-6).pow(-1.0 / 1.5)
        else:
            state["used"] = buf.sample(0.4)[0]
            state["priorities"] = torch.randn(batch, device="cuda", generator=gen).abs() + 1e-6
        state["row_priorities"] = _make_priorities("normal", case["insert"], gen) if case["with_priorities"] else None
    return state


def _sample(buf, case):
    if case.get("following"):
        return buf.sample_with_next(0.4, slot_field=1, row_field=0)
    return buf.sample(0.4)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "returns":
        out = state["returns"](state["reward"], state["done"], state["value"])
        if not case["grad"]:
            return out
        grads = torch.autograd.grad(out, (state["reward"], state["value"]), state["loss_grad"])
        return (out.detach(),) + grads
    buf = state["buf"]
    if kind == "per_sample":
        if case["nbatch"] > 1:
            return buf.sample_many(case["nbatch"], 0.4)
        return _sample(buf, case)
    if kind == "uniform":
        buf.insert(state["rows"])
        return buf.sample() + tuple(state["rings"])
    if kind == "reservoir":
        buf.push(*state["rows"])
        return buf.sample() + tuple(state["rings"])
    rows, row_priorities = state["rows"], state["row_priorities"]
    if case["calls"] == 1:
        out = buf.update_priorities_insert_and_sample(state["used"], state["priorities"], *rows, beta=0.4,
                                                      insert_priorities=row_priorities)
    else:
        if case["calls"] == 2:
            buf.update_priorities_and_insert(state["used"], state["priorities"], *rows, insert_priorities=row_priorities)
        else:
            buf.update_priorities(state["used"], state["priorities"])
            buf.insert(*rows, priorities=row_priorities)
        out = _sample(buf, case)
    if not case["update"]:
        state["used"] = out[0]  # the next step's priorities are those of this batch
    return out + tuple(state["rings"])


def _tree_nodes(entries, capacity):
    """Nodes above and among the leaves that `entries` writes to distinct leaves change."""
    depth = max(0, (capacity - 1).bit_length())
    return sum(min(entries, 1 << level) for level in range(depth + 1))


def work(case):
    kind = case["kind"]
    if kind == "returns":
        n = case["timesteps"] * case["envs"]
        elements = n * case["inner"]
        forward = 8 * elements + n + 4 * case["envs"] * case["inner"]
        return {"bytes": (2 if case["grad"] else 1) * forward, "flops": (4 if case["grad"] else 2) * elements}
    size = _row_bytes(case["rows"])
    total = 2 * size * case["batch"] * case.get("nbatch", 1)  # the sampled rows, read and written
    flops = 0
    if case.get("following"):
        total += 2 * int(np.prod(_fields(case["rows"])[0][1])) * case["batch"]
    if kind in ("per_step", "per_sample"):
        strata = case["batch"] * case.get("nbatch", 1)
        total += strata * 12 + 4 * _tree_nodes(strata, case["capacity"])  # index and weight; the nodes the descents compare with
        flops += strata * 100
    if "insert" in case:
        total += 2 * size * case["insert"]
    if kind == "per_step":
        update = case["update"] or case["batch"]
        total += 12 * update + 4 * case["insert"] * case["with_priorities"]
        # sum and minimum of every node on the way up: the sibling read, the node written
        total += 16 * (_tree_nodes(update, case["capacity"]) + _tree_nodes(case["insert"], case["capacity"]))
        flops += 60 * update
    return {"bytes": total, "flops": flops}


def tolerance(case):
    if case["kind"] == "returns":
        # float32 sums of up to 2000 discounted terms: against the same recurrence in float64 results and gradients
        # differ by up to 3.0e-7 (2-norm), the worst element by 2.7e-6 of the root mean square
        return {"rel": 1.2e-6, "max": 1.1e-5}
    if case["kind"] in ("per_step", "per_sample"):
        # rows and slots are copies; the importance weights are float32 quotients and powers: against float64 they
        # differ by up to 7.8e-8 (2-norm), the worst one by 1.7e-7
        return {"rel": 3e-7, "max": 7e-7, "differ": 0.0}
    return "exact"
