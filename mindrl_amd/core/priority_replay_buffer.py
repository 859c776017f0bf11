"""PriorityReplayBuffer with the interface of
mindspore_rl/core/priority_replay_buffer.py:30-138, backed by libmrb.so."""
import ctypes as C
import os

import numpy as np
import torch

from .. import _lib
from ._rows import (FieldLayout, create_with_layout, device, flat_on_device, get_counters, load_fields, pointers,
                    save_fields, set_counters, storage_views, stream_ptr)


class PriorityReplayBuffer:
    """Proportional prioritized replay (Schaul et al.) resident in HBM: FIFO rows
    plus a sum tree and a min tree over next_pow2(capacity) leaves.

    Same constructor and methods as the reference class
    (mindspore_rl/core/priority_replay_buffer.py:60-138).

    Args:
        alpha (float): priority exponent; 0 = uniform, 1 = fully prioritized.
        capacity (int): number of rows kept.
        sample_size (int): rows returned by sample().
        shapes, types: shape / element type of each tensor of an element.
        seed0, seed1 (int): generator seed; seed1 if non-zero, else seed0, else entropy.
        output_ring (int): 0 (the default): sample() returns fresh tensors on every call, as the
            reference does. N > 0 (opt-in, for loops that consume a batch before drawing the N-th next
            one): sample() hands out its result tensors from N preallocated sets in turn, so a call
            allocates nothing; a returned batch is then overwritten by the N-th sample() call after
            it - clone() what must live longer.
        packed_rows (bool or int): False (default): every field is a [capacity, *shape_i] array of its own, the
            reference's layout. True (or a byte limit): rows of at most 64 (that many) bytes are kept packed in
            one array, so that a sampled row's fields share cache lines; storage() then returns strided views.
            Results never differ.
    """

    def __init__(self, alpha, capacity, sample_size, shapes, types, seed0=0, seed1=0, output_ring=0, packed_rows=False):
        self._dev = device()
        self._layout = FieldLayout(shapes, types)
        self._capacity = int(capacity)
        self._sample_size = int(sample_size)
        self._alpha = float(alpha)
        seed = int(seed1) or int(seed0) or int.from_bytes(os.urandom(8), "little")
        h = C.c_int64(0)
        create_with_layout(packed_rows, lambda: _lib.check(_lib.lib().mrb_per_create(
            self._capacity, self._alpha, len(self._layout), self._layout.c_bytes, seed & (2**64 - 1), C.byref(h))))
        self._h = h.value
        self._native = self._layout.native(self._h, self._dev)
        self._handle = torch.tensor([self._h], dtype=torch.int64)
        self._keep = None
        self._ring_size = int(output_ring)
        self._ring, self._ring_at = None, 0  # output sets, built by the first sample()

    def _next_outputs(self):
        """The next preallocated (indices, weights, fields) set."""
        if self._ring is None:
            n = self._sample_size
            self._ring = [(torch.empty(n, dtype=torch.int64, device=self._dev),
                           torch.empty(n, dtype=torch.float32, device=self._dev), self._layout.empty(n, self._dev))
                          for _ in range(self._ring_size)]
        out = self._ring[self._ring_at]
        self._ring_at = (self._ring_at + 1) % self._ring_size
        return out

    def _outputs(self, out):
        """Where a sample goes that is not to fresh tensors: (indices, weights, [fields]), or None."""
        if out is not None:
            idx, w, fields = out
            return idx, w, self._layout.check_out(fields, self._sample_size, self._dev)
        return self._next_outputs() if self._ring_size > 0 else None

    def _check_given(self, given):
        """Raises if a sample cannot go to `given` (asked when the native call has taken it for something to convert)."""
        for t, dtype in zip(given or (), (torch.int64, torch.float32)):
            if t.dtype != dtype or t.device != self._dev or not t.is_contiguous() or t.numel() < self._sample_size:
                raise ValueError("out must hold contiguous int64 indices, float32 weights and the fields on %s, of sample_size = "
                                 "%d rows" % (self._dev, self._sample_size))

    def _uniforms(self, uniforms, n, what):
        u = flat_on_device(uniforms, torch.float32, self._dev)
        if u.numel() != n:
            raise ValueError("uniforms must hold %s values" % what)
        return u

    def _entries(self, indices, priorities):
        idx = flat_on_device(indices, torch.int64, self._dev)
        pr = flat_on_device(priorities, torch.float32, self._dev)
        if idx.numel() != pr.numel():
            raise ValueError("indices and priorities differ in length")
        return idx, pr

    def _row_priorities(self, priorities, rows, name):
        if priorities is None:
            return None
        pr = flat_on_device(priorities, torch.float32, self._dev)
        if pr.numel() != self._layout.batch_of(rows):
            raise ValueError("%s must hold one value per pushed row" % name)
        return pr

    # -- reference methods ---------------------------------------------------
    def insert(self, *transition, priorities=None):
        """Pushes one transition (tensors of shape_i) or a batch ([n, *shape_i]); the
        oldest row is replaced when full; new rows take the running max priority
        (priority_replay_buffer.py:78-90). `priorities` (f32[n]), if given, are
        applied to the new rows as update_priorities would. Returns the handle
        tensor int64[1]."""
        if len(transition) == 1 and isinstance(transition[0], (list, tuple)):
            transition = tuple(transition[0])
        if self._native.per_push(transition, priorities) is None:
            priorities = self._row_priorities(priorities, transition, "priorities")
            transition = self._layout.put(lambda rows: self._native.per_push(rows, priorities), transition, self._dev)
        self._keep = (transition, priorities)
        return self._handle

    # the reference's own test calls the method by this name (tests/st/test_priority_replay_buffer.py:46)
    push = insert

    def sample(self, beta, uniforms=None, out=None):
        """Stratified proportional sample of `sample_size` rows
        (priority_replay_buffer.py:92-106).

        Returns (indices int64[B], weights f32[B], *transitions [B, *shape_i]).
        `uniforms` (f32[B] in [0,1)) replaces the buffer's generator, stratum k
        using uniforms[k]. `out` = (indices, weights, [fields]) writes into the caller's tensors.
        Without `out` the result is a set of fresh tensors, unless the buffer was built with
        `output_ring` > 0: then it comes from that ring of preallocated output sets and stays valid
        until `output_ring` further sample() calls have been made."""
        n = self._sample_size
        given = self._outputs(out)
        if given is None:
            res = self._native.per_sample(n, beta, uniforms)
            if res is None:
                uniforms = self._uniforms(uniforms, n, "sample_size = %d" % n)
                res = self._native.per_sample(n, beta, uniforms)
        else:
            if uniforms is not None:
                uniforms = self._uniforms(uniforms, n, "sample_size = %d" % n)
            if self._native.per_sample_into(n, beta, uniforms, *given) is None:
                self._check_given(given)
                raise ValueError("out must hold dense tensors")
            res = (given[0], given[1]) + tuple(given[2])
        self._keep = uniforms
        return res

    def sample_with_next(self, beta, slot_field, row_field, uniforms=None):
        """sample(beta) plus, in the same launch, field `row_field` of the row whose slot number each sampled
        row holds in its field `slot_field` (an int64[1] field): for transitions that store the next
        observation as a slot number instead of a copy. Returns sample()'s tuple with one more tensor
        [B, *shape_row_field] at the end - what `gather(transitions[slot_field])[row_field]` would give, without
        the second launch and the second tree descent. Fresh output tensors on every call."""
        n = self._sample_size
        slot_field, row_field = int(slot_field), int(row_field)
        if not 0 <= slot_field < len(self._layout) or not 0 <= row_field < len(self._layout):
            raise ValueError("slot_field and row_field must name fields of the transition")
        res = self._native.per_sample_next(n, beta, uniforms, slot_field, row_field)
        if res is None:
            uniforms = self._uniforms(uniforms, n, "sample_size = %d" % n)
            res = self._native.per_sample_next(n, beta, uniforms, slot_field, row_field)
        self._keep = uniforms
        return res

    def sample_many(self, nbatch, beta, uniforms=None):
        """`nbatch` batches in one launch: what `nbatch` successive sample(beta) calls would return on an
        unchanged buffer, stacked: (indices int64[nbatch, B], weights f32[nbatch, B], *transitions
        [nbatch, B, *shape_i]). For learners that draw several batches between priority updates; one launch
        amortises the launch and the tree descent. `uniforms`: f32[nbatch, B] or None (generator)."""
        nbatch, n = int(nbatch), self._sample_size
        res = self._native.per_sample_many(nbatch, n, beta, uniforms)
        if res is None:
            uniforms = self._uniforms(uniforms, nbatch * n, "nbatch * sample_size = %d" % (nbatch * n))
            res = self._native.per_sample_many(nbatch, n, beta, uniforms)
        self._keep = uniforms
        return res

    def update_priorities(self, indices, priorities):
        """leaf[indices[j]] = priorities[j] ** alpha in order, last write wins
        (priority_replay_buffer.py:108-120). Returns the handle tensor."""
        if self._native.per_update(indices, priorities) is None:
            indices, priorities = self._entries(indices, priorities)
            self._native.per_update(indices, priorities)
        self._keep = (indices, priorities)
        return self._handle

    def update_priorities_and_insert(self, indices, priorities, *transition, insert_priorities=None):
        """update_priorities(indices, priorities) followed by insert(*transition, priorities=insert_priorities),
        as ONE library call (mrb_per_update_push): the result is the two calls', bit for bit, with fewer kernel
        launches - a learner's step is bound by them (the reference's loop issues the two back to back,
        mindspore_rl/algorithm/dqn/dqn_trainer.py:76-87). Returns the handle tensor."""
        if len(transition) == 1 and isinstance(transition[0], (list, tuple)):
            transition = tuple(transition[0])
        if self._native.per_update_push(indices, priorities, transition, insert_priorities) is None:
            indices, priorities = self._entries(indices, priorities)
            ipr = insert_priorities = self._row_priorities(insert_priorities, transition, "insert_priorities")
            transition = self._layout.put(lambda rows: self._native.per_update_push(indices, priorities, rows, ipr),
                                          transition, self._dev)
        self._keep = (indices, priorities, transition, insert_priorities)
        return self._handle

    def update_priorities_insert_and_sample(self, indices, priorities, *transition, beta, insert_priorities=None,
                                            uniforms=None, out=None):
        """update_priorities(indices, priorities), insert(*transition, priorities=insert_priorities) and
        sample(beta, uniforms, out) as ONE library call (mrb_per_update_push_sample): a learner's whole step on the
        buffer (mindspore_rl/algorithm/dqn/dqn_trainer.py:76-87 and the sample of the next iteration). The results
        are the three calls', bit for bit; on a small buffer (capacity up to 16,384, up to 384 entries, one
        transition, up to 512 sampled rows) they take one kernel launch instead of two or three. Returns what
        sample() returns."""
        if len(transition) == 1 and isinstance(transition[0], (list, tuple)):
            transition = tuple(transition[0])
        b = self._sample_size
        given = self._outputs(out)
        res = self._native.per_step(indices, priorities, transition, insert_priorities, b, beta, uniforms, given)
        if res is None:
            self._check_given(given)
            indices, priorities = self._entries(indices, priorities)
            ipr = insert_priorities = self._row_priorities(insert_priorities, transition, "insert_priorities")
            if uniforms is not None:
                uniforms = self._uniforms(uniforms, b, "sample_size = %d" % b)
            results = []

            def step(rows):
                r = self._native.per_step(indices, priorities, rows, ipr, b, beta, uniforms, given)
                results.append(r)
                return r

            transition = self._layout.put(step, transition, self._dev)
            res = results[-1]
        self._keep = (indices, priorities, transition, insert_priorities, uniforms)
        return res if given is None else (given[0], given[1]) + tuple(given[2])

    def gather(self, indices, out=None):
        """Rows at the given slots (int64, each in [0, size)): one [n, *shape_i] tensor per field.
        For transitions that store the slot of their successor instead of a copy of it, e.g.
        `next_rows = buf.gather(sampled_next_idx)`."""
        if out is None:
            res = self._native.per_gather(indices)
            if res is None:
                indices = flat_on_device(indices, torch.int64, self._dev)
                res = self._native.per_gather(indices)
            self._keep = indices
            return res
        idx = flat_on_device(indices, torch.int64, self._dev)
        n = idx.numel()
        dst = self._layout.check_out(out, n, self._dev)
        _lib.check(_lib.lib().mrb_per_gather(self._h, idx.data_ptr(), n, pointers(dst), stream_ptr()))
        self._keep = idx
        return tuple(dst)

    def full(self):
        """Always False, as in the reference (priority_replay_buffer.py:122-124)."""
        return torch.tensor(False)

    def reset(self):
        """Not supported, as in the reference (priority_replay_buffer.py:126-128)."""
        raise ValueError("reset() is not supported by PriorityReplayBuffer.")

    def destroy(self):
        """Releases the native buffer (priority_replay_buffer.py:130-138)."""
        if self._h:
            h, self._h = self._h, 0
            self._ring = None
            _lib.check(_lib.lib().mrb_per_destroy(h))
        return self._handle

    # -- extras ----------------------------------------------------------------
    def size(self):
        return self._state()[0]

    @property
    def max_priority(self):
        return self._state(True)[2]

    @property
    def capacity(self):
        return self._capacity

    @property
    def sample_size(self):
        return self._sample_size

    def _state(self, with_max=False):
        s, hd, mp = C.c_int64(0), C.c_int64(0), C.c_float(0)
        _lib.check(_lib.lib().mrb_per_state(self._h, C.byref(s), C.byref(hd), C.byref(mp) if with_max else None,
                                            stream_ptr()))
        return s.value, hd.value, mp.value

    def export_tree(self):
        """(sum_heap, min_heap) as numpy float32[2 * leaves], root at 1, leaf i at leaves + i."""
        leaves = C.c_int64(0)
        _lib.check(_lib.lib().mrb_per_export_tree(self._h, None, None, C.byref(leaves), stream_ptr()))
        s = np.empty(2 * leaves.value, np.float32)
        m = np.empty(2 * leaves.value, np.float32)
        _lib.check(_lib.lib().mrb_per_export_tree(self._h, s.ctypes.data, m.ctypes.data, None, stream_ptr()))
        return s, m

    def storage(self):
        """Views of the row storage, one [capacity, *shape_i] tensor per field."""
        return storage_views(self._h, self._layout, self._capacity, self, self._dev)

    def state_dict(self):
        """Everything needed to rebuild this buffer: rows, the leaves of the sum tree (internal nodes
        are rebuilt on load, which reproduces them bit for bit), size, pushes, running max priority and
        the generator's position. (The reference never persists its buffers; this is this library's
        own format.)"""
        size, pushes, seed, calls = get_counters(_lib.lib().mrb_per_get_counters, self._h)
        sum_heap, _ = self.export_tree()
        leaves = sum_heap.size // 2
        return {"kind": "priority", "capacity": self._capacity, "alpha": self._alpha, "size": size, "pushes": pushes,
                "seed": seed & ((1 << 64) - 1), "calls": calls, "max_priority": float(self.max_priority),
                "leaves": torch.from_numpy(sum_heap[leaves:leaves + size].copy()),
                "fields": save_fields(self.storage(), size)}

    def load_state_dict(self, state):
        """Restores a state_dict() taken from a buffer of the same capacity, alpha, shapes and types.
        Nothing of this buffer changes unless the whole state fits."""
        if state.get("kind") != "priority" or state["capacity"] != self._capacity:
            raise ValueError("state does not belong to a PriorityReplayBuffer of capacity %d" % self._capacity)
        if np.float32(state["alpha"]) != np.float32(self._alpha):
            # the saved leaves are priorities ** alpha: they mean something else under another exponent
            raise ValueError("state was saved with alpha %r, this buffer has alpha %r" % (state["alpha"], self._alpha))
        leaves = torch.as_tensor(state["leaves"]).to(device=self._dev, dtype=torch.float32).contiguous()
        size, pushes = int(state["size"]), int(state["pushes"])
        if leaves.numel() != size or size != min(pushes, self._capacity) or pushes < 0:
            raise ValueError("state holds %d leaves for size %d after %d pushes" % (leaves.numel(), size, pushes))
        load_fields(self.storage(), state["fields"], self._layout)
        # the tree first, the counters last: a failure on the way leaves size and pushes as they were
        _lib.check(_lib.lib().mrb_per_load_leaves(self._h, leaves.data_ptr() if leaves.numel() else None,
                                                  leaves.numel(), float(state["max_priority"]), stream_ptr()))
        set_counters(_lib.lib().mrb_per_set_counters, self._h, [size, pushes, state["seed"], state["calls"]])
        torch.cuda.current_stream().synchronize()

    def check(self):
        """Synchronises; raises if a kernel recorded a data error since the last check."""
        flags = C.c_uint32(0)
        _lib.check(_lib.lib().mrb_per_check(self._h, C.byref(flags), stream_ptr()))
        f = flags.value
        if f & _lib.DERR_INDEX:
            raise IndexError("update_priorities: index outside [0, capacity)")
        if f & _lib.DERR_PRIORITY:
            raise ValueError("update_priorities: negative or non-finite priority")
        if f & _lib.DERR_TOTAL:
            raise ValueError("sample: total priority is not positive and finite")
        if f & _lib.DERR_OVERLAP:
            raise RuntimeError("calls that change the buffer ran side by side (on several streams, not ordered)")
        return f

    def set_option(self, name, value):
        """Sets a launch option of this buffer ("row_split"; prioritized buffers also "sample_path", "row_wave",
        "lds_levels", "fused_rebuild", "device_counters"). Options change how kernels are launched, never a
        result."""
        _lib.set_option(self._h, name, value)

    def __del__(self):
        # the native buffer (rows, trees) is released with the Python object if destroy() was not called
        try:
            if getattr(self, "_h", 0):
                self.destroy()
        except Exception:  # interpreter shutdown: the library or torch may already be gone
            pass

    def __repr__(self):
        return "PriorityReplayBuffer<>"
