"""DiscountedReturn with the interface of mindspore_rl/utils/discounted_return.py:25-92."""
import torch

from .. import _lib
from ..core._rows import device
from ..dtype import as_torch_dtype


class DiscountedReturn:
    r"""Discounted return :math:`G_t = R_t + \gamma (1 - done_t) G_{t+1}` over sequences that may
    hold several episodes, `done` marking the episode ends and `last_state_value` the value after
    the final step (mindspore_rl/utils/discounted_return.py:25-59).

    Args:
        gamma (float): discount factor in [0, 1].
        need_bprop (bool): the reference then avoids its fused operator so that autograd can
            differentiate the loop (discounted_return.py:81-92); here the returned tensor is then
            differentiable with respect to reward and last_state_value (the backward pass is the
            same recurrence forwards in time, one launch).
        dtype: output type; float32 only.

    Inputs: reward [Timestep, Batch, ...] float32, done [Timestep, Batch] bool,
    last_state_value [Batch, ...] float32 (the Batch axis may be omitted everywhere,
    as in tests/st/test_discounted_return.py:47-53). Returns a tensor shaped like reward.
    """

    def __init__(self, gamma, need_bprop=False, dtype=torch.float32):
        if gamma > 1.0 or gamma < 0.0:
            raise ValueError(f"The discounted factor should be a number in range [0, 1], but got {gamma}.")
        if as_torch_dtype(dtype) != torch.float32:
            raise TypeError("DiscountedReturn computes in float32")
        self.gamma = float(gamma)
        self.need_bprop = bool(need_bprop)
        self._dev = device()
        self._native = _lib.native().discounted_return

    def construct(self, reward, done, last_state_value):
        out = self._native(reward, done, last_state_value, self.gamma, self.need_bprop, _lib.check, self._dev.index)
        if out is None:
            r = torch.as_tensor(reward).to(device=self._dev, dtype=torch.float32).contiguous()
            d = torch.as_tensor(done).to(device=self._dev, dtype=torch.bool).contiguous()
            v = torch.as_tensor(last_state_value).to(device=self._dev, dtype=torch.float32).contiguous()
            if r.dim() == 0 or r.shape[0] != d.shape[0]:
                raise ValueError("reward and done must share the leading Timestep axis")
            timesteps = r.shape[0]
            batch = d.numel() // timesteps if timesteps else 0
            if batch == 0 or r.numel() == 0 or d.numel() != timesteps * batch or r.numel() % (timesteps * batch):
                raise ValueError("done must be [Timestep, Batch] and reward [Timestep, Batch, ...]")
            if v.numel() != batch * (r.numel() // (timesteps * batch)):
                raise ValueError("last_state_value must be [Batch, ...] matching reward")
            reward, done, last_state_value = r, d, v
            out = self._native(r, d, v, self.gamma, self.need_bprop, _lib.check, self._dev.index)
            if out is None:
                raise ValueError("reward, done and last_state_value must be dense tensors")
        if not out.requires_grad:  # (a result with a history holds what its gradient needs: no more is kept alive)
            self._keep = (reward, done, last_state_value)
        return out

    __call__ = construct
