"""The discounted return and its gradient at the sizes where the tiled kernel's groups and chunks end, and on both sides
of every line of the dispatch, bit for bit against the oracle's recurrence."""
import numpy as np
import pytest
import torch

from gpu_util import t2n

pytestmark = pytest.mark.gpu


# groups of 16 / 32 / 64 columns and chunks of 64 steps (one short, exact, one over), fewer columns than a quad or a
# group, several values per environment, the per-column kernel (many columns, or a short time axis)
SHAPES = [(1, 1, 1), (2, 3, 1), (64, 4, 1), (65, 5, 1), (63, 15, 1), (128, 16, 1), (129, 17, 1), (256, 31, 1), (257, 7, 3),
          (320, 4096, 1), (70, 4097, 1), (191, 8191, 1), (130, 1400, 3), (128, 8193, 1), (127, 8195, 1), (33, 8200, 1),
          (32, 8200, 1), (129, 16385, 1), (128, 16385, 1), (3, 40961, 1), (1000, 33, 1)]


def oracle_gradient(orc, grad, done, gamma):
    """A_t = grad_t + c_{t-1} A_{t-1}: the oracle's backward recurrence on time-reversed inputs, flags moved by one."""
    flags = np.concatenate([done[:-1][::-1], np.zeros_like(done[:1])])
    a = orc.discounted_return(np.ascontiguousarray(grad[::-1]), np.ascontiguousarray(flags), np.zeros_like(grad[0]), gamma)
    keep = ((np.float32(1) - done[-1].astype(np.float32)) * np.float32(gamma))[:, None]
    return a[::-1], keep * a[0]


@pytest.mark.parametrize("shape", SHAPES)
def test_return_and_gradient_bit_exact(shape):
    from mindrl_amd.utils import DiscountedReturn
    from oracle import orc
    t, b, inner = shape
    rng = np.random.default_rng(t * 31 + b)
    r = rng.normal(size=shape).astype(np.float32)
    d = rng.random((t, b)) < 0.05
    v = rng.normal(size=(b, inner)).astype(np.float32)
    w = rng.normal(size=shape).astype(np.float32)
    reward = torch.from_numpy(r).cuda().requires_grad_(True)
    value = torch.from_numpy(v).cuda().requires_grad_(True)
    out = DiscountedReturn(0.97, need_bprop=True)(reward, torch.from_numpy(d).cuda(), value)
    assert np.array_equal(t2n(out.detach()), orc.discounted_return(r, d, v, 0.97))
    grad_reward, grad_value = torch.autograd.grad(out, (reward, value), torch.from_numpy(w).cuda())
    want_reward, want_value = oracle_gradient(orc, w, d, 0.97)
    assert np.array_equal(t2n(grad_reward), want_reward)
    assert np.array_equal(t2n(grad_value), want_value)


# the pipeline's first, second and third chunk and the stages behind its loop of three, each with a last chunk of one step, of
# half and whole, at either side of sixteen and eight steps; the lines between the kernels and the groups' widths
EDGES = [(t, b, inner) for b, inner in ((5, 1), (3, 2), (4101, 1)) for t in (1, 16, 17, 32, 33, 48, 64, 96, 97, 128, 129, 192, 193, 256, 257, 320, 321, 385)]
EDGES += [(33, 32768, 1), (33, 32769, 1), (64, 32769, 1), (65, 32769, 1), (65, 40961, 1), (127, 8193, 1), (128, 4097, 1), (127, 4097, 1),
          (255, 40961, 1), (256, 40961, 1), (257, 65537, 1), (130, 2731, 3), (100, 5461, 3), (33, 10900, 1), (33, 10901, 1), (48, 24400, 1),
          (48, 24401, 1), (63, 37900, 1), (63, 37901, 1), (64, 31000, 1), (64, 31001, 1), (65, 24900, 1), (65, 24901, 1), (95, 40960, 1),
          (95, 40961, 1), (40, 5733, 3), (40, 5734, 3)]


@pytest.mark.parametrize("shape", EDGES)
def test_every_stage_of_the_pipeline(shape):
    """Results and both gradients bit for bit, with infinities and numbers that are none among the inputs: they reach every earlier
    (of the gradient: later) step of their column up to the next end, and no other column."""
    from mindrl_amd.utils import DiscountedReturn
    from oracle import orc
    t, b, inner = shape
    rng = np.random.default_rng(t * 7 + b + inner)
    r, w = rng.normal(size=shape).astype(np.float32), rng.normal(size=shape).astype(np.float32)
    for x in (r, w):
        x[rng.integers(0, t), rng.integers(0, b)] = np.inf
        x[rng.integers(0, t), rng.integers(0, b)] = np.nan
    d = rng.random((t, b)) < 0.03
    v = rng.normal(size=(b, inner)).astype(np.float32)
    reward, value = torch.from_numpy(r).cuda().requires_grad_(True), torch.from_numpy(v).cuda().requires_grad_(True)
    out = DiscountedReturn(0.99, need_bprop=True)(reward, torch.from_numpy(d).cuda(), value)
    got = (out.detach(),) + torch.autograd.grad(out, (reward, value), torch.from_numpy(w).cuda())
    for g, want in zip(got, (orc.discounted_return(r, d, v, 0.99),) + oracle_gradient(orc, w, d, 0.99)):
        assert np.array_equal(t2n(g), want, equal_nan=True)


def test_forward_mode_is_refused():
    import torch.autograd.forward_ad as fw
    from mindrl_amd.utils import DiscountedReturn
    done, value = torch.zeros(5, 3, dtype=torch.bool, device="cuda"), torch.zeros(3, device="cuda")
    with fw.dual_level():
        reward = fw.make_dual(torch.ones(5, 3, device="cuda", requires_grad=True), torch.ones(5, 3, device="cuda"))
        with pytest.raises(NotImplementedError):
            DiscountedReturn(0.9, need_bprop=True)(reward, done, value)


def test_saved_flags_pass_through_hooks():
    """A hook may hand the flags back in another layout; a gradient may come as an expanded or negated view."""
    from mindrl_amd.utils import DiscountedReturn
    reward = torch.randn(70, 9, device="cuda", requires_grad=True)
    value = torch.randn(9, device="cuda", requires_grad=True)
    done = torch.rand(70, 9, device="cuda") < 0.1
    returns = DiscountedReturn(0.9, need_bprop=True)
    want = torch.autograd.grad(returns(reward, done, value), (reward, value), torch.full((70, 9), 2.0, device="cuda"))
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.cuda().t().contiguous().t()):
        out = returns(reward, done, value)
    got = torch.autograd.grad(out, (reward, value), torch.full((), 2.0, device="cuda").expand(70, 9))
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    negated = torch._neg_view(torch.full((70, 9), -2.0, device="cuda"))
    got = torch.autograd.grad(returns(reward, done, value), (reward, value), negated)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("need_bprop", [False, True])
def test_empty_inputs_are_refused(need_bprop):
    from mindrl_amd.utils import DiscountedReturn
    returns = DiscountedReturn(0.9, need_bprop=need_bprop)
    for reward, done, value in (((5, 3, 0), (5, 3), (3, 0)), ((5, 0), (5, 0), (0,)), ((0, 3), (0, 3), (3,)), ((0,), (0,), ())):
        with pytest.raises(ValueError):
            returns(torch.zeros(reward, device="cuda"), torch.zeros(done, dtype=torch.bool, device="cuda"),
                    torch.zeros(value, device="cuda"))


def test_computes_on_the_device_of_its_own():
    """Inputs on another device are moved to the one the object was made on: the native call takes none of them as they are."""
    from mindrl_amd import _lib
    reward, done = torch.ones(5, 3, device="cuda"), torch.zeros(5, 3, dtype=torch.bool, device="cuda")
    value = torch.zeros(3, device="cuda")
    call = _lib.native().discounted_return
    assert call(reward, done, value, 0.9, False, _lib.check, reward.device.index) is not None
    assert call(reward, done, value, 0.9, False, _lib.check, reward.device.index + 1) is None
