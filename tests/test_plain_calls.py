"""Which calls skip the dispatcher: ordinary eager ones only.  Under a dispatch mode, a profiler,
compilation, a functorch transform, a forward-mode level or a backward that is itself recorded, and
on tensors whose memory does not hold their values, the operators go through their custom ops, and
both ways give the same results."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from metal_kernelops import _native as nat

DEV = "cuda"


class Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.ops = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.ops.append(str(func))
        return func(*args, **(kwargs or {}))


def test_plain_call_rules():
    t = torch.ones(3)
    leaf = torch.ones(3, requires_grad=True)
    assert nat.plain_call(t, None, torch.nn.Parameter(t, requires_grad=False))
    assert not nat.plain_call(t, leaf)
    with torch.no_grad():
        assert nat.plain_call(t, leaf)
        with Seen():
            assert not nat.plain_call(t)
        with torch.device("cpu"):  # a function mode
            assert not nat.plain_call(t)
        with torch.autograd.forward_ad.dual_level():
            assert not nat.plain_call(t)
        seen = []
        torch.func.vmap(lambda v: (seen.append(nat.plain_call(v, t)), v)[1])(torch.ones(2, 3))
        assert seen == [False]
        seen = []
        torch.jit.trace(lambda v: (seen.append(nat.plain_call(v)), v + 1)[1], (t,), check_trace=False)
        assert seen[0] is False

        class Sub(torch.Tensor):
            pass

        assert not nat.plain_call(t, t.as_subclass(Sub))


def test_tensors_not_read_from_memory_are_not_plain():
    # The dispatcher materialises these before a kernel sees them; their memory holds the negated
    # values, or nothing.
    t = torch.ones(3)
    odd = {"negated": torch._neg_view(t), "zero": torch._efficientzerotensor((3,)),
           "functional": torch._to_functional_tensor(t), "meta": t.to("meta")}
    assert odd["negated"].contiguous().is_neg()  # a dense layout alone does not materialise it
    with torch.no_grad():
        for name, v in odd.items():
            assert not nat.plain_call(t, v), name


def test_a_recording_profiler_sees_the_op():
    t = torch.ones(3)
    with torch.no_grad():
        assert nat.plain_call(t)
        with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]):
            assert not nat.plain_call(t)
        assert nat.plain_call(t)


def _calls():
    from metal_kernelops import selective_scan
    from metal_kernelops.cv import causal_conv1d_fn, mamba2_chunk_scan
    g = torch.Generator().manual_seed(1)

    def r(*shape):
        return torch.randn(shape, generator=g).to(DEV)

    return {
        "selscan": (selective_scan, [r(1, 8, 20), r(1, 8, 20).abs(), -r(8, 4).abs(), r(1, 1, 4, 20), r(1, 1, 4, 20)]),
        "ssd": (lambda *a: mamba2_chunk_scan(*a)[0],
                [r(1, 20, 2, 8), r(1, 20, 2).abs(), -r(2).abs(), r(1, 20, 1, 8), r(1, 20, 1, 8)]),
        "conv1d": (causal_conv1d_fn, [r(1, 8, 20), r(8, 4), r(8)]),
    }


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["selscan", "ssd", "conv1d"])
def test_modes_still_see_the_op(name):
    fn, args = _calls()[name]
    with torch.no_grad():
        plain = fn(*args)
        with Seen() as mode:
            seen = fn(*args)
    assert any(f"mko.{name}_fwd" in op for op in mode.ops), mode.ops
    assert torch.equal(plain, seen)
    leaves = [t.clone().requires_grad_(True) for t in args]
    dy = torch.ones_like(plain)
    plain_grads = torch.autograd.grad(fn(*leaves), leaves, dy)
    with torch.autograd.set_multithreading_enabled(False), Seen() as mode:
        seen_grads = torch.autograd.grad(fn(*leaves), leaves, dy)
    assert any(f"mko.{name}_bwd" in op for op in mode.ops), mode.ops
    assert all(torch.equal(a, b) for a, b in zip(plain_grads, seen_grads))
    # a recorded backward keeps going through the op, which refuses to be differentiated
    grads = torch.autograd.grad(fn(*leaves), leaves, dy, create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(grads[0].sum(), leaves[:1])


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["selscan", "ssd", "conv1d"])
def test_negated_views_and_zero_tensors_are_materialised(name):
    fn, args = _calls()[name]
    plain = [-args[0]] + args[1:]
    zeros = [torch.zeros_like(args[0])] + args[1:]
    with torch.no_grad():
        assert torch.equal(fn(torch._neg_view(args[0]), *args[1:]), fn(*plain))
        assert torch.equal(fn(torch._efficientzerotensor(tuple(args[0].shape), device=DEV), *args[1:]), fn(*zeros))
    leaves = [t.clone().requires_grad_(True) for t in args]
    dy = torch.randn_like(fn(*args))
    got = torch.autograd.grad(fn(*leaves), leaves, torch._neg_view(dy))
    want = torch.autograd.grad(fn(*leaves), leaves, -dy)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["selscan", "ssd", "conv1d"])
def test_profiler_names_the_op(name):
    fn, args = _calls()[name]
    leaves = [t.clone().requires_grad_(True) for t in args]
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        with torch.no_grad():
            out = fn(*args)
        torch.autograd.grad(fn(*leaves), leaves, torch.ones_like(out))
    seen = [e.key for e in prof.key_averages()]
    assert f"mko::{name}_fwd" in seen and f"mko::{name}_bwd" in seen, seen
