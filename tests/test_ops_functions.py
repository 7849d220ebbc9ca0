"""The stand-alone operators' autograd functions: subclasses of
torch.autograd.Function with forward and backward, as the reference's
(ops.py:32-265); a subclass runs its own, and torch.jit.trace records a call."""
import pytest
import torch

import mhc_ascend_amd as mhc
from mhc_ascend_amd import ops

FUNCTIONS = [ops.SinkhornKnoppFunction, ops.RMSNormFunction, ops.StreamAggregateFunction,
             ops.StreamDistributeMixAddFunction]


@pytest.mark.parametrize("fn", FUNCTIONS)
def test_is_an_autograd_function(fn):
    assert issubclass(fn, torch.autograd.Function)
    assert "forward" in vars(fn) and "backward" in vars(fn)


def test_subclass_runs_its_own_forward():
    class Twice(ops.SinkhornKnoppFunction):
        @staticmethod
        def forward(ctx, inp, num_iters=20, eps=1e-8):
            return 2 * inp

        @staticmethod
        def backward(ctx, g):
            return 3 * g, None, None

    x = torch.ones(2, 3, 3, requires_grad=True)
    out = Twice.apply(x, 5, 1e-8)
    out.sum().backward()
    assert bool((out == 2).all()) and bool((x.grad == 3).all())


def _args(device, seed):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g).to(device)
    B, n, C = 7, 4, 64
    return {ops.SinkhornKnoppFunction: (torch.exp(rnd(B, n, n)),), ops.RMSNormFunction: (rnd(B, C), 1 + rnd(C)),
            ops.StreamAggregateFunction: (rnd(B, n, C), rnd(B, n)),
            ops.StreamDistributeMixAddFunction: (rnd(B, C), rnd(B, n), torch.exp(rnd(B, n, n)), rnd(B, n, C))}


CALLS = {ops.SinkhornKnoppFunction: mhc.sinkhorn_knopp, ops.RMSNormFunction: mhc.rmsnorm,
         ops.StreamAggregateFunction: mhc.stream_aggregate,
         ops.StreamDistributeMixAddFunction: mhc.stream_distribute_mix_add}


@pytest.mark.gpu
@pytest.mark.parametrize("fn", FUNCTIONS)
def test_trace_records_the_call(device, fn):
    traced = torch.jit.trace(lambda *a: CALLS[fn](*a), _args(device, 1)[fn], check_trace=False)
    other = _args(device, 2)[fn]
    assert torch.equal(traced(*other), CALLS[fn](*other))


@pytest.mark.gpu
@pytest.mark.parametrize("fn", FUNCTIONS)
def test_python_function_and_node_agree(device, fn):
    """forward / backward as a subclass runs them, against the C++ node: bitwise."""
    plain = type("Plain", (fn,), {})
    grads = []
    for f in (plain, fn):
        args = [a.requires_grad_(True) for a in _args(device, 3)[fn]]
        out = f.apply(*args)
        g = torch.linspace(-1, 1, out.numel(), device=device).view(out.shape)
        grads.append([out, *torch.autograd.grad(out, args, g)])
    assert all(torch.equal(a, b) for a, b in zip(*grads))
