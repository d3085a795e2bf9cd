"""GPU test of forward-mode differentiation: the kernels have no forward derivative, and a call that is asked for one must say
so (a result without a tangent reads as a derivative of zero)."""

import pytest
import torch
import torch.autograd.forward_ad as fwd

import adasplash_amd as A
from adasplash_amd import dense
from tests.gpu_util import DEV

pytestmark = pytest.mark.gpu


def _calls():
    g = torch.Generator(device=DEV).manual_seed(1)
    rand = lambda *shape: torch.randn(*shape, generator=g, device=DEV)  # noqa: E731
    qkv = [rand(1, 2, 64, 64) for _ in range(3)]
    step = [rand(1, 2, 1, 64), rand(1, 2, 100, 64), rand(1, 2, 100, 64)]
    slopes = torch.tensor([0.5, 0.25], device=DEV)
    return {
        "rows": ([rand(4, 100)], A.triton_entmax),
        "attention": (qkv, A.adasplash),
        "attention_block_mask": (qkv, lambda q, k, v: A.adasplash(q, k, v, alpha=1.333, is_causal=False)),
        "decode": (step + [slopes], lambda q, k, v, s: dense.slow_entmax_attention(q, k, v, is_causal=True, alibi_slopes=s)),
    }


@pytest.mark.parametrize("grad", [False, True])  # (with and without a reverse-mode graph)
@pytest.mark.parametrize("name,which", [("rows", 0), ("attention", 0), ("attention", 1), ("attention", 2), ("attention_block_mask", 0),
                                        ("decode", 0), ("decode", 1), ("decode", 3)])
def test_a_tangent_is_refused(name, which, grad):
    args, fn = _calls()[name]
    args = [t.requires_grad_(grad) for t in args]
    with fwd.dual_level():
        args = [fwd.make_dual(t, torch.ones_like(t)) if i == which else t for i, t in enumerate(args)]
        with pytest.raises(NotImplementedError):
            fn(*args)
        with torch.no_grad(), pytest.raises(NotImplementedError):
            fn(*args)


def test_a_tangent_of_v_passes_through_a_decoding_step():
    """The output is linear in v, and the dense path that serves such a call carries the tangent."""
    (q, k, v, s), fn = _calls()["decode"]
    with fwd.dual_level():
        t = torch.randn_like(v)
        got = fwd.unpack_dual(fn(q, k, fwd.make_dual(v, t), s)).tangent
    assert (got - fn(q, k, t, s)).abs().max().item() < 1e-4


def test_a_decoding_step_on_tensors_that_are_more_than_their_data():
    """vmap over v, and caches that are views with a sign (as the imaginary part of a conjugate is): the dense path's
    operators honour both."""
    (q, k, v, s), fn = _calls()["decode"]
    vs = torch.stack([v, 2 * v])
    got = torch.func.vmap(lambda x: fn(q, k, x, s))(vs)
    assert (got - torch.stack([fn(q, k, x, s) for x in vs])).abs().max().item() < 1e-4
    assert (fn(q, torch._neg_view(k), v, s) - fn(q, -k, v, s)).abs().max().item() < 1e-4
    assert (fn(q, k, torch._neg_view(v), s) - fn(q, k, -v, s)).abs().max().item() < 1e-4
