"""AdaSplash-2: causal entmax-1.5 attention with GQA and variable lengths on gfx950.

Same call surface as the reference module of this name: ``sparse_attn(q, k, v, niter=1, varlen=None)``
(``adasplash/adasplash_v2.py:1567-1591``), same argument checks as the autograd wrapper there
(``adasplash/adasplash_v2.py:1243-1276``).
"""

from . import _attention, _lib

BMASK_TILE = 64


def sparse_attn(q, k, v, niter=1, varlen=None):
    """Causal entmax-1.5 sparse attention.

    q: ``(batch, n_heads, seq_len, head_dim)``; k, v: ``(batch, n_kv_heads, seq_len, head_dim)`` with
    ``n_heads`` a multiple of ``n_kv_heads``; ``niter``: refinement passes of the threshold solver after
    its histogram bracket; ``varlen``: optional ``(batch,)`` int32/int64 valid lengths (right padding),
    padded output rows are zero.  Returns a tensor like ``q``.
    """
    # (checks, buffers, launches and autograd: csrc/torch_binding.cpp)
    return _lib.native().attention(q, k, v, 2, 1.5, True, niter, varlen, _attention.keep_code())


def _install_callable_module():
    import inspect
    import sys
    import types

    class _CallableModule(types.ModuleType):
        def __call__(self, *args, **kwargs):
            return sparse_attn(*args, **kwargs)

    module = sys.modules[__name__]
    module.__class__ = _CallableModule
    module.__signature__ = inspect.signature(sparse_attn)


_install_callable_module()
