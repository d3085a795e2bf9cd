"""Row-wise alpha-entmax backed by the gfx950 rows kernel.

Same call surface as the reference module of this name (``adasplash/triton_entmax_v2.py:690-731``):
``triton_entmax(x, alpha=1.5, n_iter=2, use_histogram=True, fast_math=False)``,
``triton_sparsemax(x, **kw)``, ``triton_entmax15(x, **kw)``.  The name is kept for drop-in use; no
Triton is involved.
"""

from . import _lib


class _EntmaxRows:
    """Counterpart of ``_entmax_triton`` (``adasplash/triton_entmax_v2.py:620-687``): ``apply(x, alpha, n_iter, use_histogram,
    fast_math)`` runs in the native host path (``csrc/torch_binding.cpp``), gradient included."""

    @staticmethod
    def apply(x, alpha=1.5, n_iter=10, use_histogram=True, fast_math=False):
        return _lib.native().entmax_rows(x, alpha, n_iter, use_histogram, fast_math)


def triton_entmax(x, alpha=1.5, n_iter=2, use_histogram=True, fast_math=False):
    """alpha-entmax over the last dimension of a contiguous tensor (any leading shape).

    For alpha outside {1.5, 2.0} the histogram initialisation is switched off and at least ten
    refinement steps are taken, as the reference does (``adasplash/triton_entmax_v2.py:713-716``).
    """
    if alpha not in (1.5, 2.0):
        use_histogram = False
        n_iter = max(n_iter, 10)
    return _EntmaxRows.apply(x, alpha, n_iter, use_histogram, fast_math)


def triton_sparsemax(x, **kwargs):
    """Sparsemax (entmax with alpha = 2.0)."""
    return triton_entmax(x, alpha=2.0, **kwargs)


def triton_entmax15(x, **kwargs):
    """Entmax-1.5 with histogram initialisation."""
    return triton_entmax(x, alpha=1.5, **kwargs)


def _install_callable_module():
    # keeps `adasplash_amd.triton_entmax_v2(x)` callable after the submodule import rebinds the name
    import inspect
    import sys
    import types

    class _CallableModule(types.ModuleType):
        def __call__(self, *args, **kwargs):
            return triton_entmax(*args, **kwargs)

    module = sys.modules[__name__]
    module.__class__ = _CallableModule
    module.__signature__ = inspect.signature(triton_entmax)


_install_callable_module()
