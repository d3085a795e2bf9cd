"""What the two attention entry points keep for the backward, and their forward and backward as plain functions that return
thresholds, tile mask and supports.  Both run in the native host path (``csrc/torch_binding.cpp``), which holds the buffers
and the choice of the C ABI's entry points once."""

from . import _lib


# What the forward of the autograd functions keeps for the backward besides q, k, v, taus and bmask: the supports it
# found (51.7 KB per 128 query rows and head, whatever the head dim), with which the backward needs no score walk of
# its own.  "auto" keeps them when they take at most twice the bytes of q -- the reference keeps a second output of
# q's size for its backward (adasplash/adasplash_v2.py:1421-1426) -- or 256 MiB; "always" and "never" say what they
# mean.  ``ADSP_KEEP_SUPPORTS`` in the environment sets the initial mode (0 / never, 1 / always, auto).
_KEEP_MODES = ("auto", "always", "never")
_keep_mode = None


def set_keep_supports(mode):
    """Choose what the attention forward keeps for its backward: ``"auto"`` (default), ``"always"`` or ``"never"``.
    Returns the previous mode."""
    global _keep_mode
    if mode not in _KEEP_MODES:
        raise ValueError(f"mode must be one of {_KEEP_MODES}; got {mode!r}")
    old = get_keep_supports()
    _keep_mode = mode
    return old


def get_keep_supports():
    global _keep_mode
    if _keep_mode is None:
        import os

        env = os.environ.get("ADSP_KEEP_SUPPORTS", "auto").lower()
        _keep_mode = {"0": "never", "1": "always"}.get(env, env if env in _KEEP_MODES else "auto")
    return _keep_mode


def keep_code():
    """The mode as the native host path takes it: an index into ("never", "always", "auto")."""
    return {"never": 0, "always": 1, "auto": 2}[_keep_mode or get_keep_supports()]


def _keeps(sup_bytes, q):
    return _lib.native().keeps_supports(keep_code(), sup_bytes, q.numel() * q.element_size())


def launch_forward(q, k, v, *, version, alpha, is_causal, niter, varlen, tile_counts=None, keep_supports=False, tile_mask=True):
    """Enqueue the fused forward on the current stream.  Returns ``(out, taus, bmask)``, and with ``keep_supports`` a
    fourth value: the buffer in which the forward keeps the supports it found for ``launch_backward`` (``None`` where the
    library keeps none: fp32, head dims other than 64 / 128, a caller that asks for the tile statistics, or a buffer
    beyond what ``set_keep_supports`` allows; ``keep_supports="always"`` asks for the buffer whatever the mode).

    The tile mask and the supports are left by the kernels that find them; a short 16-bit call of the entry points goes
    to others.  ``tile_mask=False`` launches what the entry points launch: without ``keep_supports`` what a call
    without a gradient does (``bmask`` is ``None``), with it what a training step does (``bmask`` where the backward reads one).
    """
    mode = None
    if keep_supports:
        mode = 1 if keep_supports == "always" else keep_code()
    out, taus, bmask, sup = _lib.native().attention_forward(q, k, v, version, alpha, is_causal, niter, varlen, mode, tile_mask, tile_counts)
    return (out, taus, bmask, sup) if keep_supports else (out, taus, bmask)


def launch_backward(q, k, v, dout, taus, bmask, *, alpha, is_causal, varlen, supports=None):
    """Enqueue the dQ and dK/dV kernels on the current stream; returns ``(dq, dk, dv)``.

    ``taus`` / ``bmask`` are the thresholds and the tile mask the forward produced, ``supports`` what it kept for this
    call (``launch_forward(..., keep_supports=True)``) or ``None``: then the dQ kernel finds the supports again.  Rows of ``dout`` past a
    sequence's valid length are never used, whatever they hold (the kernels mask them as the reference's
    loads do, adasplash/adasplash_v2.py:1030-1033).
    """
    return _lib.native().attention_backward(q, k, v, dout, taus, bmask, alpha, is_causal, varlen, supports)
