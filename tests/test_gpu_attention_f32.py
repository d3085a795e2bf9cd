"""The single-precision kernels on 32 rows a workgroup (head dims 64 and 128) against the oracle, at the sizes where their split
can go wrong: lengths around a block of 32 and a step of four of them, lists that overflow (flat scores, which send a
workgroup from the lists to walks) and that do not, padding that holds NaN, grouped K/V heads, every alpha mode.

Tolerance 1e-4 as in the other single-precision tests of forward and backward."""

import math

import pytest
import torch

import adasplash_amd as A
from adasplash_amd import _attention, _lib
from adasplash_amd.adasplash_block_mask import tile_sparsity
from oracle import exact
from tests.gpu_util import DEV, max_err

pytestmark = pytest.mark.gpu
TOL = 1e-4


def run(q, k, v, dout, varlen, alpha, causal, grouped):
    qg, kg, vg = (t.to(DEV).requires_grad_(True) for t in (q, k, v))
    vl = None if varlen is None else varlen.to(DEV)
    if grouped:
        out = A.adasplash_v2(qg, kg, vg, varlen=vl)
    else:
        out = A.adasplash_v1(qg, kg, vg, alpha=alpha, is_causal=causal, varlen=vl)
    out.backward(dout.to(DEV))
    return out.detach(), qg.grad, kg.grad, vg.grad


@pytest.mark.parametrize("scale", [0.125, 1.0, 3.0])  # of q: flat scores (lists overflow), ordinary, peaked
@pytest.mark.parametrize("alpha,causal,Hq,Hkv,D", [(1.5, True, 4, 2, 64), (1.5, True, 2, 2, 128), (1.333, False, 2, 2, 64),
                                                   (2.0, False, 1, 1, 128), (1.5, False, 2, 2, 64), (1.125, True, 1, 1, 64)])
def test_lengths_around_blocks_and_steps(alpha, causal, Hq, Hkv, D, scale):
    g = torch.Generator().manual_seed(3)
    N = 517
    varlen = torch.tensor([517, 1, 32, 33, 127, 129, 384], dtype=torch.int32)
    B = len(varlen)
    q = scale * torch.randn(B, Hq, N, D, generator=g)
    k, v = (torch.randn(B, Hkv, N, D, generator=g) for _ in range(2))
    dout = torch.randn(B, Hq, N, D, generator=g)
    want = [exact.dense_entmax_attention(q, k, v, alpha, causal, varlen)]
    want += list(exact.dense_entmax_attention_grads(q, k, v, dout, alpha, causal, varlen))
    for b, n in enumerate(varlen.tolist()):  # the padding may hold anything
        for t in (q, k, v):
            t[b, :, n:] = float("nan")
    got = run(q, k, v, dout, varlen, alpha, causal, Hq != Hkv)
    for name, a, w in zip(("out", "dq", "dk", "dv"), got, want):
        assert torch.isfinite(a).all(), name
        for b, n in enumerate(varlen.tolist()):
            assert (a[b, :, n:] == 0).all(), name
        assert max_err(a, w) < TOL, name


@pytest.mark.parametrize("N,scale", [(64, 1.0), (2048, 1.0), (2048, 0.125), (4096, 3.0)])
def test_same_bits_on_every_call_and_long_rows(N, scale):
    g = torch.Generator().manual_seed(4)
    q = scale * torch.randn(1, 4, N, 64, generator=g)
    k, v = (torch.randn(1, 1, N, 64, generator=g) for _ in range(2))
    dout = torch.randn(1, 4, N, 64, generator=g)
    first = run(q, k, v, dout, None, 1.5, True, True)
    again = run(q, k, v, dout, None, 1.5, True, True)
    assert all(torch.equal(a, b) for a, b in zip(first, again))
    want = [exact.dense_entmax_attention(q, k, v, 1.5, True)]
    want += list(exact.dense_entmax_attention_grads(q, k, v, dout, 1.5, True))
    # Beyond unit scale the bound grows with q: scores of that size round by as much more, a probability's root u moves by
    # what its score is off, and dK sums u (dP - delta) q.
    tol = TOL * max(1.0, scale)
    for name, a, w in zip(("out", "dq", "dk", "dv"), first, want):
        assert max_err(a, w) < tol, name


@pytest.mark.parametrize("scale", [0.125, 1.0, 3.0])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("alpha,causal,Hq,Hkv,D", [(1.5, True, 4, 2, 64), (1.5, True, 2, 2, 128), (1.333, False, 2, 2, 64), (2.0, False, 1, 1, 128)])
def test_16bit_inference_lengths_around_blocks_and_steps(dtype, alpha, causal, Hq, Hkv, D, scale):
    """Without a gradient short 16-bit calls take the same forward; the bound is that of the other 16-bit forward tests."""
    g = torch.Generator().manual_seed(5)
    N = 517
    varlen = torch.tensor([517, 1, 32, 33, 127, 129, 384], dtype=torch.int32)
    B = len(varlen)
    q = (scale * torch.randn(B, Hq, N, D, generator=g)).to(dtype)
    k, v = (torch.randn(B, Hkv, N, D, generator=g).to(dtype) for _ in range(2))
    want = exact.dense_entmax_attention(q, k, v, alpha, causal, varlen)
    for b, n in enumerate(varlen.tolist()):
        for t in (q, k, v):
            t[b, :, n:] = float("nan")
    args = [t.to(DEV) for t in (q, k, v)]
    vl = varlen.to(DEV)
    run16 = lambda: A.adasplash_v2(*args, varlen=vl) if Hq != Hkv else A.adasplash_v1(*args, alpha=alpha, is_causal=causal, varlen=vl)
    got = run16()
    assert torch.equal(got, run16())
    assert torch.isfinite(got).all()
    for b, n in enumerate(varlen.tolist()):
        assert (got[b, :, n:] == 0).all()
    assert max_err(got, want) < 2e-2


@pytest.mark.parametrize("scale", [0.125, 1.0, 3.0])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("alpha,causal,Hq,Hkv,D", [(1.5, True, 4, 2, 64), (1.5, True, 2, 2, 128), (1.333, False, 2, 2, 64), (2.0, False, 1, 1, 128)])
def test_16bit_gradients_lengths_around_blocks_and_steps(dtype, alpha, causal, Hq, Hkv, D, scale):
    """Short 16-bit training steps; bounds as in the other 16-bit tests (outputs 2e-2, gradients 4e-2 of their magnitude), where
    the gradients of k scale with q."""
    g = torch.Generator().manual_seed(6)
    N = 517
    varlen = torch.tensor([517, 1, 32, 33, 127, 129, 384], dtype=torch.int32)
    B = len(varlen)
    q = (scale * torch.randn(B, Hq, N, D, generator=g)).to(dtype)
    k, v = (torch.randn(B, Hkv, N, D, generator=g).to(dtype) for _ in range(2))
    dout = torch.randn(B, Hq, N, D, generator=g).to(dtype)
    want = [exact.dense_entmax_attention(q, k, v, alpha, causal, varlen)]
    want += list(exact.dense_entmax_attention_grads(q, k, v, dout, alpha, causal, varlen))
    for b, n in enumerate(varlen.tolist()):
        for t in (q, k, v):
            t[b, :, n:] = float("nan")
    got = run(q, k, v, dout, varlen, alpha, causal, Hq != Hkv)
    again = run(q, k, v, dout, varlen, alpha, causal, Hq != Hkv)
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    for name, a, w in zip(("out", "dq", "dk", "dv"), got, want):
        assert torch.isfinite(a).all(), name
        for b, n in enumerate(varlen.tolist()):
            assert (a[b, :, n:] == 0).all(), name
        if alpha == 2.0 and name in ("dq", "dk"):
            # sparsemax's derivative jumps at the border of the support: a key that rounding puts on the other side changes its row
            num, den = (a.double().cpu() - w.double()).norm(), w.double().norm()
            assert num < 2e-2 * den, name
        else:
            assert max_err(a, w) < (2e-2 if name == "out" else 4e-2 * max(1.0, scale)), name


@pytest.mark.parametrize("scale", [0.125, 1.0])
@pytest.mark.parametrize("alpha,causal,Hq,Hkv,D", [(1.5, True, 2, 1, 64), (1.5, True, 1, 1, 128), (1.333, False, 1, 1, 64)])
@pytest.mark.parametrize("dout_scale", [1e-6, 1.0, 3e4])
def test_f16_dq_for_gradients_at_the_ends_of_the_types_range(dout_scale, alpha, causal, Hq, Hkv, D, scale):
    """dQ's weights u (dP - delta) are held to fp32: neither upstream gradients near f16's smallest numbers nor weights
    beyond its largest (dout of 3e4 gives some of 1e5) may cost anything.  k and q are scaled against each other so that dq
    itself is an ordinary number.  Bound on the error (2-norm, relative): rounding dq to f16 leaves at most 2^-11 of each
    entry; thresholds and sums in fp32 add less than that again."""
    g = torch.Generator().manual_seed(8)
    N = 517
    kscale = 256.0 if dout_scale < 1.0 else (1.0 if dout_scale == 1.0 else 2.0 ** -10)
    varlen = torch.tensor([517, 130], dtype=torch.int32)
    q = (scale / kscale * torch.randn(2, Hq, N, D, generator=g)).half()
    k = (kscale * torch.randn(2, Hkv, N, D, generator=g)).half()
    v = torch.randn(2, Hkv, N, D, generator=g).half()
    dout = (dout_scale * torch.randn(2, Hq, N, D, generator=g)).clamp(-6e4, 6e4).half()
    want = exact.dense_entmax_attention_grads(q, k, v, dout, alpha, causal, varlen)[0]
    got = run(q, k, v, dout, varlen, alpha, causal, Hq != Hkv)[1].double().cpu()
    assert torch.isfinite(got).all()
    assert (got - want).norm() < 2.0 ** -10 * want.norm()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,Hq,Hkv,N,short", [(1, 8, 2, 512, True), (2, 16, 16, 2048, False)])
def test_the_plain_functions_launch_what_the_entry_points_launch(B, Hq, Hkv, N, short, dtype):
    """``launch_forward(tile_mask=False)``, alone and with ``keep_supports``, and ``launch_backward`` behind it: the bits of a call
    without a gradient and of a training step.  A short 16-bit call leaves neither tile mask nor supports there, and
    both by default."""
    g = torch.Generator().manual_seed(9)
    q = torch.randn(B, Hq, N, 64, generator=g).to(dtype).to(DEV)
    k, v = (torch.randn(B, Hkv, N, 64, generator=g).to(dtype).to(DEV) for _ in range(2))
    dout = torch.randn(B, Hq, N, 64, generator=g).to(dtype).to(DEV)
    kw = dict(version=2, alpha=1.5, is_causal=True, niter=1, varlen=None)
    out, taus, bmask = _attention.launch_forward(q, k, v, tile_mask=False, **kw)
    assert bmask is None and torch.equal(out, A.adasplash_v2(q, k, v))
    out, taus, bmask, sup = _attention.launch_forward(q, k, v, tile_mask=False, keep_supports=True, **kw)
    reads = dtype == torch.bfloat16 and not short
    assert (bmask is not None) == reads and (sup is not None) == reads
    got = _attention.launch_backward(q, k, v, dout, taus, bmask, alpha=1.5, is_causal=True, varlen=None, supports=sup)
    want_out, *want = run(q, k, v, dout, None, 1.5, True, True)
    assert torch.equal(out, want_out) and all(torch.equal(a, b) for a, b in zip(got, want))
    out, taus, bmask, sup = _attention.launch_forward(q, k, v, keep_supports=True, **kw)
    assert bmask is not None and (sup is not None) == (dtype == torch.bfloat16)
    assert max_err(out, want_out.float().cpu()) < 2e-2


def _untouched(nbytes):
    return torch.full((max(nbytes, 16),), 0xA5, device=DEV, dtype=torch.uint8)


def _short_16bit_forward(q, k, v, alpha, causal):
    """The forward without tile mask through the C ABI, and proof that it took the kernel on 32 rows: only the others write
    to the workspace."""
    lib = _lib.load()
    B, Hq, N, D = q.shape
    Hkv, dt = k.shape[1], _lib.dtype_code(q)
    ws = _untouched(lib.adsp_attn_workspace_bytes(B, Hq, Hkv, N, D, dt))
    out, taus = torch.full_like(q, float("nan")), torch.empty(B, Hq, N, device=DEV)
    head = (q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), taus.data_ptr(), None, None, 0)
    stream = _lib.current_stream(q.device)
    if causal:
        st = lib.adsp_attn_v2_fwd(*head, B, Hq, Hkv, N, D, dt, 1, ws.data_ptr(), ws.numel(), stream)
    else:
        st = lib.adsp_attn_v1_fwd(*head, B, Hq, N, D, dt, alpha, 0, 10, ws.data_ptr(), ws.numel(), None, stream)
    assert st == 0 and (ws == 0xA5).all()
    return out, taus


@pytest.mark.parametrize("scale", [0.125, 1.0, 3.0])
@pytest.mark.parametrize("N,Hq,Hkv,D,alpha,causal,dtype", [
    (8192, 1, 1, 64, 1.5, True, torch.bfloat16), (8192, 1, 1, 128, 1.5, True, torch.float16), (4095, 4, 1, 64, 1.5, True, torch.float16),
    (1024, 16, 4, 128, 1.5, True, torch.bfloat16), (4096, 1, 1, 128, 1.5, False, torch.bfloat16), (4096, 1, 1, 64, 1.333, False, torch.float16),
    (2048, 4, 4, 64, 2.0, False, torch.bfloat16)])
def test_16bit_inference_on_long_sequences(N, Hq, Hkv, D, alpha, causal, dtype, scale):
    """Walks of up to 64 steps a wave, to the longest sequences that take this route: rows around steps and blocks and at both
    ends, thresholds and outputs.  Thresholds: fp32 sums over 16-bit products, and steps until one is below 2e-5."""
    g = torch.Generator().manual_seed(10)
    q = (scale * torch.randn(1, Hq, N, D, generator=g)).to(dtype).to(DEV)
    k, v = (torch.randn(1, Hkv, N, D, generator=g).to(dtype).to(DEV) for _ in range(2))
    out, taus = _short_16bit_forward(q, k, v, alpha, causal)
    rows = sorted({r for r in (0, 1, 31, 32, 127, 128, 1023, 1024, N // 2 + 5, N - 33, N - 32, N - 2, N - 1) if r < N})
    for h in {0, Hq - 1}:
        kk = k[0, h // (Hq // Hkv)].double().cpu()
        s = q[0, h, rows].double().cpu() @ kk.t() / D ** 0.5
        if causal:
            s = s.masked_fill(torch.arange(N)[None, :] > torch.tensor(rows)[:, None], float("-inf"))
        p, tau = exact.entmax_rows(s, alpha, return_tau=True)
        assert max_err(out[0, h, rows], p @ v[0, h // (Hq // Hkv)].double().cpu()) < 2e-2
        assert (taus[0, h, rows].double().cpu() - tau.double().view(-1)).abs().max().item() < 5e-5 * max(1.0, scale)


@pytest.mark.parametrize("scale", [0.125, 1.0, 3.0])
@pytest.mark.parametrize("N,Hq,Hkv,D,alpha,causal,dtype", [
    (4096, 1, 1, 64, 1.5, True, torch.bfloat16), (1024, 4, 1, 64, 1.5, True, torch.float16), (3072, 1, 1, 128, 1.5, True, torch.bfloat16),
    (3072, 1, 1, 64, 1.5, False, torch.bfloat16), (2048, 3, 3, 128, 1.5, False, torch.float16), (2048, 1, 1, 64, 1.333, False, torch.bfloat16)])
def test_16bit_gradients_on_long_sequences(N, Hq, Hkv, D, alpha, causal, dtype, scale):
    """Training steps at the ends of the route's range, whole tensors; bounds as in the other 16-bit tests."""
    g = torch.Generator().manual_seed(11)
    q = (scale * torch.randn(1, Hq, N, D, generator=g)).to(dtype)
    k, v = (torch.randn(1, Hkv, N, D, generator=g).to(dtype) for _ in range(2))
    dout = torch.randn(1, Hq, N, D, generator=g).to(dtype)
    assert _lib.load().adsp_attn_bwd_reads_bmask(1, Hq, Hkv, N, D, _lib.dtype_code(q), alpha, int(causal)) == 0
    varlen = torch.tensor([N], dtype=torch.int32)  # (N need not be a power of two)
    got = run(q, k, v, dout, varlen, alpha, causal, causal)
    want = [exact.dense_entmax_attention(q, k, v, alpha, causal, varlen)]
    want += list(exact.dense_entmax_attention_grads(q, k, v, dout, alpha, causal, varlen))
    for name, a, w in zip(("out", "dq", "dk", "dv"), got, want):
        assert max_err(a, w) < (2e-2 if name == "out" else 4e-2 * max(1.0, scale)), name


@pytest.mark.parametrize("alpha,dtype", [(1.5, torch.float32), (1.333, torch.float32), (1.125, torch.float32), (1.5, torch.bfloat16)])
@pytest.mark.parametrize("members", [8, 20, 26, 31, 32, 33, 80, 97])
def test_lists_that_fill_up_between_two_solves(members, alpha, dtype):
    """Late keys of one wave (blocks 16, 20, 24, 28 of 32 keys each: the first wave's between the solves after 4 and 8 steps), so many
    of them above all others that the wave's list of every row fits, just fits, or overflows; the keys in front of them
    leave entries that then lie below the bound.  fp32: as everywhere here; bf16: 2^-8 of the result, its rounding and the weights'."""
    g = torch.Generator().manual_seed(members)
    N, D = 1031, 64
    axis = torch.zeros(D)
    axis[0] = 1.0
    q = (0.3 * torch.randn(1, 1, N, D, generator=g) + 4.0 * axis).to(dtype)
    k = torch.randn(1, 1, N, D, generator=g)
    k[..., 0] = 0.2 * torch.randn(1, 1, N, generator=g)
    late = [32 * (16 + 4 * (i % 4)) + i // 4 for i in range(members)]
    k[0, 0, late, 0] = 1.0 + 0.05 * torch.randn(members, generator=g)
    k = k.to(dtype)
    v = torch.randn(1, 1, N, D, generator=g).to(dtype)
    vl = torch.tensor([N], dtype=torch.int32)
    want = exact.dense_entmax_attention(q, k, v, alpha, False, vl)
    got = A.adasplash_v1(*(t.to(DEV) for t in (q, k, v)), alpha=alpha, is_causal=False, varlen=vl.to(DEV)).double().cpu()
    assert (got - want).norm() <= (2e-6 if dtype == torch.float32 else 2.0 ** -8) * want.norm()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("norm", [1.0, 100.0, 1000.0])
def test_dq_of_an_outlying_row_of_v_that_is_barely_a_member(D, norm):
    """Key 0 is the only member of its block and wave's first, with u = 2^-10 of 300 members, and its V row is `norm` times the others'.  u is exact (q has one
    column, tau is given as 1, and u is what fp32 makes of scores that it holds exactly), so what is left is dP, delta and the sums: 2e-6 as
    below; a dQ whose sums are taken around that key's dP is off by 5e-5 and more (K has a mean of 1, which makes them large)."""
    g = torch.Generator().manual_seed(14)
    N, members = 512, 300
    n, left = torch.zeros(N, dtype=torch.int64), (1 << 20) - 1  # u in units of 2^-10: sum u^2 = 1
    n[0] = 1
    at = (torch.randperm(N - 128, generator=g)[:members] + 128).tolist()
    for i, j in enumerate(at):
        n[j] = math.isqrt(left) if i >= members - 8 else max(1, int(math.sqrt(left / (members - i)) * (0.7 + 0.6 * torch.rand((), generator=g).item())))
        left -= int(n[j]) ** 2
    z = torch.where(n > 0, 1.0 + n / 1024, -torch.ones(N))
    q = torch.zeros(1, 1, N, D)
    q[..., 0] = 16.0
    k, v, dout = (torch.randn(1, 1, N, D, generator=g) for _ in range(3))
    k += 1.0
    k[0, 0, :, 0] = z * (D / 64) ** 0.5  # (exact at head dim 64 only)
    v[:, :, 0] *= norm
    qscale = torch.tensor(0.5 * D ** -0.5, dtype=torch.float32).double()
    u = ((16.0 * k[0, 0, :, 0].double()) * qscale - 1.0).float().double().clamp_min(0.0)
    dp = dout[0, 0].double() @ v[0, 0].double().t()
    want = (u * (dp - (dp @ u / u.sum())[:, None])) @ k[0, 0].double() / D ** 0.5
    a = [t.to(DEV) for t in (q, k, v, dout)]
    _, taus, bmask = _attention.launch_forward(*a[:3], version=1, alpha=1.5, is_causal=False, niter=4, varlen=None)
    got = _attention.launch_backward(*a, torch.ones_like(taus), bmask, alpha=1.5, is_causal=False, varlen=None)[0][0, 0].double().cpu()
    assert (got - want).norm() <= 2e-6 * want.norm()


@pytest.mark.parametrize("alpha,causal,D", [(1.5, True, 64), (1.5, False, 128), (1.333, False, 64), (2.0, False, 64)])
@pytest.mark.parametrize("tails,k_mean", [(1.5, 0.0), (0.0, 3.0), (1.5, 3.0)])
def test_errors_with_heavy_tails_and_a_common_part_of_k(alpha, causal, D, tails, k_mean):
    """V rows whose norms have heavy tails (dP differs from block to block), and K with a mean, which cancels in dQ as the weights' derivatives add up to
    0: 2e-6 as below, times the K that cancels over the K that does not."""
    g = torch.Generator().manual_seed(15)
    N = 512
    q, k, v, dout = (torch.randn(1, 2, N, D, generator=g) for _ in range(4))
    if tails:
        v *= torch.rand(1, 2, N, 1, generator=g) ** (-1.0 / tails)
    k += k_mean
    want = [exact.dense_entmax_attention(q, k, v, alpha, causal)]
    want += list(exact.dense_entmax_attention_grads(q, k, v, dout, alpha, causal))
    bound = 2e-6 * max(1.0, k_mean)
    for name, a, w in zip(("out", "dq", "dk", "dv"), run(q, k, v, dout, None, alpha, causal, False), want):
        rel = ((a.double().cpu() - w.double()).norm() / w.double().norm()).item()
        assert rel < bound, (name, rel)


@pytest.mark.parametrize("alpha,causal,Hq,Hkv,D,q_scale,v_mean", [(1.5, True, 4, 2, 64, 1.0, 0.0), (1.5, True, 2, 1, 128, 3.0, 0.0), (1.5, True, 2, 2, 64, 0.125, 10.0),
                                                                  (1.5, True, 2, 2, 128, 1.0, 10.0), (1.333, False, 2, 2, 64, 1.0, 0.0), (2.0, False, 2, 2, 128, 1.0, 0.0)])
def test_errors_are_those_of_single_precision(alpha, causal, Hq, Hkv, D, q_scale, v_mean):
    """Products of three-part operands, and dQ from sums around a row's running delta: 2e-6 is 17 roundings of 2^-23, about twice what products in
    single precision show for a V of mean 10; a product with a third part that is left out costs about 5e-6 of a score."""
    g = torch.Generator().manual_seed(12)
    N, varlen = 289, torch.tensor([289, 250], dtype=torch.int32)
    q = q_scale * torch.randn(2, Hq, N, D, generator=g)
    k, v = (torch.randn(2, Hkv, N, D, generator=g) for _ in range(2))
    v += v_mean
    dout = torch.randn(2, Hq, N, D, generator=g)
    want = [exact.dense_entmax_attention(q, k, v, alpha, causal, varlen)]
    want += list(exact.dense_entmax_attention_grads(q, k, v, dout, alpha, causal, varlen))
    for name, a, w in zip(("out", "dq", "dk", "dv"), run(q, k, v, dout, varlen, alpha, causal, Hq != Hkv), want):
        rel = ((a.double().cpu() - w.double()).norm() / w.double().norm()).item()
        assert rel < 2e-6, (name, rel)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("scale", [1.0, 0.05])  # of q: lists that hold, and that overflow
@pytest.mark.parametrize("side,value,times", [("k", -math.inf, 1.0), ("k", math.inf, 1.0), ("k", math.nan, 1.0), ("q", math.inf, 1.0), ("k", -3e38, 100.0), ("k", 3e38, 100.0)])
def test_scores_that_are_not_finite(D, scale, side, value, times):
    """An infinite or NaN operand, and products beyond the type's range: as the kernels on 128 rows a workgroup, which form them in single precision.  A row with a
    score of +inf is 0, as are its gradients; keys of score -inf or NaN have no weight and no gradients."""
    g = torch.Generator().manual_seed(16)
    N = 256
    q, k, v, dout = (torch.randn(1, 2, N, D, generator=g) for _ in range(4))
    q *= scale
    q[..., 5], k[..., 5] = (times, 0.0) if side == "k" else (0.0, 1.0)
    at = slice(17, None, 40)
    (k if side == "k" else q)[:, :, at, 5] = value
    want = tile_sparsity(*(t.to(DEV) for t in (q, k, v)), alpha=1.5)[0]
    out, dq, dk, dv = run(q, k, v, dout, None, 1.5, False, False)
    assert torch.isfinite(want).all() and max_err(out, want.cpu()) < TOL
    top = value == math.inf or value > 1e38
    assert bool((out[:, :, at] == 0).all()) == top
    if top and side == "k":
        assert (dq == 0).all() and (dk == 0).all() and (dv == 0).all()
    elif side == "q":
        assert (dq[:, :, at] == 0).all() and torch.isfinite(dv).all()
    else:
        assert (dk[:, :, at] == 0).all() and (dv[:, :, at] == 0).all() and torch.isfinite(dk).all() and torch.isfinite(dv).all()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("scale", [1.0, 0.05])
def test_an_infinite_value_stays_in_its_column(D, scale):
    """V with an infinite entry: infinite in the rows that have the key, and nowhere but in its column."""
    g = torch.Generator().manual_seed(17)
    q, k, v = (torch.randn(1, 2, 256, D, generator=g) for _ in range(3))
    q *= scale
    p = exact.entmax_rows(exact.attention_scores(q, k, False)[0], 1.5)[..., 17]
    want = exact.dense_entmax_attention(q, k, v, 1.5)
    v[:, :, 17, 3] = math.inf
    out = A.adasplash_v1(*(t.to(DEV) for t in (q, k, v)), alpha=1.5, is_causal=False).cpu()
    assert (out[..., 3][p > 1e-6] == math.inf).all()
    keep = [c for c in range(D) if c != 3]
    assert max_err(out[..., keep], want[..., keep]) < TOL


@pytest.mark.parametrize("D", [64, 128])
def test_largest_finite_values_stay_finite(D):
    """The first of a value's three parts is cut off, not rounded: the type's largest value stays finite, and times 0 it is 0."""
    g = torch.Generator().manual_seed(13)
    q, k, v, dout = (torch.randn(1, 2, 128, D, generator=g) for _ in range(4))
    q[..., 5] = 0.0
    k[..., 5] = torch.finfo(torch.float32).max
    got = run(q, k, v, dout, None, 1.5, True, False)
    k[..., 5] = 0.0
    want = run(q, k, v, dout, None, 1.5, True, False)
    for name, a, w in zip(("out", "dk", "dv"), (got[0], got[2], got[3]), (want[0], want[2], want[3])):
        assert torch.equal(a, w), name
    keep = [c for c in range(D) if c != 5]  # (column 5 of dQ is sums of the largest value, in which u K overflows)
    assert torch.equal(got[1][..., keep], want[1][..., keep])


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("small,exponent", [("dout", -100), ("v", -100), ("q", -100), ("dout", -116), ("v", -116), ("q", -116)])
def test_small_magnitudes(D, small, exponent):
    """Operands whose third part reaches below bf16's smallest number, 2^-133, lose it: up to 2^-134 of a value, 2^-18 of one of 2^-116 and nothing above 2^-110.
    2e-6 as above, and twice that."""
    g = torch.Generator().manual_seed(18)
    t = dict(zip(("q", "k", "v", "dout"), (torch.randn(1, 2, 256, D, generator=g) for _ in range(4))))
    t[small] *= 2.0 ** exponent
    if small == "q":
        t["k"] *= 2.0 ** -exponent  # the scores stay what they are
    a = list(t.values())
    want = [exact.dense_entmax_attention(*a[:3], 1.5, True)] + list(exact.dense_entmax_attention_grads(*a, 1.5, True))
    bound = 2e-6 + (2 * 2.0 ** (-134 - exponent) if exponent < -110 else 0.0)
    for name, got, w in zip(("out", "dq", "dk", "dv"), run(*a, None, 1.5, True, False), want):
        rel = ((got.double().cpu() - w).norm() / w.norm()).item()
        assert rel < bound, (name, rel)
