"""The 16-bit kernels that visit all pairs of a row (head dims 64 and 128) against the oracle, where their split can go wrong: lengths
around a block of 32, a tile of 128 and a workgroup's rows, workgroups of 128, 64 and 32 rows, padding that holds NaN, grouped
K/V heads, every alpha mode.

Bound on the error of a whole tensor (2-norm, relative): a weight is rounded to the type before it multiplies a row, and the result
once more, each by at most 2^-9 (bf16) or 2^-11 (f16) of itself, together at most 2^-8 or 2^-10.  alpha = 2: a key that
rounding puts on the other side of the support's border changes its row's gradient at once, 2e-2 as in the other tests."""

import os

import pytest
import torch

import adasplash_amd as A
from adasplash_amd import _attention, _lib
from oracle import exact
from tests.gpu_util import DEV

pytestmark = pytest.mark.gpu
UNIT = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -11}


def problem(B, Hq, Hkv, N, D, dtype, scale, lengths):
    g = torch.Generator().manual_seed(12)
    q = (scale * torch.randn(B, Hq, N, D, generator=g)).to(dtype)
    k, v = (torch.randn(B, Hkv, N, D, generator=g).to(dtype) for _ in range(2))
    dout = torch.randn(B, Hq, N, D, generator=g).to(dtype)
    varlen = torch.tensor([lengths[b % len(lengths)] for b in range(B)], dtype=torch.int32)
    return q, k, v, dout, varlen


def check(got, q, k, v, dout, varlen, alpha, causal, items):
    """``got``: output alone or output and gradients; compared on the given batch items, zeros behind every item's length"""
    q, k, v, dout, vl = q[items], k[items], v[items], dout[items], varlen[items]
    want = [exact.dense_entmax_attention(q, k, v, alpha, causal, vl)]
    if len(got) > 1:
        want += list(exact.dense_entmax_attention_grads(q, k, v, dout, alpha, causal, vl))
    for name, a, w in zip(("out", "dq", "dk", "dv"), got, want):
        assert torch.isfinite(a).all(), name
        for b, n in enumerate(varlen.tolist()):
            assert (a[b, :, n:] == 0).all(), name
        err = ((a[items].double().cpu() - w.double()).norm() / w.double().norm()).item()
        assert err < (2e-2 if alpha == 2.0 and name in ("dq", "dk") else 2 * UNIT[a.dtype]), (name, err)


def run(q, k, v, dout, varlen, alpha, causal, train=True):
    q, k, v = (t.clone() for t in (q, k, v))
    for b, n in enumerate(varlen.tolist()):  # the padding may hold anything
        for t in (q, k, v):
            t[b, :, n:] = float("nan")
    q, k, v = (t.to(DEV).requires_grad_(train) for t in (q, k, v))
    vl = varlen.to(DEV)
    if q.shape[1] != k.shape[1]:
        out = A.adasplash_v2(q, k, v, niter=10, varlen=vl)
    else:
        out = A.adasplash_v1(q, k, v, alpha=alpha, is_causal=causal, niter=10, varlen=vl)
    if not train:
        return (out,)
    out.backward(dout.to(DEV))
    return out.detach(), q.grad, k.grad, v.grad


@pytest.fixture
def no_supports():
    old = os.environ.get("ADSP_SPARSE")
    os.environ["ADSP_SPARSE"] = "0"
    yield
    if old is None:
        os.environ.pop("ADSP_SPARSE", None)
    else:
        os.environ["ADSP_SPARSE"] = old


@pytest.mark.parametrize("scale", [0.125, 1.0])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,N,D,alpha,causal,lengths", [
    # rows of an item, queries and keys: from 8192 workgroups of 128 rows, from 2048 of 64, below of 32
    (1, 16, 16, 1027, 64, 1.5, True, [1027]), (1, 16, 4, 1027, 128, 1.5, True, [1027]), (2, 8, 2, 577, 64, 1.5, True, [577, 513]),
    (6, 2, 1, 300, 128, 1.5, True, [300, 1, 31, 32, 129, 257]), (6, 2, 2, 300, 64, 1.333, False, [300, 1, 31, 32, 129, 257]),
    (2, 8, 8, 577, 128, 1.333, False, [577, 127]), (1, 13, 13, 1283, 128, 1.5, False, [1283]), (1, 16, 16, 1030, 64, 2.0, False, [1025]),
    (2, 8, 8, 515, 128, 2.0, False, [515, 65])])
def test_gradients_on_all_pairs(no_supports, B, Hq, Hkv, N, D, alpha, causal, lengths, dtype, scale):
    q, k, v, dout, varlen = problem(B, Hq, Hkv, N, D, dtype, scale, lengths)
    got = run(q, k, v, dout, varlen, alpha, causal)
    assert all(torch.equal(a, b) for a, b in zip(got, run(q, k, v, dout, varlen, alpha, causal)))
    check(got, q, k, v, dout, varlen, alpha, causal, list(range(B)))


@pytest.mark.parametrize("scale", [0.125, 1.0])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,N,D,alpha,causal,lengths", [
    (70, 8, 4, 500, 64, 1.5, True, [500, 1, 255, 499, 64]), (6, 12, 12, 500, 128, 1.333, False, [500, 129]), (2, 4, 4, 1024, 64, 1.5, True, [1024, 515]),
    (1, 2, 2, 1997, 64, 2.0, False, [1997]), (1, 4, 2, 1023, 128, 1.5, True, [1023]),
    # rows of the batch: from 32768 workgroups of 128 rows, from 16384 of 64, below of 32
    (65, 8, 8, 64, 64, 1.5, True, [64, 63, 33, 32, 1]), (33, 16, 8, 64, 128, 1.5, True, [64, 31, 2]), (40, 8, 2, 97, 64, 1.5, True, [97, 96, 65]),
    (3, 2, 2, 415, 128, 1.333, False, [415, 385, 128]), (20, 12, 12, 99, 64, 2.0, False, [99, 34])])
def test_gradients_of_short_problems(B, Hq, Hkv, N, D, alpha, causal, lengths, dtype, scale):
    q, k, v, dout, varlen = problem(B, Hq, Hkv, N, D, dtype, scale, lengths)
    assert _lib.load().adsp_attn_bwd_reads_bmask(B, Hq, Hkv, N, D, _lib.dtype_code(q), alpha, int(causal)) == 0
    got = run(q, k, v, dout, varlen, alpha, causal)
    assert all(torch.equal(a, b) for a, b in zip(got, run(q, k, v, dout, varlen, alpha, causal)))
    check(got, q, k, v, dout, varlen, alpha, causal, sorted({*range(min(B, len(lengths))), B - 1}))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq,Hkv,D,alpha,causal", [(2, 1, 64, 1.5, True), (1, 1, 128, 1.5, False), (1, 1, 64, 1.333, False), (1, 1, 128, 2.0, False)])
@pytest.mark.parametrize("N,scale", [(64, 1.0), (129, 0.125), (512, 0.125), (513, 3.0), (1024, 1.0), (1025, 0.125), (2048, 3.0)])
def test_forward_with_resident_scores(N, scale, Hq, Hkv, D, alpha, causal, dtype):
    """Four waves to 512 keys, eight to 1024, sixteen to 2048.  The weights are multiplied as two 16-bit parts, so that the result's
    rounding is all that is lost, and at most as much again for thresholds and sums in fp32."""
    lengths = [N, 1, 31, N // 2 + 1]
    q, k, v, dout, varlen = problem(4, Hq, Hkv, N, D, dtype, scale, lengths)
    got = run(q, k, v, dout, varlen, alpha, causal, train=False)
    assert torch.equal(got[0], run(q, k, v, dout, varlen, alpha, causal, train=False)[0])
    check(got, q, k, v, dout, varlen, alpha, causal, list(range(4)))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,alpha,causal", [(64, 1.5, True), (128, 1.5, False), (64, 1.333, False), (128, 2.0, False)])
@pytest.mark.parametrize("N,length", [(1700, 1700), (2048, 2048), (2048, 2017), (2048, 1537)])
def test_forward_with_the_most_resident_scores(N, length, D, alpha, causal, dtype):
    """One head, at most 4096 blocks of 32 x 32 scores: sixteen waves with up to four blocks of keys each serve it at both head dims (D = 128
    and more than 1024 keys: up to 8000).  A training step's forward is the same."""
    q, k, v, dout, varlen = problem(1, 1, 1, N, D, dtype, 1.0, [length])
    got = run(q, k, v, dout, varlen, alpha, causal, train=False)
    assert torch.equal(got[0], run(q, k, v, dout, varlen, alpha, causal)[0])
    check(got, q, k, v, dout, varlen, alpha, causal, [0])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq,Hkv,D,alpha,causal", [(2, 1, 64, 1.5, True), (1, 1, 128, 1.5, False), (1, 1, 64, 1.125, False), (1, 1, 128, 2.0, False)])
@pytest.mark.parametrize("N,scale", [(97, 1.0), (256, 0.125), (257, 0.125), (577, 1.0), (1153, 3.0), (1300, 0.125), (2309, 0.125)])
def test_forward_on_all_pairs(no_supports, N, scale, Hq, Hkv, D, alpha, causal, dtype):
    """Rows that are all in the sample of 256 keys, just beyond it, and with a step on half of the tiles (from 1024 keys); without
    a gradient and, where the output walk corrects the threshold, with one."""
    lengths = [N, 1, 64, N // 2 + 1]
    q, k, v, dout, varlen = problem(4, Hq, Hkv, N, D, dtype, scale, lengths)
    for train in (False, True):
        check(run(q, k, v, dout, varlen, alpha, causal, train), q, k, v, dout, varlen, alpha, causal, list(range(4)))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("size", [40.0, 160.0])
def test_one_key_far_above_a_sampled_threshold(no_supports, size, D, dtype):
    """Key 200 is in none of the blocks that the first threshold is sampled from, but in the tiles of the step on half of them: its
    score, 25600 (D = 64) above in units of the threshold for size 160, to the power 8 and once more is beyond fp32."""
    q, k, v, dout, varlen = problem(1, 2, 2, 1152, D, dtype, 1.0, [1152])
    q[:], k[:, :, 200] = size, size
    check(run(q, k, v, dout, varlen, 1.125, False, train=False), q, k, v, dout, varlen, 1.125, False, [0])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("alpha", [1.5, 1.333])
@pytest.mark.parametrize("N", [1280, 4096])
def test_rows_whose_last_step_is_just_small_enough(no_supports, N, alpha, D, dtype):
    """The walks end for 128 rows together.  Here these are equal and every row block has a spread of its own, so the last steps lie all over
    the range that the rule allows, and a row's error is that of its own threshold, not a mean.  Bound, row by row: the weight's and the
    result's rounding, each at most a unit and half of that on average; what a step of x leaves, about x^2 relative to the weights (1.6e-3
    for bf16), joins them as a root of squares."""
    q, k, v, dout, varlen = problem(1, 8, 8, N, D, dtype, 1.0, [N])
    spread = torch.logspace(-1.5, 0.3, 8 * N // 128).reshape(1, 8, N // 128, 1, 1)
    q = (q.float().reshape(1, 8, N // 128, 128, D)[:, :, :, :1] * spread).expand(1, 8, N // 128, 128, D).reshape(q.shape).to(dtype)
    got = run(q, k, v, dout, varlen, alpha, False, train=False)[0].double().cpu()[:, :, ::128]
    want = exact.dense_entmax_attention(q[:, :, ::128], k, v, alpha, False, None).double()
    err = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert err.max() < 2 * UNIT[dtype], err.max()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("N", [300, 1100, 1792, 2309, 4096])
@pytest.mark.parametrize("scores", ["even", "exponential", "two clusters", "equal", "few values", "rising", "one far above"])
def test_thresholds_of_scores_that_are_not_normal(no_supports, scores, N, D, dtype):
    """The start and the steps go by a normal distribution and by densities: they may be far off without harm.  A row's scores are a distribution of its
    own times a spread of its own.  Bound on its error, row by row: the two roundings as above, and half of that again for what the last step may leave
    where the density misleads it (Newton's steps, which the kernel took before: up to 3.3e-2 for one key far above the others)."""
    g = torch.Generator().manual_seed(N)
    x = torch.rand(N, generator=g)
    x = {"even": x, "exponential": -x.clamp(min=1e-6).log(), "two clusters": (x < 0.1).float() + 0.05 * torch.randn(N, generator=g), "equal": torch.ones(N),
         "few values": (8 * x).floor() / 8, "rising": torch.arange(N) / N, "one far above": torch.where(torch.arange(N) == 200, 40.0, x)}[scores]
    q, k, v, dout, varlen = problem(1, 1, 1, N, D, dtype, 1.0, [N])
    q.zero_()
    q[0, 0, :, 0] = torch.logspace(-1, 2, N).to(dtype)
    k[0, 0, :, 0] = x.to(dtype)
    got = run(q, k, v, dout, varlen, 1.5, False, train=False)[0].double().cpu()
    rows = torch.arange(0, N, 7)
    want = exact.dense_entmax_attention(q[:, :, rows], k, v, 1.5, False, None).double()
    err = (got[:, :, rows] - want).norm(dim=-1) / want.norm(dim=-1)
    assert err.max() < 3 * UNIT[dtype], err.max()


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("N", [1100, 2048, 4096])
@pytest.mark.parametrize("values", [4, 7, 9, 15, 23, 39])
def test_thresholds_of_scores_of_few_values(no_supports, values, N, D):
    """Normal scores on a grid of 1 / values times three spreads: members come and go by hundreds, which the steps' densities do not expect.  Every row has a spread
    of its own.  Bound, row by row: the weight's and the result's rounding, 2^-11 each at most -- equal weights round alike --, on average half of that, and as a root of squares
    what is left of the threshold, sums off by 5e-4 and as much of the weights.  (f16: bf16's roundings alone reach 4.5e-3 here, as much as a wrong threshold.)"""
    dtype = torch.float16
    g = torch.Generator().manual_seed(values)
    x = (values * torch.randn(N, generator=g) / 3).round() / values
    q, k, v, dout, varlen = problem(1, 8, 8, N, D, dtype, 1.0, [N])
    q.zero_()
    k.zero_()
    spread = torch.logspace(-1.7, 0.3, 8 * N)  # of the scores times 1/2
    q[..., 0] = (spread * 2 * D ** 0.5 / x.std()).reshape(1, 8, N).to(dtype)
    k[..., 0] = x.to(dtype)
    got = run(q, k, v, dout, varlen, 1.5, False, train=False)[0].double().cpu()[:, :, ::37]
    want = exact.dense_entmax_attention(q[:, :, ::37], k, v, 1.5, False, None).double()
    err = (got - want).norm(dim=-1) / want.norm(dim=-1)
    assert err.max() < 2 * UNIT[dtype], err.max()


@pytest.mark.parametrize("scores", ["even", "rising"])
def test_scores_with_an_upper_end_take_no_longer_than_normal_ones(no_supports, scores):
    """Normal scores of spread 1/4 (about 70 members of 4096 keys) take about three walks over the keys in front of the output's, even ones of that spread (400 members)
    two at most.  A start above all keys, where a normal distribution would have its members, took six: 1.35 to 1.4 times as long as the normal ones.
    Bound: 1.15, for the clock's wandering."""
    N, H, D = 4096, 32, 64
    g = torch.Generator().manual_seed(3)
    times = {}
    for name in ("normal", scores):
        x = {"normal": torch.randn(1, H, N, D, generator=g), "even": torch.rand(1, H, N, D, generator=g), "rising": (torch.arange(N) / N)[:, None].expand(1, H, N, D)}[name]
        k = ((x - x.mean(2, keepdim=True)) / x.std(2, keepdim=True)).bfloat16().to(DEV)
        q = torch.nn.functional.one_hot(torch.arange(N) % D, D).expand(1, H, N, D).mul(0.25 / 0.5 * D ** 0.5).bfloat16().to(DEV)  # (z: half of the scaled score)
        v = torch.randn(1, H, N, D, generator=g).bfloat16().to(DEV)
        took = []
        for _ in range(8):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(4):
                A.adasplash_v1(q, k, v, alpha=1.5, is_causal=False, niter=10)
            end.record()
            end.synchronize()
            took.append(start.elapsed_time(end))
        times[name] = min(took)
    assert times[scores] < 1.15 * times["normal"], times


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("N", [300, 1100, 2309])
@pytest.mark.parametrize("scores", ["normal", "equal", "few values"])
def test_kept_thresholds_of_few_equal_and_many_members(no_supports, scores, N, D, dtype):
    """The threshold that a backward reads is a factor on all of a row's weights.  Rows of one member up to all keys; against 64 bits, relative to the mean of u:
    fp32 sums of N terms (N / 2 * 2^-24 at most) and what a last step leaves, 5e-3 at most, of which a step on the output walk's sums leaves the square."""
    g = torch.Generator().manual_seed(N)
    x = {"normal": torch.randn(N, generator=g), "equal": torch.ones(N), "few values": (8 * torch.rand(N, generator=g)).floor() / 8}[scores]
    q, k, v, _, _ = problem(1, 1, 1, N, D, dtype, 1.0, [N])
    q.zero_()
    q[0, 0, :, 0] = torch.logspace(-1, 2, N).to(dtype)
    k[0, 0, :, 0] = x.to(dtype)
    tau = _attention.launch_forward(q.to(DEV), k.to(DEV), v.to(DEV), version=1, alpha=1.5, is_causal=False, niter=10, varlen=None)[1][0, 0].double().cpu()
    rows = torch.arange(0, N, 3)
    _, p, want, _ = exact.dense_entmax_attention(q[:, :, rows], k, v, 1.5, False, None, return_aux=True)
    u = p[0, 0].double().sqrt()
    err = (tau[rows] - want[0, 0].double()).abs() / (u.sum(1) / (u > 0).sum(1))
    assert err.max() < N / 2 * 2.0 ** -24 + 2 * 5e-3 ** 2, err.max()


@pytest.mark.parametrize("alpha", [1.5, 1.333])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("key", [40, 300, 1030])
def test_tile_mask_has_no_marks_of_rows_behind_the_end(no_supports, key, D, alpha):
    """One key has all of the weight, and no first threshold's sample sees it.  The last row block has 76 rows, the others behind it
    are loaded as copies of the last one and take no part in the walks."""
    q, k = torch.zeros(1, 1, 1100, D), torch.zeros(1, 1, 1100, D)
    q[..., 0] = 1.0
    k[..., 0] = -64.0
    k[:, :, key, 0] = 0.0
    v = torch.randn(1, 1, 1100, D, generator=torch.Generator().manual_seed(1))
    q, k, v = (t.to(DEV, torch.bfloat16) for t in (q, k, v))
    bmask = _attention.launch_forward(q, k, v, version=1, alpha=alpha, is_causal=False, niter=10, varlen=None)[2].cpu()
    assert (bmask == 1 << (key // 64)).all(), bmask


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("far", [640, 1099])
def test_tile_mask_has_weights_too_small_for_the_sum(no_supports, far, D):
    """Key 0 has nearly all of the weight, key ``far`` 1e-8 of it: adding that changes nothing in fp32, but the key is a member."""
    q, k = torch.zeros(1, 1, 1100, D), torch.zeros(1, 1, 1100, D)
    root = D ** 0.5
    q[..., :2] = 1.0
    k[..., 0] = -64.0
    k[:, :, 0] = 0.0
    k[:, :, far, 0], k[:, :, far, 1] = -2 * root, 2e-4 * root if D == 64 else 0.0  # 1e-4 above the threshold (22.627 rounds to 22.625)
    v = torch.randn(1, 1, 1100, D, generator=torch.Generator().manual_seed(1))
    q, k, v = (t.to(DEV, torch.bfloat16) for t in (q, k, v))
    bmask = _attention.launch_forward(q, k, v, version=1, alpha=1.5, is_causal=False, niter=10, varlen=None)[2].cpu()
    want = torch.zeros_like(bmask)
    want[:] = 1 | 1 << (far // 64)  # (one word a row block)
    assert torch.equal(bmask, want)


@pytest.mark.parametrize("supports", [True, False])
@pytest.mark.parametrize("Hq,Hkv,D", [(2, 2, 64), (2, 1, 128)])
@pytest.mark.parametrize("dout_scale", [1e-2, 200.0, 300.0, 1000.0])
def test_f16_gradients_of_a_scaled_loss(request, dout_scale, Hq, Hkv, D, supports):
    """Upstream gradients as a loss scaler makes them: of a few hundred, u (dP - delta) is within f16's range only as long as u is
    at most 1 (it reaches some 2e4 for a spread of 1000).  The short route (dQ's weights in two parts), and the other one (one part)."""
    if not supports:
        request.getfixturevalue("no_supports")
    q, k, v, dout, varlen = problem(1, Hq, Hkv, 512, D, torch.float16, 1.0, [512])
    dout = (dout_scale * dout.float()).half()
    got = run(q, k, v, dout, varlen, 1.5, True)
    check(got, q, k, v, dout, varlen, 1.5, True, [0])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("spread", [0.5e-3, 1e-3, 2e-3, 4e-3])
@pytest.mark.parametrize("N,D,causal", [(512, 128, False), (1024, 64, True), (2048, 64, False), (2048, 128, False)])
def test_resident_scores_that_are_nearly_equal(N, D, causal, spread, dtype):
    """alpha = 2: a weight is about 1 / N here, and so is the border's place: a threshold off by a few 1e-4 loses some of the support."""
    q, k, v, dout, varlen = problem(1, 1, 1, N, D, dtype, spread ** 0.5, [N])
    k = (spread ** 0.5 * k.float()).to(dtype)
    got = run(q, k, v, dout, varlen, 2.0, causal, train=False)
    check(got, q, k, v, dout, varlen, 2.0, causal, [0])
    assert _lib.load().adsp_attn_bwd_reads_bmask(1, 1, 1, N, D, _lib.dtype_code(q), 2.0, int(causal)) == 0
    check(run(q, k, v, dout, varlen, 2.0, causal), q, k, v, dout, varlen, 2.0, causal, [0])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("spread", [1e-3, 2e-3, 4e-3])
@pytest.mark.parametrize("N,D,causal", [(512, 128, False), (1024, 64, True), (2048, 64, False), (2048, 128, False)])
@pytest.mark.parametrize("alpha", [1.9, 1.99])
def test_resident_scores_that_are_nearly_equal_close_to_two(alpha, N, D, causal, spread, dtype):
    """The same for a generic alpha, whose sum is nearly piecewise linear.  (dQ and dK have u^(2 - alpha) of the border's keys: its
    rounding in fp32 counts as at alpha = 2; they are not compared here.)"""
    q, k, v, dout, varlen = problem(1, 1, 1, N, D, dtype, spread ** 0.5, [N])
    k = (spread ** 0.5 * k.float()).to(dtype)
    check(run(q, k, v, dout, varlen, alpha, causal, train=False), q, k, v, dout, varlen, alpha, causal, [0])


def test_gradients_leave_out_what_a_causal_mask_hides(no_supports):
    """Rows of K and V that later queries alone see may be infinite for the earlier ones."""
    q, k, v, dout, varlen = problem(1, 2, 2, 160, 64, torch.bfloat16, 1.0, [160])
    want = run(q[:, :, :150], k[:, :, :150], v[:, :, :150], dout[:, :, :150], torch.tensor([150], dtype=torch.int32), 1.5, True)
    v[:, :, 150:] = float("inf")
    dq = run(q, k, v, dout, varlen, 1.5, True)[1]
    assert torch.isfinite(dq[:, :, :150]).all() and torch.equal(dq[:, :, :150], want[1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,scale", [(300, 1.0), (2309, 0.125)])
def test_an_alpha_that_is_two_in_single_precision(N, scale, dtype):
    """1 / (alpha - 1) rounds to 1 in fp32, and zero to the power of zero is no weight: the bits of alpha = 2."""
    q, k, v, dout, varlen = problem(1, 2, 2, N, 64, dtype, scale, [N - 3])
    want = run(q, k, v, dout, varlen, 2.0, False)
    got = run(q, k, v, dout, varlen, 2.0 - 1e-9, False)
    assert all(torch.isfinite(a).all() and torch.equal(a, w) for a, w in zip(got, want))
