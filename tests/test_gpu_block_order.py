"""GPU test of the dense kernels' block numbering (xcd_block_map in csrc/common.h): the workgroups of a launch are dealt
to (K/V head, block, member of the group) by a rule that depends on the number of heads, of blocks per head and on
the mask.  Whatever the rule, a batch must give what its items give one by one: a block that the numbering left out,
or dealt to the wrong place, shows as a row block that differs."""

import os

import pytest
import torch

from adasplash_amd import _attention
from tests.gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.fixture
def dense_only():
    old = os.environ.get("ADSP_SPARSE")
    os.environ["ADSP_SPARSE"] = "0"
    yield
    if old is None:
        os.environ.pop("ADSP_SPARSE", None)
    else:
        os.environ["ADSP_SPARSE"] = old


# (B, Hq, Hkv, N, D, causal): heads per XCD 1, 2, 3 and a count that is no multiple of 8; sets of several heads, of
# one head, and a last set that is smaller than the others (24 heads of 128 blocks: sets of two, three per XCD)
CASES = [
    (1, 8, 8, 512, 64, True),
    (2, 8, 8, 1024, 64, True),
    (3, 8, 8, 256, 64, True),
    (3, 32, 8, 4096, 64, True),
    (1, 6, 3, 512, 64, True),
    (2, 16, 8, 2048, 128, True),
    (2, 8, 8, 1024, 64, False),
]


@pytest.mark.parametrize("B,Hq,Hkv,N,D,causal", CASES)
def test_a_batch_equals_its_items_forward_and_backward(dense_only, B, Hq, Hkv, N, D, causal):
    g = torch.Generator().manual_seed(B * 1000 + N + D)
    q = torch.randn(B, Hq, N, D, generator=g).bfloat16().to(DEV)
    k = torch.randn(B, Hkv, N, D, generator=g).bfloat16().to(DEV)
    v = torch.randn(B, Hkv, N, D, generator=g).bfloat16().to(DEV)
    dout = torch.randn(B, Hq, N, D, generator=g).bfloat16().to(DEV)
    version, alpha = (2, 1.5) if causal else (1, 1.5)

    def run(qq, kk, vv, dd):
        out, taus, bmask = _attention.launch_forward(qq, kk, vv, version=version, alpha=alpha, is_causal=causal, niter=2, varlen=None)
        dq, dk, dv = _attention.launch_backward(qq, kk, vv, dd, taus, bmask, alpha=alpha, is_causal=causal, varlen=None)[:3]
        return out, taus, dq, dk, dv

    whole = run(q, k, v, dout)
    for b in range(B):
        one = run(q[b:b + 1].contiguous(), k[b:b + 1].contiguous(), v[b:b + 1].contiguous(), dout[b:b + 1].contiguous())
        for name, w, o in zip(("out", "taus", "dq", "dk", "dv"), whole, one):
            assert torch.equal(w[b], o[0]), f"{name}: batch item {b} differs from the item run alone"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,Hq,Hkv,N,D,causal", [(2, 8, 8, 1024, 64, True), (5, 8, 8, 200, 64, True), (4, 16, 8, 520, 128, True), (3, 8, 8, 1000, 64, False)])
def test_a_padded_batch_equals_its_items(dense_only, B, Hq, Hkv, N, D, causal, dtype):
    """The same where the batch has lengths: the heads of a set then change places from round to round (sets of one, two, four and five heads)."""
    g = torch.Generator().manual_seed(B * 1000 + N + D)
    q, dout = (torch.randn(B, Hq, N, D, generator=g).to(DEV, dtype) for _ in range(2))
    k, v = (torch.randn(B, Hkv, N, D, generator=g).to(DEV, dtype) for _ in range(2))
    lens = torch.tensor([N - b * N // 5 for b in range(B)], dtype=torch.int32, device=DEV)

    def run(b):
        qq, kk, vv, dd, ll = (t[b].contiguous() for t in (q, k, v, dout, lens))
        out, taus, bmask = _attention.launch_forward(qq, kk, vv, version=2 if causal else 1, alpha=1.5, is_causal=causal, niter=2, varlen=ll)
        return out, *_attention.launch_backward(qq, kk, vv, dd, taus, bmask, alpha=1.5, is_causal=causal, varlen=ll)[:3]

    whole = run(slice(0, B))
    for b in range(B):
        for name, w, o in zip(("out", "dq", "dk", "dv"), whole, run(slice(b, b + 1))):
            assert torch.equal(w[b], o[0]), f"{name}: batch item {b} differs from the item run alone"


# not causal, with lengths: the kernels on all pairs take the items longest first (equal lengths, a length of 0, 64 items, and 65, whose order stays), every
# second round over the XCDs backwards (rounds of eight items, four, two and one; a last round that is whole and one that is not), and keep their order in launches
# of many workgroups (20 x 24 heads and 30 x 24, on both sides of the line for the fp32 gradients)
@pytest.mark.parametrize("lens,H,N", [([70, 200, 200, 0, 129, 1], 3, 200), ([70, 200, 33, 0, 129, 1, 64], 4, 200), ([70, 200, 33, 0, 129, 1, 64, 150], 6, 200), ([70, 150, 33, 20], 8, 150),
                                      ([1 + 37 * i % 61 for i in range(20)], 24, 64), ([1 + 37 * i % 61 for i in range(30)], 24, 64),
                                      ([1 + 37 * i % 61 for i in range(19)], 1, 64), ([1 + 37 * i % 61 for i in range(64)], 1, 64), ([1 + 37 * i % 61 for i in range(65)], 1, 64)])
@pytest.mark.parametrize("bits,dtype", [(torch.int32, torch.bfloat16), (torch.int64, torch.bfloat16), (torch.int32, torch.float32)])
def test_items_of_a_padded_batch_longest_first(dense_only, lens, H, N, bits, dtype):
    g = torch.Generator().manual_seed(len(lens))
    B = len(lens)
    q, k, v, dout = (torch.randn(B, H, N, 64, generator=g).to(dtype).to(DEV) for _ in range(4))
    varlen = torch.tensor(lens, dtype=bits, device=DEV)

    def run(rows):
        a = [t[rows].contiguous() for t in (q, k, v, dout)]
        out, taus, bmask = _attention.launch_forward(*a[:3], version=1, alpha=1.5, is_causal=False, niter=4, varlen=varlen[rows].contiguous())
        return out, *_attention.launch_backward(*a, taus, bmask, alpha=1.5, is_causal=False, varlen=varlen[rows].contiguous())[:3]

    whole = run(slice(None))
    for b in range(0, B, 1 if B < 10 else 7):
        for name, w, o in zip(("out", "dq", "dk", "dv"), whole, run(slice(b, b + 1))):
            assert torch.equal(w[b], o[0]), f"{name}: batch item {b} differs from the item run alone"


# at most one row block per workgroup of the kernels on the supports, two or three heads per XCD, a last round over the CUs that is not full
@pytest.mark.parametrize("B,Hq,Hkv,N,D", [(2, 8, 8, 1024, 64), (3, 8, 8, 2048, 64), (2, 16, 8, 2048, 128)])
def test_a_batch_equals_its_items_on_the_supports(B, Hq, Hkv, N, D):
    g = torch.Generator().manual_seed(B + N)
    q, dout = (torch.randn(B, Hq, N, D, generator=g).bfloat16().to(DEV) for _ in range(2))
    k, v = (torch.randn(B, Hkv, N, D, generator=g).bfloat16().to(DEV) for _ in range(2))

    def run(rows):
        a = [t[rows].contiguous() for t in (q, k, v, dout)]
        out, taus, bmask = _attention.launch_forward(*a[:3], version=2, alpha=1.5, is_causal=True, niter=2, varlen=None)
        return out, taus, *_attention.launch_backward(*a, taus, bmask, alpha=1.5, is_causal=True, varlen=None)[:3]

    whole = run(slice(None))
    for b in range(B):
        for name, w, o in zip(("out", "taus", "dq", "dk", "dv"), whole, run(slice(b, b + 1))):
            assert torch.equal(w[b], o[0]), f"{name}: batch item {b} differs from the item run alone"


# fp32, causal: blocks longest first over an XCD's heads, against heads run alone, which take the general order (one and eight heads per XCD, 64 blocks, 64
# blocks that are not empty and more, lengths of 0, a part of a block and equal ones; without lengths, where N is a power of two: launches that are
# under way at once, and longer ones that the general order divides evenly and does not)
LENGTHS_CAUSAL = [([70, 200, 0], 16, 8, 200, 64), ([2048], 8, 8, 2048, 64), ([1024, 1024], 8, 8, 1024, 64), ([33, 1, 300, 300], 16, 16, 300, 64), ([700, 64, 511], 16, 8, 700, 128)]
WHOLE_CAUSAL = [([2048], 8, 8, 2048, 64), ([1024, 1024], 8, 8, 1024, 64), ([512] * 8, 32, 8, 512, 64), ([1024] * 8, 8, 8, 1024, 64), ([2048] * 6, 8, 8, 2048, 64)]


@pytest.mark.parametrize("bits,lens,Hq,Hkv,N,D", [(bits, *c) for bits in (torch.int32, torch.int64) for c in LENGTHS_CAUSAL] + [(None, *c) for c in WHOLE_CAUSAL])
def test_causal_blocks_longest_first(bits, lens, Hq, Hkv, N, D):
    g = torch.Generator().manual_seed(N)
    B, group = len(lens), Hq // Hkv
    q, dout = (torch.randn(B, Hq, N, D, generator=g).to(DEV) for _ in range(2))
    k, v = (torch.randn(B, Hkv, N, D, generator=g).to(DEV) for _ in range(2))
    varlen = None if bits is None else torch.tensor(lens, dtype=bits, device=DEV)

    def run(rows, heads):
        qh = slice(heads.start * group, heads.stop * group)
        a = [t[rows, h].contiguous() for t, h in ((q, qh), (k, heads), (v, heads), (dout, qh))]
        vl = None if varlen is None else varlen[rows].contiguous()
        out, taus, bmask = _attention.launch_forward(*a[:3], version=2, alpha=1.5, is_causal=True, niter=2, varlen=vl)
        return out, *_attention.launch_backward(*a, taus, bmask, alpha=1.5, is_causal=True, varlen=vl)[:3]

    whole = run(slice(None), slice(0, Hkv))
    for b in range(B):
        for h in (0, Hkv // 2, Hkv - 1):
            for name, w, o in zip(("out", "dq", "dk", "dv"), whole, run(slice(b, b + 1), slice(h, h + 1))):
                n = o.shape[1]
                assert torch.equal(w[b, h * n:(h + 1) * n], o[0]), f"{name}: item {b}, head {h}"
