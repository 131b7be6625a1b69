"""Blocks of 512 and 256 queries in 16 x 16 tiles: last tiles and last blocks of every size, logits whose row sums leave the range the
16-bit probabilities keep, and keys that beat everything before them, against the closed form in 64 bits on sampled rows."""

import pytest
import torch

from come_amd import _lib
from come_amd.cuda_extension import flash_attn_varlen_qkvpacked_func, flash_attn_varlen_qkvpacked_func_w_perkey_bias
from come_amd.cuda_extension.flash_attn import flash_attn_fwd_cuda

pytestmark = pytest.mark.gpu
DEV = "cuda"
HEADS = 16                                           # x 16 blocks of 512 queries = 256 workgroups of 8 wavefronts
BF16, F16 = torch.bfloat16, torch.float16
# relative 2-norm of the error: probabilities are rounded to the 16-bit type (bf16 to nearest, 2^-9; fp16 toward zero, 2^-10), outputs
# to nearest (2^-9, 2^-11); folded, q is rounded once more, which moves a logit by 2^-9 of its size: below 1 for unit vectors
BOUND = {(BF16, "exact"): 2 ** -8, (BF16, "folded"): 1.5 * 2 ** -8, (F16, "exact"): 1.5 * 2 ** -10}
MODES = [(BF16, "exact"), (BF16, "folded"), (F16, "exact")]


def check(qkv, bias, mode, lengths, bound):
    cu = torch.tensor([0] + lengths, device=DEV).cumsum(0).to(torch.int32)
    kw = dict(softmax_scale=0.125, return_attn_probs=True, scale_mode=mode)
    if bias is None:
        out, lse, _ = flash_attn_varlen_qkvpacked_func(qkv, cu, max(lengths), **kw)
        bias = qkv.new_zeros(sum(lengths))
    else:
        out, lse, _ = flash_attn_varlen_qkvpacked_func_w_perkey_bias(qkv, cu, max(lengths), perkey_bias=bias, **kw)
    assert bool(torch.isfinite(out).all()) and bool(torch.isfinite(lse).all())
    start = 0
    for L in lengths:
        rows = sorted({*range(0, min(L, 40)), *range(max(L - 70, 0), L), *range(17, L, 509)})
        at = torch.as_tensor(rows, device=DEV)
        q, k, v = (qkv[start:start + L, i].double().transpose(0, 1).contiguous() for i in range(3))
        scores = torch.matmul(q[:, at], k.transpose(1, 2).contiguous()) * 0.125 + bias[start:start + L].double()
        ref = torch.matmul(torch.softmax(scores, -1), v).transpose(0, 1)
        err = (out[start + at].double() - ref).norm() / ref.norm()
        assert float(err) <= bound, float(err)
        torch.testing.assert_close(lse[:, start + at].double(), torch.logsumexp(scores, -1), atol=2e-3, rtol=1e-3)
        start += L


def inputs(total, dtype, heads=HEADS):
    g = torch.Generator(device=DEV).manual_seed(total)
    qkv = torch.randn(total, 3, heads, 64, generator=g, device=DEV)
    qkv[:, :2] /= qkv[:, :2].square().mean(-1, keepdim=True).sqrt()            # as out of a LayerNorm
    bias = torch.where(torch.rand(total, generator=g, device=DEV) < 0.1, 9.0, 1.0).log().to(dtype)
    return qkv.to(dtype), bias


@pytest.mark.parametrize("dtype,mode", MODES, ids=str)
@pytest.mark.parametrize("L", [7681, 7697, 7712, 7713, 7743, 7744, 7745, 8128, 8191, 8192])
def test_last_tiles(L, dtype, mode):
    qkv, bias = inputs(L, dtype)
    check(qkv, bias, mode, [L], BOUND[dtype, mode])


@pytest.mark.parametrize("dtype,mode", MODES, ids=str)
@pytest.mark.parametrize("lengths", [[14000], [5200, 4600, 300]], ids=str)
def test_pieces(lengths, dtype, mode):
    heads = 12
    assert _lib.load().come_attn_work_bytes(len(lengths), sum(lengths), heads, max(lengths)) > 0
    qkv, bias = inputs(sum(lengths), dtype, heads)
    check(qkv, bias, mode, lengths, BOUND[dtype, mode])


# launches of more than two workgroups of 4 wavefronts per CU, none of whose segments is long enough for 8
@pytest.mark.parametrize("dtype,mode", MODES, ids=str)
@pytest.mark.parametrize("lengths", [[2177, 2208, 2209, 2303, 2304], [3840, 2431, 2369, 257, 2400]], ids=str)
def test_four_wavefronts(lengths, dtype, mode):
    qkv, bias = inputs(sum(lengths), dtype)
    check(qkv, bias, mode, lengths, BOUND[dtype, mode])


@pytest.mark.parametrize("lengths", [[801, 1374, 97, 640, 1000, 1, 512, 129, 1200, 1311, 1290, 258]], ids=str)
def test_four_wavefronts_short(lengths):
    qkv, bias = inputs(sum(lengths), F16)
    check(qkv, bias, "exact", lengths, BOUND[F16, "exact"])


# exact: logits that climb by `climb` nats over the segment, a last bit of the row sums at a time, and one key `jump` nats above all
# before it.  q . k of the ramp is exact (one component each), so the bound holds as for unit vectors.
@pytest.mark.parametrize("dtype", [BF16, F16], ids=str)
@pytest.mark.parametrize("climb,jump", [(60, 0), (0, 12), (0, 100), (60, 100)], ids=str)
@pytest.mark.parametrize("lengths", [[7713], [2177, 2208, 2209, 2303, 2304]], ids=["512", "256"])
def test_reference_points(lengths, climb, jump, dtype):
    qkv, bias = inputs(sum(lengths), dtype)
    qkv[:, 0, :, 0] = 16.0
    start = 0
    for L in lengths:
        ramp = torch.arange(L, device=DEV) * (climb / L / 2)
        if jump:
            ramp[L // 2 + 5] += (climb + jump) / 2
        qkv[start:start + L, 1, :, 0] = ramp.to(dtype)[:, None]
        start += L
    check(qkv, bias, "exact", lengths, BOUND[dtype, "exact"])


@pytest.mark.parametrize("dtype,mode", MODES, ids=str)
def test_first_keys_masked(dtype, mode):
    L = 7713
    qkv, bias = inputs(L, dtype)
    bias[:40] = float("-inf")
    check(qkv, bias, mode, [L], BOUND[dtype, mode])


WIDE, NARROW = [7713], [2177, 2208, 2209, 2303, 2304]           # launches of 512 and of 256 queries a workgroup


# Row sums that leave the range in the middle of the key loop, in every arithmetic; the bias carries them, whose values here are exact in 16
# bits.  rising: the reference points move every few half-tiles; step: once, by 40 nats; late: one key 120 nats above the rest,
# beyond what a move can follow; low: all scores 100 nats below the reference point of the folded arithmetic.
@pytest.mark.parametrize("dtype,mode", MODES, ids=str)
@pytest.mark.parametrize("kind", ["rising", "step", "late", "low"])
@pytest.mark.parametrize("lengths", [WIDE, NARROW], ids=["512", "256"])
def test_reference_points_of_the_bias(lengths, kind, dtype, mode):
    qkv, bias = inputs(sum(lengths), dtype)
    start = 0
    for L in lengths:
        own = bias[start:start + L]
        if kind == "rising":
            own[:] = (torch.arange(L, device=DEV) // 32 * 4).to(dtype)
        elif kind == "step":
            own[L // 2 + 5:] = 40.0
        elif kind == "late":
            own[L // 2 + 5] = 120.0
        else:
            own[:] = -100.0
        start += L
    check(qkv, bias, mode, lengths, BOUND[dtype, mode])


# what is masked: a row's first keys, whole tiles and half-tiles in the middle, all but one key in sixteen
MASKED = {"first-40": [(0, 40)], "tiles": [(64, 256), (1024, 1056), (1120, 1152), (2048, 2170)], "most": [(16 * t + 1, 16 * t + 16) for t in range(482)]}


@pytest.mark.parametrize("dtype,mode", MODES, ids=str)
@pytest.mark.parametrize("masked", MASKED)
@pytest.mark.parametrize("lengths", [WIDE, NARROW], ids=["512", "256"])
def test_masked_keys(lengths, masked, dtype, mode):
    qkv, bias = inputs(sum(lengths), dtype)
    start = 0
    for L in lengths:
        for first, last in MASKED[masked]:
            bias[start + first:start + min(last, L)] = float("-inf")
        start += L
    check(qkv, bias, mode, lengths, BOUND[dtype, mode])


@pytest.mark.parametrize("dtype,mode", MODES, ids=str)
@pytest.mark.parametrize("lengths", [WIDE, NARROW], ids=["512", "256"])
def test_without_bias(lengths, dtype, mode):
    check(inputs(sum(lengths), dtype)[0], None, mode, lengths, BOUND[dtype, mode])


@pytest.mark.parametrize("dtype,mode", MODES, ids=str)
@pytest.mark.parametrize("with_bias", [True, False], ids=["bias", "plain"])
@pytest.mark.parametrize("lengths", [WIDE, NARROW], ids=["512", "256"])
def test_strides(lengths, with_bias, dtype, mode):
    """q, k and v of strides of their own, an output that allows 8-byte stores only: the bits of the packed call, and nothing beside them."""
    total = sum(lengths)
    qkv, bias = inputs(total, dtype)
    cu = torch.tensor([0] + lengths, device=DEV).cumsum(0).to(torch.int32)

    def call(q, k, v, out):
        tail = (max(lengths), max(lengths), 0.0, 0.125, False, False, -1, -1, 0.0, False, None)
        if with_bias:
            return flash_attn_fwd_cuda.varlen_fwd_w_perkey_bias(q, k, v, out, cu, cu, None, None, None, None, bias, *tail, fold_scale=mode == "folded")[0]
        return flash_attn_fwd_cuda.varlen_fwd(q, k, v, out, cu, cu, None, None, None, None, *tail, fold_scale=mode == "folded")[0]

    want = call(*qkv.unbind(1), None)
    own = []
    for t, pad in zip(qkv.unbind(1), (0, 8, 24)):
        wide = torch.zeros(total, HEADS, 64 + pad, dtype=dtype, device=DEV)
        wide[:, :, :64] = t
        own.append(wide[:, :, :64])
    own[0] = own[0].transpose(0, 1).contiguous().transpose(0, 1)                 # heads first
    wide = torch.full((total, HEADS, 68), 7.0, dtype=dtype, device=DEV)
    out = call(*own, wide[:, :, 4:])
    assert out.data_ptr() == wide.data_ptr() + 8
    assert torch.equal(out, want)
    assert bool((wide[:, :, :4] == 7.0).all())


# A row's bits do not depend on the pipeline that the size of a launch asks for: 16 heads of 7900 keys (512 queries a workgroup) against 6 of them
# at a time, three segments of about 3000 keys (256 queries) against each of them alone, which run in 32 x 32 tiles with one key group (the last
# block of every segment has more than 128 queries: fewer would run as two key groups).
@pytest.mark.parametrize("masked", [False, True], ids=["all", "masked"])
@pytest.mark.parametrize("dtype,mode", MODES, ids=str)
@pytest.mark.parametrize("lengths", [[7900], [3000, 2950, 2990]], ids=["512", "256"])
def test_same_bits_as_32x32_tiles(lengths, dtype, mode, masked):
    qkv, bias = inputs(sum(lengths), dtype)
    if masked:
        bias[20:50] = bias[1024:1100] = float("-inf")

    def call(qkv, bias, lengths):
        cu = torch.tensor([0] + lengths, device=DEV).cumsum(0).to(torch.int32)
        return flash_attn_varlen_qkvpacked_func_w_perkey_bias(qkv, cu, max(lengths), perkey_bias=bias, softmax_scale=0.125, return_attn_probs=True, scale_mode=mode)[:2]

    out, lse = call(qkv, bias, lengths)
    if len(lengths) == 1:
        parts = [(slice(None), slice(h, h + 6)) for h in (0, 6, HEADS - 6)]
    else:
        parts = [(slice(sum(lengths[:i]), sum(lengths[:i + 1])), slice(None)) for i in range(len(lengths))]
    for rows, heads in parts:
        own = bias[rows]
        got, got_lse = call(qkv[rows, :, heads].contiguous(), own, [own.shape[0]])
        assert torch.equal(out[rows, heads], got)
        assert torch.equal(lse[heads, rows], got_lse)
