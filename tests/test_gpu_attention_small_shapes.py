"""Attention launches of few or short segments on both sides of the sizes at which the workgroup shape changes (128-query
workgroups of two key groups with a CU each or sharing one, of four key groups, 256-query ones), with a ragged last block, a
last tile of one key and groups of keys that get no tile, against float64."""

import math

import pytest
import torch

from come_amd.cuda_extension.flash_attn import (flash_attn_varlen_qkvpacked_func,
                                                flash_attn_varlen_qkvpacked_func_w_perkey_bias)

pytestmark = pytest.mark.gpu


def _reference(qkv, lengths, bias, scale):
    out, at = [], 0
    for n in lengths:
        q, k, v = qkv[at:at + n].double().permute(1, 2, 0, 3)
        s = (q @ k.transpose(1, 2)) * scale + bias[at:at + n].double()
        out.append((s.softmax(-1) @ v).transpose(0, 1))
        at += n
    return torch.cat(out)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("heads,lengths", [
    (16, [1]), (16, [64]), (16, [65]), (16, [128, 129]), (16, [383, 385]),           # one or two tiles, the second group empty
    (16, [766]), (16, [2048]), (16, [2049]),                                         # 256 workgroups, and 16 more
    (6, [1792]), (6, [1793]), (6, [2500]),                                           # 28 tiles, 29: four key groups
    (16, [640] * 3), (16, [513] * 3), (16, [705] * 3), (16, [900, 1000]),            # nearly every CU taken, short and long
    (16, [640] * 6), (16, [766] * 3),                                                # 480 workgroups; 288, or 144 of 256 queries
], ids=lambda v: str(v) if isinstance(v, int) else f"{len(v)}x{v[0]}")
def test_shapes(heads, lengths, dtype):
    g = torch.Generator().manual_seed(sum(lengths) + heads)
    total = sum(lengths)
    qkv = torch.randn(total, 3, heads, 64, generator=g).to(dtype)
    bias = torch.where(torch.rand(total, generator=g) < 0.1, 9.0, 1.0).log().to(dtype)
    cu = torch.tensor([0] + lengths).cumsum(0).to(torch.int32).cuda()
    got = flash_attn_varlen_qkvpacked_func_w_perkey_bias(qkv.cuda(), cu, max(lengths), perkey_bias=bias.cuda(), softmax_scale=0.125)
    want = _reference(qkv.cuda(), lengths, bias.cuda(), 0.125)
    # probabilities and the output are rounded to 16 bits: each by a relative 2^-9 (bf16, nearest), the probabilities of fp16 by
    # up to 2^-10 (truncated); an output is a mean of values whose absolute weighted mean bounds what the first rounding moves
    eps = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -10
    size = _reference(torch.cat((qkv[:, :2], qkv[:, 2:].abs()), 1).cuda(), lengths, bias.cuda(), 0.125)
    assert ((got.double() - want).abs() <= 2.5 * eps * size + eps * want.abs() + 1e-6).all()


@pytest.mark.parametrize("mode", ["exact", "folded"])
@pytest.mark.parametrize("rows", [0, 32, None], ids=["first_tile", "second_tile", "all"])
@pytest.mark.parametrize("keys", [(16, 700), (6, 2100), (16, 4200)], ids=lambda v: str(v[1]))
def test_row_sums_leave_their_range_at_every_place_of_a_tile(keys, rows, mode):
    """One key a head whose score stands 48 nats (2^69) above the others, at another place of its key tile in every head,
    seen by the first or the second 32 of every 64 queries or by all: the row sums are looked at once per tile of 64 keys, and
    the reference point moves in the slot behind."""
    from come_amd.cuda_extension.flash_attn import _forward

    heads, n = keys
    g = torch.Generator().manual_seed(n)
    qkv = torch.randn(n, 3, heads, 64, generator=g)
    qkv[:, :2, :, 63] = 0.0
    for h in range(heads):
        qkv[n // 2 + 9 * h, 1, h, 63] = 384.0                  # 48 nats at a scale of 1/8
    sees = torch.ones(n, dtype=torch.bool) if rows is None else (torch.arange(n) % 64) // 32 == rows // 32
    qkv[:, 0, :, 63] = sees.float()[:, None]
    qkv = qkv.bfloat16().cuda()
    bias = torch.zeros(n, dtype=torch.bfloat16, device="cuda")
    cu = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    got = _forward(qkv, cu, n, bias, 0.0, 0.125, False, (-1, -1), 0.0, None, False, scale_mode=mode)[0]
    want = _reference(qkv, [n], bias, 0.125)
    eps = 2.0 ** -9
    size = _reference(torch.cat((qkv[:, :2], qkv[:, 2:].abs()), 1), [n], bias, 0.125)
    # folded: the 16-bit q moves a logit by up to 2^-9 of the sum of its products' sizes, here at most 7 nats without the one key
    # that stands above (whose row then holds nothing but that key's value)
    moved = 2.0 ** -9 * 7 if mode == "folded" else 0.0
    assert ((got.double() - want).abs() <= (2.5 * eps + 2 * moved) * size + eps * want.abs() + 1e-6).all()


@pytest.mark.parametrize("below", [1.0, 3.0, 5.0, 7.0, 9.0, 11.0])
@pytest.mark.parametrize("heads,n", [(16, 766), (6, 2100), (16, 1374), (2, 5000)])
def test_first_keys_below_the_others_in_fp16(heads, n, below):
    """The first 70 keys, which the reference points are taken from, stand 1 - 11 nats below the others: row sums of fp16
    probabilities that just stay within the room above the reference point, leave it, and leave the type."""
    g = torch.Generator().manual_seed(n)
    qkv = torch.randn(n, 3, heads, 64, generator=g).half().cuda()
    bias = torch.zeros(n)
    bias[:70] = -below
    bias = bias.half().cuda()
    cu = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    got = flash_attn_varlen_qkvpacked_func_w_perkey_bias(qkv, cu, n, perkey_bias=bias, softmax_scale=0.125)
    want = _reference(qkv, [n], bias, 0.125)
    size = _reference(torch.cat((qkv[:, :2], qkv[:, 2:].abs()), 1), [n], bias, 0.125)
    eps = 2.0 ** -10
    assert ((got.double() - want).abs() <= 2.5 * eps * size + eps * want.abs() + 1e-6).all()


@pytest.mark.parametrize("above", [6.0, 8.0, 9.0, 10.0, 11.0, 12.0])
@pytest.mark.parametrize("heads,n", [(16, 1600), (6, 2100), (16, 6000)])
def test_first_keys_above_the_others_in_fp16(heads, n, above):
    """Five keys at the head of the segment stand 6 - 12 nats above the others, which share what is left of the attention: their
    probabilities are small beside those that the reference points are taken from.  The first keys' values are zero and the
    others' the same in every row, so that what truncation takes from the small probabilities adds up in the outputs."""
    g = torch.Generator().manual_seed(n)
    qkv = torch.randn(n, 3, heads, 64, generator=g)
    value = (qkv[0, 2].sign() * (0.5 + torch.rand(heads, 64, generator=g))).half()
    qkv[:, 2] = value
    qkv[:5, 2] = 0.0
    qkv = qkv.half().cuda()
    bias = torch.zeros(n)
    bias[:5] = above
    bias = bias.half().cuda()
    cu = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    got = flash_attn_varlen_qkvpacked_func_w_perkey_bias(qkv, cu, n, perkey_bias=bias, softmax_scale=0.125)
    for h in range(heads):
        q, k = qkv[:, 0, h].double(), qkv[:, 1, h].double()
        s = (q @ k.T) * 0.125 + bias.double()
        w = (s - s[:, :32].amax(1, keepdim=True)).exp()
        share = w[:, 5:].sum(1) / w.sum(1)
        # A probability is stored truncated, at no less than half its size relative to the largest of the first 32 keys: it loses
        # up to a relative 2^-10, or 2^-24 where it is subnormal, 2^-23 of the largest.  What the others lose is missing from the
        # share, what the first five lose from the rest; the second order and the sums in fp32 are within a twentieth, the scores
        # in fp32 within 2^-16.
        lost = (w * 2.0 ** -10).clamp_min(2.0 ** -23)
        moved = 1.05 * (lost[:, 5:].sum(1) * (1 - share) + lost[:, :5].sum(1) * share) / w.sum(1)
        c = value[h].double().cuda()
        want = share[:, None] * c
        bound = (moved + share * (2.0 ** -11 + 2.0 ** -16))[:, None] * c.abs() + 2.0 ** -25
        assert ((got[:, h].double() - want).abs() <= bound).all()


@pytest.mark.parametrize("heads,n", [(2, 32768), (16, 17000)])
def test_reference_points_at_zero_in_fp16(heads, n):
    """Scores that are multiples of 1/64 in log2 units, all moved by a whole number: every sum and difference on the way to the
    probabilities is exact, so the outputs are the same bits - also where a row's reference point comes out at zero."""
    g = torch.Generator().manual_seed(n)
    qkv = torch.zeros(n, 3, heads, 64)
    qkv[:, :2, :, :8] = torch.randint(-4, 5, (n, 2, heads, 8), generator=g) / 8
    qkv[:, 2] = torch.randn(n, heads, 64, generator=g)
    qkv[:, 0, :, 61:] = 1.0
    qkv[0, 1] = 0.0
    qkv[0, 1, :, 62] = -0.75                                     # one key near zero, the others about 2^-16 of it
    qkv[1:, 1, :, 61] = -16.75
    cu = torch.tensor([0, n], dtype=torch.int32, device="cuda")
    outs = []
    for moved in (1, 0, -1, -2, 3):
        qkv[:, 1, :, 63] = moved
        # (the float nearest to ln 2: one unit of a score is one binary order)
        outs.append(flash_attn_varlen_qkvpacked_func(qkv.half().cuda(), cu, n, softmax_scale=math.log(2.0)))
    for o in outs[1:]:
        assert torch.equal(outs[0], o)
