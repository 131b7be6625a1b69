"""Launches of short segments whose workgroups compute several query blocks one after another: first loads of a block issued
while the one before it is still being written out.  What could go wrong there is a block that sees the state of another:
ring stages, seeds, reference points, the flag that asks for a second computation, the list of blocks itself.

Tolerance: as for the launch shapes - probabilities, values and outputs are rounded to 16 bits, at most 3 * 2^-9 of
sum_j p_j |v_j| < 2.5, 1e-2 with room; log-sum-exp 4e-3 from the rounded probabilities, and with the scale folded into a
16-bit q another 2^-9 |q| |k| / 8 = 1.6e-2 (heads of norm 8) that a row of one or two keys can show in full."""

import math
import random

import pytest
import torch

import oracle
from come_amd.common import RotaryPositionEmbedding2D, prepare_packed_self_attention_qkv
from come_amd.cuda_extension import flash_attn_varlen_qkvpacked_func_w_perkey_bias
from come_amd.cuda_extension.flash_attn import _forward

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _inputs(lens, H, seed):
    g = torch.Generator().manual_seed(seed)
    P = sum(lens)
    qkv = torch.randn(P, 3, H, 64, generator=g).bfloat16()
    bias = torch.where(torch.rand(P, generator=g) < 0.3, math.log(9.0), 0.0).bfloat16()
    return qkv, bias, torch.tensor([0] + lens).cumsum(0).to(torch.int32)


LSE = {"exact": 4e-3, "folded": 2e-2}


def _lens(n, seed):
    """Every remainder of a query block and of a key tile, empty and one-token segments among them."""
    rng = random.Random(seed)
    return [rng.choice([0, 1, 128, 129, 192, 193, 256, 257, 384, 385, 512]) if i % 5 == 0 else rng.randint(1, 700) for i in range(n)]


@pytest.mark.parametrize("mode", ["exact", "folded"])
@pytest.mark.parametrize("n,H", [(100, 16), (256, 7), (64, 16), (65, 24)])
def test_several_blocks_per_workgroup_against_the_oracle(n, H, mode):
    lens = _lens(n, n)
    qkv, bias, cu = _inputs(lens, H, n)
    ref, ref_lse = oracle.biased_varlen_attention(qkv, cu, bias)
    out, lse, _ = flash_attn_varlen_qkvpacked_func_w_perkey_bias(qkv.to(DEV), cu.to(DEV), max(lens), perkey_bias=bias.to(DEV),
                                                                 return_attn_probs=True, scale_mode=mode)
    torch.testing.assert_close(out.float().cpu(), ref, atol=1e-2, rtol=1e-2)
    torch.testing.assert_close(lse.cpu(), ref_lse, atol=LSE[mode], rtol=1e-3)


@pytest.mark.parametrize("mode", ["exact", "folded"])
def test_blocks_that_are_computed_again_between_others(mode):
    """Every third segment has a late key far above everything before it: the block is computed a second time, its
    neighbours in the same workgroup are not."""
    lens = [300 + 7 * i for i in range(50)]
    qkv, bias, cu = _inputs(lens, 16, 5)
    bounds = cu.tolist()
    for i, (s, e) in enumerate(zip(bounds[:-1], bounds[1:])):
        if i % 3 == 0:
            bias[s + (e - s) * 3 // 4] = 120.0
    ref, ref_lse = oracle.biased_varlen_attention(qkv, cu, bias)
    out, lse, _ = flash_attn_varlen_qkvpacked_func_w_perkey_bias(qkv.to(DEV), cu.to(DEV), max(lens), perkey_bias=bias.to(DEV),
                                                                 return_attn_probs=True, scale_mode=mode)
    torch.testing.assert_close(out.float().cpu(), ref, atol=1e-2, rtol=1e-2)
    torch.testing.assert_close(lse.cpu(), ref_lse, atol=LSE[mode], rtol=1e-3)


@pytest.mark.parametrize("heads", [51, 52])
def test_longest_list_of_a_workgroup_and_one_block_more(heads):
    """256 segments of 385 tokens: 51 heads stay below the length of a workgroup's list, 52 are launched block by block."""
    n, L = 256, 385
    g = torch.Generator(device=DEV).manual_seed(heads)
    qkv = torch.randn(n * L, 3, heads, 64, device=DEV, generator=g, dtype=torch.bfloat16)
    cu = torch.arange(n + 1, device=DEV, dtype=torch.int32) * L
    bias = torch.zeros(n * L, device=DEV, dtype=torch.bfloat16)
    out = flash_attn_varlen_qkvpacked_func_w_perkey_bias(qkv, cu, L, perkey_bias=bias).view(n, L, heads, 64)
    for head in range(0, heads, 10):
        q, k, v = (qkv.view(n, L, 3, heads, 64)[:, :, i, head].float() for i in range(3))
        ref = torch.bmm(torch.softmax(torch.bmm(q, k.transpose(1, 2).contiguous()) * 0.125, -1), v)
        torch.testing.assert_close(out[:, :, head].float(), ref, atol=1e-2, rtol=1e-2)


def test_block_reference_and_deferred_q_keep_their_bits():
    lens = [700 + 3 * i for i in range(30)]
    qkv, bias, cu = (t.to(DEV) for t in _inputs(lens, 16, 9))
    P = sum(lens)
    norm = torch.nn.LayerNorm(64, device=DEV, dtype=torch.bfloat16)
    rope = RotaryPositionEmbedding2D(100.0)
    pos = torch.randint(0, 38, (P, 2), device=DEV, generator=torch.Generator(device=DEV).manual_seed(1))
    with torch.no_grad():
        two = prepare_packed_self_attention_qkv(qkv.clone(), norm, norm, rope, pos, torch.bfloat16, max_position=37)
        one = prepare_packed_self_attention_qkv(qkv.clone(), norm, norm, rope, pos, torch.bfloat16, max_position=37, defer_q=True)
        a, b = (flash_attn_varlen_qkvpacked_func_w_perkey_bias(t, cu, max(lens), perkey_bias=bias) for t in (two, one))
        assert torch.equal(a, b)
        # one reference point per block: the bits of a segment are its own, alone in a launch or among others
        whole = _forward(two, cu, max(lens), bias, 0.0, 0.125, False, (-1, -1), 0.0, None, False, block_reference=True)[0]
        for i in (0, 13, 29):
            s, e = int(cu[i]), int(cu[i + 1])
            part = two[s:e].clone()
            part.come_qk_bound = two.come_qk_bound
            alone = _forward(part, cu[i:i + 2] - cu[i], e - s, bias[s:e].clone(), 0.0, 0.125, False, (-1, -1), 0.0, None, False,
                             block_reference=True)[0]
            assert torch.equal(whole[s:e], alone)
