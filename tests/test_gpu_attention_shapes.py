"""The launch shapes of the 64-wide varlen attention at the sizes where they can go wrong: every remainder of a query
block (64, 128 and 256 queries are the steps of the shapes) and of a key group's share of the tiles, segment counts on
both sides of a wavefront (64) and of the compact grid (256), reference points that move while several key groups work
on one block, rows whose sums leave the range from below.

Tolerance: probabilities, values and outputs are rounded to the 16-bit type, so a row is off by at most
3 * 2^-9 (bf16; fp16 3 * 2^-12) of sum_j p_j |v_j|; inputs are |v| < 5, the sums far below 2.5 for all but rows of a
single key, where the output is v itself: 3 * 2^-9 * 2.5 < 1.5e-2 and, single keys being exact, 1e-2 holds throughout.
The log-sum-exp sees the row sum of rounded probabilities: 2^-9 relative, 4e-3 absolute."""

import math

import pytest
import torch

import oracle
from come_amd.cuda_extension import flash_attn_varlen_qkvpacked_func_w_perkey_bias

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = {
    # 128-query blocks, 2 x 2 wavefronts: every remainder of the query tiles, one key tile or an odd number of them
    "edges": ([1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 383, 384, 385, 0], 3),
    "tiles": ([32, 33, 95, 96, 97, 160, 161, 321, 449], 2),
    # 128-query blocks, 2 x 4 wavefronts: from one key tile in every group to groups of unequal shares
    "four-groups": ([1000], 2), "four-groups-unequal": ([1601], 16), "four-groups-few-keys": ([700, 3, 1100], 2),
    # 256-query blocks, last blocks of up to 128 queries in two key groups
    "blocks-256": ([769, 800, 896, 897, 1024, 640, 513, 800] * 2, 16), "block-256-less": ([130] * 20, 16),
    # segment counts around a wavefront and around the limit of the compact grid
    "64-segments": ([1 + 5 * (i % 37) for i in range(64)], 2), "65-segments": ([1 + 5 * (i % 37) for i in range(65)], 2),
    "256-segments": ([1 + i % 67 for i in range(256)], 2), "257-segments": ([1 + i % 67 for i in range(257)], 2),
    "none-but-the-last": ([0] * 200 + [300], 1),
}


def _inputs(lens, H, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    P = sum(lens)
    qkv = torch.randn(P, 3, H, 64, generator=g).to(dtype)
    bias = torch.where(torch.rand(P, generator=g) < 0.3, math.log(9.0), 0.0).to(dtype)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    return qkv, bias, cu


def _check(qkv, bias, cu, lens, mode):
    ref, ref_lse = oracle.biased_varlen_attention(qkv, cu, bias)
    out, lse, _ = flash_attn_varlen_qkvpacked_func_w_perkey_bias(qkv.to(DEV), cu.to(DEV), max(lens), perkey_bias=bias.to(DEV),
                                                                 return_attn_probs=True, scale_mode=mode)
    torch.testing.assert_close(out.float().cpu(), ref, atol=1e-2, rtol=1e-2)
    torch.testing.assert_close(lse.cpu(), ref_lse, atol=4e-3, rtol=1e-3)


@pytest.mark.parametrize("kind", ["bf16", "folded", "f16"])
@pytest.mark.parametrize("name", CASES)
def test_launch_shapes_against_the_oracle(name, kind):
    lens, H = CASES[name]
    dtype = torch.float16 if kind == "f16" else torch.bfloat16
    _check(*_inputs(lens, H, dtype, seed=len(lens)), lens, "folded" if kind == "folded" else "exact")


@pytest.mark.parametrize("kind", ["bf16", "folded", "f16"])
@pytest.mark.parametrize("ramp", ["rising", "late", "low"])
@pytest.mark.parametrize("lens,H", [([1100], 2), ([300, 500, 129], 3), ([800, 897] * 8, 16)], ids=["2x4", "2x2", "mixed"])
def test_reference_points_of_key_groups(lens, H, ramp, kind):
    """rising: every tile's largest score lies above the last one's; late: one key far above the rest; low: all scores
    far below the first reference point of the folded arithmetic (and ordinary for the other)."""
    dtype = torch.float16 if kind == "f16" else torch.bfloat16
    qkv, bias, cu = _inputs(lens, H, dtype, seed=7)
    bounds = cu.tolist()
    for s, e in zip(bounds[:-1], bounds[1:]):
        if ramp == "rising":
            bias[s:e] = (torch.arange(e - s) // 32 * 4).to(dtype)
        elif ramp == "late":
            bias[s + (e - s) * 3 // 4] = 120.0
        else:
            bias[s:e] -= 100.0
    _check(qkv, bias, cu, lens, "folded" if kind == "folded" else "exact")


@pytest.mark.parametrize("lens", [[1374] * 2, [700], [5, 300, 64, 257], [2748], [9000]], ids=["2x1374", "700", "ragged", "2748", "9000"])
def test_block_reference_bits_do_not_depend_on_the_launch(lens):
    """A segment alone and the same segment among others (another launch shape, another grid): equal bits; and within the
    tolerance of the oracle."""
    from come_amd.cuda_extension.flash_attn import _forward

    def run(t, cu, longest):
        t.come_qk_bound = 20.0                             # folded: the harness's qk-norm gives such a bound
        return _forward(t, cu, longest, None, 0.0, 0.125, False, (-1, -1), 0.0, None, False, block_reference=True)[0]

    H = 2
    qkv, _, cu = _inputs(lens, H, torch.bfloat16, seed=3)
    ref, _ = oracle.biased_varlen_attention(qkv, cu, None)
    out = run(qkv.to(DEV), cu.to(DEV), max(lens))
    torch.testing.assert_close(out.float().cpu(), ref, atol=1e-2, rtol=1e-2)
    many = 40 if max(lens) < 2000 else 3
    again = run(qkv.repeat(many, 1, 1, 1).to(DEV), torch.tensor([0] + lens * many).cumsum(0).to(torch.int32).to(DEV), 4000 if max(lens) < 4000 else max(lens))
    if max(lens) < 4096:                                   # (blocks of 256 queries in both)
        assert torch.equal(again.view(many, -1, H, 64), out.unsqueeze(0).expand(many, -1, -1, -1))
    torch.testing.assert_close(again[-sum(lens):].float().cpu(), ref, atol=1e-2, rtol=1e-2)
