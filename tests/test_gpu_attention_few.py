"""Launches of up to eight segments, whose blocks are dealt to the XCDs segment by segment: the same results as for the same segments
with empty ones behind them, which are more than that way takes, and the closed form on the borders of blocks."""

import pytest
import torch

from come_amd import _lib
from come_amd.cuda_extension import flash_attn_varlen_qkvpacked_func_w_perkey_bias

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("heads,lens", [
    (1, [1]),
    (5, [64, 0, 129, 1, 257, 0, 128, 300]),          # eight segments, empty ones among them
    (3, [513, 512, 511]),
    (6, [2100, 130, 90, 2100]),                      # equal lengths
    (12, [800, 1374, 1000]),
    (16, [300, 2900, 4000]),                         # the longest last
    (6, [7000, 0, 5000]),
    (7, [4100, 4700]),
    (16, [4200, 2800, 1160]),                        # 8 wavefronts, heads a multiple of 8
    (12, [5200, 4600, 300]),                         # with key shares
    (5, [600, 30000]),
], ids=str)
def test_every_block_once(heads, lens, dtype):
    total = sum(lens)
    g = torch.Generator(device=DEV).manual_seed(total + heads)
    qkv = torch.randn(total, 3, heads, 64, generator=g, device=DEV).to(dtype)
    bias = (torch.rand(total, generator=g, device=DEV) * 3).log().clamp(min=-4).to(dtype)
    cu = torch.tensor([0] + lens, device=DEV).cumsum(0).to(torch.int32)
    more = torch.cat((cu, cu[-1:].expand(9)))

    def run(offsets):
        out, lse, _ = flash_attn_varlen_qkvpacked_func_w_perkey_bias(qkv, offsets, max(lens), perkey_bias=bias, softmax_scale=0.125,
                                                                     return_attn_probs=True)
        assert bool(torch.isfinite(out).all()) and bool(torch.isfinite(lse).all())
        return out, lse

    out, lse = run(cu)
    other, other_lse = run(more)
    # both within half a unit of the 16-bit outputs and 2^-9 (2^-10) of the probabilities: three units of the larger one at most
    unit = 2 ** -8 if dtype == torch.bfloat16 else 2 ** -10
    torch.testing.assert_close(out.float(), other.float(), atol=3 * unit * float(out.float().abs().max()), rtol=3 * unit)
    torch.testing.assert_close(lse, other_lse, atol=2e-3, rtol=1e-3)
    start = 0
    for L in lens:
        rows = sorted({*range(0, L, 128), *range(127, L, 128), L - 1} - {-1})[-64:]
        at = torch.as_tensor(rows, device=DEV, dtype=torch.int64)
        q, k, v = (qkv[start:start + L, i].double().transpose(0, 1).contiguous() for i in range(3))
        scores = torch.matmul(q[:, at], k.transpose(1, 2).contiguous()) * 0.125 + bias[start:start + L].double()
        ref = torch.matmul(torch.softmax(scores, -1), v).transpose(0, 1)
        assert float((out[start + at].double() - ref).norm()) <= unit * float(ref.norm()) * 1.5
        start += L


def test_key_shares_are_met():
    assert _lib.load().come_attn_work_bytes(3, 10100, 12, 5200) > 0 and _lib.load().come_attn_work_bytes(2, 30600, 5, 30000) > 0
