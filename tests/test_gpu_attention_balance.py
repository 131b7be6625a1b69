"""Long launches whose query blocks are dealt to the XCDs in equal shares: head counts that are and are no multiple of 8, segments of unequal
length (one shorter than a block, one empty), with and without the key-split tail, against the closed form on sampled rows."""

import numpy as np
import pytest
import torch

from come_amd import _lib
from come_amd.cuda_extension import flash_attn_varlen_qkvpacked_func_w_perkey_bias

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("heads,lens,split", [
    (6, [10000, 10000], False),                    # one full round of 512-query blocks
    (12, [5200, 4600, 300], True),
    (1, [65000, 60000, 700], False),
    (3, [22000, 18000], False),
    (12, [14000], True),
    (6, [9000, 0, 9300, 40], False),
    (5, [30000, 600], True),
    (6, [14000, 0, 9000, 40], True),
    (8, [300, 0] + [4700] * 7, True),              # more segments than are dealt one by one, heads a multiple of eight
    (16, [4500 - 167 * i for i in range(10)], False),
    (2, [40000] + [30] * 260, None),               # more segments than a wavefront counts
], ids=str)
def test_every_block_once(heads, lens, split):
    total = sum(lens)
    if split is not None:
        assert (_lib.load().come_attn_work_bytes(len(lens), total, heads, max(lens)) > 0) == split
    g = torch.Generator(device=DEV).manual_seed(total)
    qkv = torch.randn(total, 3, heads, 64, generator=g, device=DEV).bfloat16()
    bias = (torch.rand(total, generator=g, device=DEV) * 3).log().clamp(min=-4).bfloat16()
    cu = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32, device=DEV)
    out, lse, _ = flash_attn_varlen_qkvpacked_func_w_perkey_bias(qkv, cu, max(lens), perkey_bias=bias, softmax_scale=0.125,
                                                                 return_attn_probs=True)
    assert bool(torch.isfinite(out).all()) and bool(torch.isfinite(lse).all())
    start = 0
    for L in lens[:6]:
        if L == 0:
            continue
        # a row of every block, and the borders of the last ones
        rows = sorted({*range(0, L, 512), *range(255, L, 512), max(L - 513, 0), max(L - 512, 0), L - 1})
        q, k, v = (qkv[start:start + L, i].float().transpose(0, 1).contiguous() for i in range(3))
        for part in np.array_split(rows, -(-len(rows) // 32)):
            at = torch.as_tensor(part, device=DEV)
            scores = torch.matmul(q[:, at], k.transpose(1, 2).contiguous()) * 0.125 + bias[start:start + L].float()
            ref = torch.matmul(torch.softmax(scores, -1), v).transpose(0, 1)
            diff = (out[start + at].float() - ref).abs()
            assert float(diff.max()) <= 1e-2 and float(diff.mean()) <= 1e-3
            torch.testing.assert_close(lse[:, start + at], torch.logsumexp(scores, -1), atol=2e-3, rtol=1e-3)
        start += L
    # a looser bound of the lengths: the same products
    loose, _, _ = flash_attn_varlen_qkvpacked_func_w_perkey_bias(qkv, cu, max(lens) + 3000, perkey_bias=bias, softmax_scale=0.125,
                                                                 return_attn_probs=True)
    torch.testing.assert_close(loose.float(), out.float(), atol=4e-3, rtol=2 ** -7)
