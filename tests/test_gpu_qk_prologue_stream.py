"""The q / k prologue of large launches (a lane streams through the tokens) against the same rows in launches small enough for
the other kernel, whose arithmetic the oracle covers: the same bits."""

import pytest
import torch

from come_amd.common import RotaryPositionEmbedding2D, prepare_packed_self_attention_qkv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("heads,tokens", [(16, 4096), (16, 4097), (16, 9001), (12, 5500), (6, 11003), (20, 3300), (40, 3001), (1, 70001)])
@pytest.mark.parametrize("what", ["both", "norm", "rope", "k_only"])
def test_same_bits_as_small_launches(heads, tokens, what, dtype):
    g = torch.Generator(device="cuda").manual_seed(tokens)
    qkv = torch.randn(tokens, 3, heads, 64, device="cuda", generator=g).to(dtype)
    pos = torch.randint(0, 38, (tokens, 2), device="cuda", generator=g)
    norms = []
    for _ in range(2):
        n = torch.nn.LayerNorm(64, device="cuda", dtype=dtype)
        n.weight.data.copy_(1 + 0.1 * torch.randn(64, device="cuda", generator=g))
        n.bias.data.copy_(0.1 * torch.randn(64, device="cuda", generator=g))
        norms.append(n if what != "rope" else torch.nn.Identity())
    rope = RotaryPositionEmbedding2D(100.0) if what != "norm" else None

    def run(x, p):
        extra = {"defer_q": True} if what == "k_only" else {}
        with torch.no_grad():
            return prepare_packed_self_attention_qkv(x.clone(), *norms, rope, p if rope is not None else None, dtype, max_position=37, **extra)

    got = run(qkv, pos)
    step = 400000 // (16 * heads)                          # rows of a launch that stays with one row a lane
    want = torch.cat([run(qkv[i:i + step], pos[i:i + step]) for i in range(0, tokens, step)])
    assert not torch.equal(want, qkv)
    assert torch.equal(got, want)
