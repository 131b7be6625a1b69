"""The suffix operators in the kernel for large tensors (20 MiB of output and more), at the edges of the blocks of 256
chunks that a wavefront copies: segments that end inside, at and beside such a block, rows of one chunk and rows longer
than a block, segments without rows, outputs on both sides of the two sizes at which the kernel changes, and the same
tokens 2 bytes off a 16-byte boundary (one thread per element).  Row copies: bit-exact."""

import pytest
import torch

import oracle
from come_amd.interface import JaggedTokens

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("shift", [0, 1], ids=["aligned", "odd"])
@pytest.mark.parametrize("C,T,lengths", [
    (8, 1, [255, 256, 257, 512, 1, 1, 1022, 1 << 21]),  # one chunk a row
    (8, 3, [1021, 3, 1 << 21, 253]),
    (24, 2, [85, 86, 170, 171, 3, 2, 683, 600001]),     # three chunks: blocks begin inside rows
    (2048, 1, [1, 2, 1, 40, 9000]),                     # one row a block
    (2056, 2, [3, 2, 30, 9000, 2]),                     # 257 chunks
    (6144, 1, [5, 1, 9, 2500]),                         # three blocks a row
    (1024, 1, [2] * 7000),                              # no block inside a segment
    (1024, 1, [0, 4000, 0, 0, 9000, 0]),                # segments without rows
    (1024, 2, [6236, 4000]), (1024, 2, [6235, 4000]),   # 20 MiB with the suffixes, and a row less
    (1024, 1, [40959, 40960]), (1024, 1, [40959, 40959]),   # 320 MiB moved, and a row less
], ids=lambda v: str(v) if not isinstance(v, list) else f"n{len(v)}")
def test_blocks_of_chunks(C, T, lengths, shift):
    g = torch.Generator().manual_seed(C + T)
    P, M = sum(lengths), len(lengths)
    offset = torch.tensor([0] + lengths).cumsum(0)
    tokens = torch.randn(1, P, C, generator=g).bfloat16()
    weight = torch.rand(P, generator=g)
    suffix = torch.randn(M, T, C, generator=g).bfloat16()
    want = oracle.add_suffix(oracle.JaggedTokens(tokens=tokens, weight=weight, offset=offset), suffix)

    def place(x):
        room = torch.empty(x.numel() + shift, dtype=x.dtype, device=DEV)
        room[shift:].copy_(x.flatten())
        return room[shift:].view(x.shape)

    got = JaggedTokens(tokens=place(tokens), weight=weight.to(DEV), offset=offset.to(DEV)).add_suffix(place(suffix))
    assert torch.equal(got.tokens.cpu(), want.tokens) and torch.equal(got.weight.cpu(), want.weight)
    assert torch.equal(got.offset.cpu(), want.offset)
    back, tail = JaggedTokens(tokens=place(got.tokens), weight=got.weight, offset=got.offset).split_suffix(T)
    assert torch.equal(back.tokens.cpu(), tokens) and torch.equal(back.weight.cpu(), weight)
    assert torch.equal(back.offset.cpu(), offset) and torch.equal(tail.cpu(), suffix)
