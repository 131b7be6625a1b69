"""Merges that find the packed positions in the mask (``come_token_merge_direct``: the packed count is expected) against planned
ones (no count expected): every output bit for bit, at the borders of the mask's words and steps, of wavefronts and rows."""

import pytest
import torch

from come_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"

# rows, start, window, grid: windows in all
CASES = [
    (1, 0, (3, 3), (3, 3)),                 # 1, nothing but windows
    (1, 5, (3, 3), (16, 17)),               # 25
    (3, 2, (3, 3), (7, 8)),                 # 12, a row's windows share a word
    (17, 1, (1, 2), (1, 30)),               # 255
    (16, 0, (1, 4), (1, 64)),               # 256, neither specials nor leftover
    (130, 1, (4, 1), (5, 3)),               # 390, rows shorter than a workgroup
    (16, 5, (3, 3), (37, 37)),              # 2304
    (1, 3, (1, 2), (1, 8193)),              # 4096, the loads in front of the token loads
    (5, 0, (2, 2), (41, 82)),               # 4100
    (16, 1, (1, 2), (1, 2048)),             # 16384, the largest
    (1, 1, (1, 2), (1, 32771)),             # 16385: planned
]


def _fits(rows, window, grid):
    return rows * (grid[0] // window[0]) * (grid[1] // window[1]) <= 16384


@pytest.mark.parametrize("chans,dtype", [(1, torch.bfloat16), (2, torch.float32), (4, torch.float16), (16, torch.bfloat16), (8, torch.float32),
                                         (24, torch.float16), (768, torch.bfloat16), (1024, torch.bfloat16), (8, torch.bfloat16), (5, torch.float32)],
                         ids=str)
@pytest.mark.parametrize("rows,start,window,grid", CASES, ids=str)
def test_direct_equals_planned(rows, start, window, grid, chans, dtype):
    (gh, gw), (H, W) = window, grid
    n = start + H * W
    if rows * n * chans > 1 << 25:
        chans = 32
    g = torch.Generator().manual_seed(rows * 1000 + chans)
    tokens = torch.randn(rows, n, chans, generator=g).to(dtype).to(DEV)
    M = (H // gh) * (W // gw)
    lib = _lib.load()
    for share in (0.0, 0.3, 1.0):
        mask = (torch.rand(rows, M, generator=g) < share).to(DEV)
        count = int(mask.sum())
        takes = lib.come_token_merge_is_direct(tokens.data_ptr(), _lib._DTYPE_CODE[dtype], rows, n, chans, gh, gw, H, W, mask.data_ptr())
        row_bytes = chans * tokens.element_size()
        assert bool(takes) == (_fits(rows, window, grid) and (row_bytes >= 32 if row_bytes % 16 == 0 else chans <= 4))
        want = _lib.host().merge_2d(tokens, start, gh, gw, H, W, mask, True, -1)
        for expected in {count, max(count - 1, 0), min(count + 1, rows * M)}:                    # right, and wrong by one
            got = _lib.host().merge_2d(tokens, start, gh, gw, H, W, mask, True, expected)
            for a, b in zip(got, want):
                assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)


def test_mask_at_an_odd_address_is_planned():
    tokens = torch.randn(2, 1 + 36, 16, device=DEV)
    flags = torch.rand(2 * 9 + 1, device=DEV) < 0.5
    mask = flags[1:].view(2, 9)
    assert not _lib.load().come_token_merge_is_direct(tokens.data_ptr(), 0, 2, 37, 16, 2, 2, 6, 6, mask.data_ptr())
    want = _lib.host().merge_2d(tokens, 1, 2, 2, 6, 6, mask.clone(), True, -1)
    got = _lib.host().merge_2d(tokens, 1, 2, 2, 6, 6, mask, True, int(mask.sum()))
    assert all(torch.equal(a, b) for a, b in zip(got, want))
