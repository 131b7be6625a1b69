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
    (512, 1, (1, 2), (1, 64)),              # 16384, one copied token a row: a wavefront of narrow ones has 32 rows
    (70, 1, (1, 2), (1, 461)),              # 16100, and 32 rows are 7360 windows
    (300, 0, (2, 2), (5, 7)),               # 1800, leftover tokens alone
    (2100, 1, (1, 2), (1, 14)),             # 14700 in many rows
    (40, 3, (1, 2), (1, 31)),               # 600, two or three tokens of a row in a wavefront
]


def _fits(rows, window, grid, chans, row_bytes):
    windows, tokens = rows * (grid[0] // window[0]) * (grid[1] // window[1]), window[0] * window[1]
    # (from 8192 windows on where they have enough to move, or their rows are too many for the plan)
    return windows <= 16384 and (windows <= 8192 or rows > 2048 or chans <= 4 or (tokens >= 8 and tokens * row_bytes >= 4096))


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
        assert bool(takes) == (_fits(rows, window, grid, chans, row_bytes) and (row_bytes >= 32 if row_bytes % 16 == 0 else chans <= 4))
        want = _lib.host().merge_2d(tokens, start, gh, gw, H, W, mask, True, -1)
        for expected in {count, max(count - 1, 0), min(count + 1, rows * M)}:                    # right, and wrong by one
            got = _lib.host().merge_2d(tokens, start, gh, gw, H, W, mask, True, expected)
            for a, b in zip(got, want):
                assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.parametrize("chans", [16, 40, 1024])
@pytest.mark.parametrize("rows,start,window,grid", [(512, 1, (1, 2), (1, 64)), (16, 1, (1, 2), (1, 2048)), (70, 1, (1, 2), (1, 461)),
                                                     (16, 2, (2, 2), (65, 64))], ids=str)
def test_taken_where_the_plan_is_preferred(rows, start, window, grid, chans):
    """``come_token_merge_direct`` itself, from 8192 windows on that have little to move."""
    (gh, gw), (H, W) = window, grid
    n, M = start + H * W, (H // gh) * (W // gw)
    g = torch.Generator().manual_seed(rows + chans)
    tokens = torch.randn(rows, n, chans, generator=g).bfloat16().to(DEV)
    mask = (torch.rand(rows, M, generator=g) < 0.4).to(DEV)
    want = _lib.host().merge_2d(tokens, start, gh, gw, H, W, mask, True, -1)
    P = want[0].shape[1]
    got = (torch.empty_like(want[0]), torch.empty_like(want[1]), torch.empty_like(want[2]), torch.empty_like(want[3]))
    lib = _lib.load()
    rc = lib.come_token_merge_direct(tokens.data_ptr(), _lib._DTYPE_CODE[tokens.dtype], rows, n, chans, start, gh, gw, H, W, mask.data_ptr(),
                                     got[0].data_ptr(), P, got[3].data_ptr(), None, got[1].data_ptr(), None, got[2].data_ptr(), None, 0,
                                     torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.come_last_error()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_mask_at_an_odd_address_is_planned():
    tokens = torch.randn(2, 1 + 36, 16, device=DEV)
    flags = torch.rand(2 * 9 + 1, device=DEV) < 0.5
    mask = flags[1:].view(2, 9)
    assert not _lib.load().come_token_merge_is_direct(tokens.data_ptr(), 0, 2, 37, 16, 2, 2, 6, 6, mask.data_ptr())
    want = _lib.host().merge_2d(tokens, 1, 2, 2, 6, 6, mask.clone(), True, -1)
    got = _lib.host().merge_2d(tokens, 1, 2, 2, 6, 6, mask, True, int(mask.sum()))
    assert all(torch.equal(a, b) for a, b in zip(got, want))
