"""The unmerge at row widths around the limits of its kernels (a thread per chunk, 128 chunks to a wavefront, whole KiB), single and
pair, against an index by torch: bit for bit, indices out of range give rows of zeros."""

import pytest
import torch

from come_amd import _lib
from come_amd.cuda_extension import co_me_cuext

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("index", [torch.int64, torch.int32], ids=["i64", "i32"])
@pytest.mark.parametrize("chunks", [1, 21, 22, 42, 43, 44, 48, 63, 64, 65, 96, 127, 128, 130, 300])
@pytest.mark.parametrize("total", [1, 2, 3, 257, 5000])
def test_widths(total, chunks, index):
    g = torch.Generator(device=DEV).manual_seed(total * 1000 + chunks)
    rows, C = max(1, total // 3), chunks * 8
    a, b = (torch.randn(rows, C, generator=g, device=DEV).bfloat16() for _ in range(2))
    rev = torch.randint(0, rows, (total,), generator=g, device=DEV).to(index)
    assert torch.equal(co_me_cuext.co_me_token_split_cuda(a, rev, C), a[rev.long()])
    assert torch.equal(co_me_cuext.co_me_token_split_pair_cuda(a, b, rev, C), torch.cat((a[rev.long()], b[rev.long()]), 1))
    # the C entry checks nothing on the device but the range of an index
    rev[total // 2] = rows
    rev[0] = -1
    out = torch.full((total, C), float("nan"), device=DEV, dtype=torch.bfloat16)
    wide = index == torch.int64
    assert _lib.load().come_token_split(a.data_ptr(), _lib.COME_BF16, rows, C, rev.data_ptr() if wide else None, None if wide else rev.data_ptr(),
                                        total, out.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    want = a[rev.long().clamp(0, rows - 1)]
    want[(rev < 0) | (rev >= rows)] = 0
    assert torch.equal(out, want)


def test_outputs_beyond_the_infinity_cache():
    """Shorter runs on an XCD from 256 MiB on, in either kernel."""
    for C in (768, 1024):
        a = torch.randn(60000, C, device=DEV).bfloat16()
        rev = torch.randint(0, 60000, (130001,), device=DEV)
        assert torch.equal(co_me_cuext.co_me_token_split_cuda(a, rev, C), a[rev])
