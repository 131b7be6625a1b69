"""Selection and selection with a plan at the sizes where another kernel or another number of keys per thread takes over."""

import pytest
import torch

import oracle
from come_amd import _lib
from come_amd.cuda_extension import co_me_cuext

pytestmark = pytest.mark.gpu
DEV = "cuda"
SIZES = [1, 2, 63, 64, 65, 191, 192, 193, 1024, 1025, 4096, 4097, 8192, 8193, 16384, 16385, 32768, 32769]


def _confidence(n, kind, dtype):
    """n windows of 1 x 2 whose sums are exact in any order and dtype."""
    g = torch.Generator().manual_seed(n)
    if kind == "spread":                       # both signs, several binary orders
        x = torch.randint(-128, 128, (1, 1, 2 * n), generator=g).float() * 2.0 ** torch.randint(-3, 4, (1, 1, 1), generator=g).float()
    elif kind == "narrow":                     # between 1 and 2.5, smooth: neighbours fall into one bin
        x = 1 + 1.5 * torch.linspace(0, 1, n).repeat_interleave(2).view(1, 1, -1)
        x = (x * 256).round() / 256 if dtype == torch.float32 else (x * 32).round() / 32
    else:                                      # two values
        x = torch.randint(0, 2, (1, 1, n), generator=g).float().repeat_interleave(2, dim=-1)
    return x.to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("kind", ["spread", "narrow", "two"])
@pytest.mark.parametrize("n", SIZES)
def test_masks(n, kind, dtype):
    conf = _confidence(n, kind, dtype)
    for ratio in (0.0, 0.37, 0.5, 1.0):
        want = oracle.select_lowest_confidence(conf, 1, 1, 2, ratio)
        got = co_me_cuext.co_me_select_windows(conf.to(DEV), 1, 1, 2, ratio, "pairwise-rank")
        assert torch.equal(got.cpu(), want)
        # with a plan: the merge that follows packs what the mask says
        tokens = torch.arange(1 + 2 * n, dtype=torch.float32).view(1, -1, 1).expand(-1, -1, 4).contiguous().to(DEV)
        out, index, counts, offsets, mask = co_me_cuext.co_me_select_merge_2d(tokens, conf.to(DEV), 1, 1, 1, 2, 1, 2 * n, ratio)
        assert torch.equal(mask.cpu(), want)
        ref, rev = oracle.token_merge_2d(tokens.cpu(), 1, 1, 2, 1, 2 * n, want)
        assert torch.equal(index.cpu().long(), rev) and torch.equal(offsets.cpu().long(), ref.offset) and torch.equal(out.cpu(), ref.tokens[0])


@pytest.mark.parametrize("n", [5, 192, 700, 5000, 9000, 20000, 40000])
def test_absolute_score_and_several_elements(n):
    g = torch.Generator().manual_seed(n)
    conf = torch.randint(0, 64, (3, 1, 2 * n), generator=g).float() / 64
    want = conf.view(3, n, 2).mean(-1) < 0.5
    got = co_me_cuext.co_me_select_windows(conf.to(DEV), 3, 1, 2, 0.5, "abs_mse")
    assert torch.equal(got.cpu(), want)
    ranked = co_me_cuext.co_me_select_windows(conf.to(DEV), 3, 1, 2, 0.4, "pairwise-rank")
    assert torch.equal(ranked.cpu(), oracle.select_lowest_confidence(conf, 3, 1, 2, 0.4))


def test_nan_selects_nothing_above_its_rank():
    """NaN keys rank above infinity, as in a sort: a threshold below them is a number, one of them compares false with all."""
    for n in (100, 3000, 12000):
        conf = torch.rand(1, 1, 2 * n, generator=torch.Generator().manual_seed(n))
        conf[0, 0, 6] = float("nan")
        top = co_me_cuext.co_me_select_windows(conf.to(DEV), 1, 1, 2, 1.0, "pairwise-rank")
        half = co_me_cuext.co_me_select_windows(conf.to(DEV), 1, 1, 2, 0.5, "pairwise-rank")
        assert int(top.sum()) == 0 and int(half.sum()) == (n - 1) // 2 + (n - 1) % 2 and not bool(half[0, 3])
    assert _lib.load().come_version() >= 304
