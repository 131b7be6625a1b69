"""The native host side of the token operators: the packed row count that the plan kernels post to the host, the merge
that is launched with the expected count (and again where window means tie), the plan that travels with a context's
mask, the one-launch plan of a caller's mask and the narrow-row merge, all against the oracle (integers and copied rows
bit for bit)."""

import pytest
import torch

import oracle
from come_amd.token_merger import CoMe_2D_TokenMerger, func_token_merge, func_token_merge_2d

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _check(jag, rev, ref, ref_rev, exact_values):
    assert torch.equal(jag.offset.cpu(), ref.offset) and jag.offset.dtype == torch.int64
    assert torch.equal(rev.cpu(), ref_rev) and torch.equal(jag.weight.cpu(), ref.weight)
    if exact_values:
        assert torch.equal(jag.tokens.cpu(), ref.tokens)
    else:                                    # bf16 means: one rounding of a sum in another order
        torch.testing.assert_close(jag.tokens.float().cpu(), ref.tokens.float(), atol=2 ** -8, rtol=2 ** -7)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("conf_kind", ["distinct", "ties", "constant"])
@pytest.mark.parametrize("frames,gh,gw,ratio", [(1, 7, 8, 0.5), (3, 16, 17, 0.0), (3, 16, 17, 1.0), (2, 37, 37, 0.5), (5, 12, 9, 0.73)])
def test_context_plan_serves_every_merge(frames, gh, gw, ratio, conf_kind, dtype):
    g = torch.Generator().manual_seed(frames * 100 + gh)
    conf = torch.rand(frames, gh, gw, generator=g)
    if conf_kind == "ties":                  # few distinct means: the expected packed count is wrong, the posted one right
        conf = (conf.mean((1, 2), keepdim=True) * 4).round().expand(frames, gh, gw).contiguous()
    elif conf_kind == "constant":
        conf = torch.ones(frames, gh, gw)
    conf = conf.to(dtype)
    tokens = torch.randint(-8, 8, (1, frames, 5 + gh * gw, 64), generator=g).float()
    pos = torch.randint(0, 38, (1, frames, 5 + gh * gw, 2), generator=g).to(torch.bfloat16)
    merger = CoMe_2D_TokenMerger(5, 3, 3, ratio, allow_remainder=True)
    ctx = merger.build_ctx(torch.empty(1, frames, 0, gh, gw, device=DEV), confidence=conf.to(DEV))
    want_mask = oracle.select_lowest_confidence(conf, 1, 3, 3, ratio)
    assert torch.equal(ctx[0].cpu(), want_mask)
    merged, (rev, _) = merger.merge(ctx, tokens.to(DEV))
    narrow, (rev2, _) = merger.merge(ctx, pos.to(DEV))
    ref, ref_rev = oracle.token_merge_2d(tokens[0], 5, 3, 3, gh, gw, want_mask, allow_remainder=True)
    _check(merged, rev, ref, ref_rev, False)
    ref2, _ = oracle.token_merge_2d(pos[0], 5, 3, 3, gh, gw, want_mask, allow_remainder=True)
    _check(narrow, rev2, ref2, ref_rev, False)
    # a mask that has been written to since is planned again
    ctx[0].logical_not_()
    flipped, (rev3, _) = merger.merge(ctx, tokens.to(DEV))
    ref3, ref_rev3 = oracle.token_merge_2d(tokens[0], 5, 3, 3, gh, gw, ~want_mask, allow_remainder=True)
    _check(flipped, rev3, ref3, ref_rev3, False)


@pytest.mark.parametrize("rows,groups", [(1, 1), (1, 255), (2, 256), (7, 257), (33, 300), (64, 1), (3000, 3), (6000, 1)])
def test_plan_of_a_callers_mask(rows, groups):
    """One launch while the workgroups' reads of the mask stay small (row and step borders of it), two beyond."""
    g = torch.Generator().manual_seed(rows + groups)
    tokens = torch.randint(-8, 8, (rows, 1 + 2 * groups, 8), generator=g).float()        # exact in any order
    mask = torch.rand(rows, groups, generator=g) < 0.5
    jag, rev = func_token_merge(tokens.to(DEV), 1, 2, mask.to(DEV))
    ref, ref_rev = oracle.token_merge_1d(tokens, 1, 2, mask)
    _check(jag, rev, ref, ref_rev, True)


@pytest.mark.parametrize("chans", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("gh,gw,H,W,S", [(3, 3, 7, 8, 2), (2, 1, 4, 3, 0), (1, 4, 5, 4, 1), (3, 3, 2, 2, 1)])
def test_narrow_rows(gh, gw, H, W, S, chans):
    g = torch.Generator().manual_seed(chans * 10 + gh)
    tokens = torch.randint(-8, 8, (3, S + H * W, chans), generator=g).half()
    mask = torch.rand(3, (H // gh) * (W // gw), generator=g) < 0.5
    jag, rev = func_token_merge_2d(tokens.to(DEV), S, gh, gw, H, W, mask.to(DEV), allow_remainder=True)
    ref, ref_rev = oracle.token_merge_2d(tokens, S, gh, gw, H, W, mask, allow_remainder=True)
    _check(jag, rev, ref, ref_rev, False)


def test_more_plans_than_words_and_plans_that_die_unread():
    """Contexts beyond the number of host words read their count back; words of contexts that nobody merged return."""
    merger = CoMe_2D_TokenMerger(1, 2, 2, 0.5)
    conf = torch.rand(1, 4, 6, generator=torch.Generator().manual_seed(0)).to(DEV)
    tokens = torch.randn(1, 1, 25, 16, generator=torch.Generator().manual_seed(1)).to(DEV)
    feature = torch.empty(1, 1, 0, 4, 6, device=DEV)
    want = merger.merge(merger.build_ctx(feature, confidence=conf), tokens)[0]
    for _ in range(2):
        ctxs = [merger.build_ctx(feature, confidence=conf) for _ in range(700)]
        for ctx in ctxs[::50] + ctxs[-1:]:
            got = merger.merge(ctx, tokens)[0]
            assert torch.equal(got.tokens, want.tokens) and torch.equal(got.offset, want.offset)
        del ctxs


def test_contexts_that_are_copied_or_saved_are_planned_again():
    import copy
    import io
    import pickle

    merger = CoMe_2D_TokenMerger(1, 2, 2, 0.5)
    conf = torch.rand(2, 4, 6, generator=torch.Generator().manual_seed(3)).to(DEV)
    tokens = torch.randn(1, 2, 25, 16, generator=torch.Generator().manual_seed(4)).to(DEV)
    ctx = merger.build_ctx(torch.empty(1, 2, 0, 4, 6, device=DEV), confidence=conf)
    want = merger.merge(ctx, tokens)[0]
    file = io.BytesIO()
    torch.save(ctx, file)
    file.seek(0)
    for other in (copy.deepcopy(ctx), copy.copy(ctx), pickle.loads(pickle.dumps(ctx)), torch.load(file, weights_only=True)):
        got = merger.merge(other, tokens)[0]
        assert torch.equal(got.tokens, want.tokens) and torch.equal(got.weight, want.weight) and torch.equal(got.offset, want.offset)
