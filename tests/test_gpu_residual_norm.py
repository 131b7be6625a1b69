"""LayerScale + residual + LayerNorm in one pass: the sum has the bits of the separate tensor operations, the normalised
value that of float64 up to its rounding; rows around every size at which the kernel changes its registers per lane."""

import pytest
import torch

from come_amd import _lib
from come_amd.harness import AggregatorConfig, AlternatingAggregator, relative_l1

# one rounding to the storage dtype, and fp32 statistics of values around one (the mean's rounding enters the difference)
EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -20}


def close_to(out, exact):
    err = (out.double() - exact).abs()
    return bool((err <= EPS[out.dtype] * exact.abs() + 4e-6).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,chunks", [(1, 1), (3, 63), (5, 64), (4, 65), (70, 96), (1031, 128), (9, 129), (2, 256), (3, 257), (5, 512)])
def test_against_separate_operations(dtype, rows, chunks):
    C = chunks * 16 // dtype.itemsize
    g = torch.Generator(device="cuda").manual_seed(rows * 1000 + chunks)
    x, y = (torch.randn(rows, C, device="cuda", generator=g).to(dtype) + i for i in range(2))
    scale, w, b = (torch.randn(C, device="cuda", generator=g).to(dtype) for _ in range(3))
    with torch.no_grad():
        for params in ((w, b), (w, None), (None, None)):
            s, n = _lib.host().residual_norm(x, y, scale, True, *params, 1e-5)
            assert torch.equal(s, x + scale * y)
            exact = torch.nn.functional.layer_norm(s.double(), (C,), *(None if p is None else p.double() for p in params), 1e-5)
            assert close_to(n, exact)
        s2, none = _lib.host().residual_norm(x, y, scale, False, None, None, 0.0)
        assert none is None and torch.equal(s2, s)
        wide = torch.randn(3, rows + 2, C, device="cuda", generator=g).to(dtype)
        n = _lib.host().layer_norm_groups(wide[:, 2:], w, b, 1e-5)
        assert n.is_contiguous() and close_to(n, torch.nn.functional.layer_norm(wide[:, 2:].double(), (C,), w.double(), b.double(), 1e-5))


@pytest.mark.gpu
def test_rows_with_infinities_stay_their_own():
    x = torch.randn(8, 1024, device="cuda").bfloat16()
    x[3, 700] = float("inf")
    one = torch.ones(1024, device="cuda").bfloat16()
    with torch.no_grad():
        s, n = _lib.host().residual_norm(x, torch.zeros_like(x), one, True, None, None, 1e-5)
    assert torch.equal(s, x)
    finite = torch.isfinite(n).all(1)
    assert finite.tolist() == [i != 3 for i in range(8)]


@pytest.mark.gpu
def test_calls_that_tensor_operations_keep():
    host = _lib.host()
    x, s = torch.randn(4, 64, device="cuda"), torch.ones(64, device="cuda")
    args = (True, None, None, 1e-5)
    assert host.residual_norm(x, x, s, *args) is None                                    # grad mode: tensor operations record
    with torch.no_grad():
        assert host.residual_norm(x, x, s, *args) is not None
        assert host.residual_norm(x[:, :63], x[:, :63], s[:63], *args) is None           # rows of 252 bytes, not contiguous
        assert host.residual_norm(x, x.bfloat16(), s, *args) is None
        assert host.residual_norm(x.double(), x.double(), s.double(), *args) is None
        assert host.residual_norm(x[:0], x[:0], s, *args) is None
        flat = torch.randn(4 * 64 + 1, device="cuda")[1:].view(4, 64)                    # not 16-byte aligned
        assert host.residual_norm(flat, x, s, *args) is None
        assert host.layer_norm_groups(x.view(2, 2, 64).transpose(0, 1), None, None, 1e-5) is None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert host.residual_norm(x, x, s, *args) is None


@pytest.mark.gpu
def test_model_with_hooks_runs_every_module_and_agrees():
    from come_amd.token_merger import CoMe_2D_TokenMerger

    torch.manual_seed(2)
    cfg = AggregatorConfig(dim=256, heads=4, mlp_dim=512, depth=4, merge_block=1, taps=(1, 3), head_hidden=64, conf_hidden=64)
    model = AlternatingAggregator(cfg).eval().to("cuda", torch.bfloat16)
    images = torch.rand(1, 2, 3, 14 * 19, 14 * 17, device="cuda")
    merger = CoMe_2D_TokenMerger(5, 3, 3, 0.5, allow_remainder=True)
    plain = model(images, merger=merger)
    calls = []
    norms = [n for blk in (*model.frame_blocks, *model.global_blocks) for n in (blk.norm1, blk.norm2)]
    for m in (*norms, *model.tap_norm, *model.frame_blocks, *model.global_blocks):
        m.register_forward_hook(lambda mod, args, out: calls.append(mod))
    hooked = model(images, merger=merger)
    assert len(calls) == len(norms) + 2 + 8
    assert torch.equal(plain["merge_mask"], hooked["merge_mask"])
    assert relative_l1(plain["maps"], hooked["maps"]) < 1e-2          # LayerNorms round the same sums from other fp32 orders


def test_argument_checks_on_the_host():
    lib = _lib.load()
    fake = 0x10000

    def call(x=fake, y=fake, scale=fake, dtype=_lib.COME_BF16, rows=4, channels=64, group=4, stride=0, w=None, out=fake, norm=fake, eps=1e-5):
        return lib.come_residual_norm(x, y, scale, dtype, rows, channels, group, stride, w, None, eps, out, norm, None)

    assert call(dtype=7) == 2 and call(channels=4100) == 2 and call(channels=4104) == 2
    assert call(x=None) == 1 and call(scale=None) == 1 and call(y=None, scale=None) == 1 and call(out=None, norm=None) == 1
    assert call(eps=-1.0) == 1 and call(w=fake + 2) == 1 and call(group=2, stride=100) == 1 and call(group=0) == 1
    assert call(rows=0) == 0
