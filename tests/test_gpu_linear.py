"""``come_linear`` against the product in 64 bits: every tile shape, remainders of rows, columns and k-steps, both activations; and
when a module's linear layers are left to the module."""

import pytest
import torch
from torch import nn

from come_amd import _lib, harness

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _run(x, w, b, gelu):
    out = torch.full((x.shape[0], w.shape[0]), float("nan"), dtype=x.dtype, device=DEV)
    lib = _lib.load()
    rc = lib.come_linear(x.data_ptr(), w.data_ptr(), None if b is None else b.data_ptr(), _lib._DTYPE_CODE[x.dtype], x.shape[0], x.shape[1],
                         w.shape[0], int(gelu), out.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0, lib.come_last_error()
    return out


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("rows,K,N", [
    (1, 64, 8), (63, 128, 72), (65, 192, 64), (200, 256, 1000),          # 64 x 64, fewer steps than stages
    (700, 512, 3072), (130, 4096, 2048), (1024, 448, 2056),             # 128 x 128
    (1500, 256, 3080), (1596, 1024, 3072),                              # 128 x 192
    (1600, 320, 4104), (2200, 1024, 3072),                              # 256 x 128
    (3000, 256, 4096), (3001, 1024, 4104),                              # 192 x 256
    (12800, 128, 4096), (12769, 1024, 4096),                            # 256 x 256
], ids=str)
def test_product(rows, K, N, dtype):
    g = torch.Generator(device=DEV).manual_seed(rows + K + N)
    x = torch.randn(rows, K, generator=g, device=DEV).to(dtype)
    w = (torch.randn(N, K, generator=g, device=DEV) / K ** 0.5).to(dtype)
    b = torch.randn(N, generator=g, device=DEV).to(dtype)
    for bias in (b, None):
        exact = x.double() @ w.double().t() + (0 if bias is None else bias.double())
        # fp32 sums: K roundings of partial sums of at most this size; 16-bit results: half a unit in the last place
        size = x.abs().float() @ w.abs().float().t() + 3
        sums = K * 2.0 ** -24 * size.double()
        half = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12
        tiny = 2.0 ** -25                                                # (fp16: half the smallest subnormal)
        y = _run(x, w, bias, False).double()
        assert bool(((y - exact).abs() <= half * 2 * exact.abs() + sums + tiny).all())
        z = _run(x, w, bias, True).double()
        want = nn.functional.gelu(exact)
        # its derivative stays below 1.13; the error function is good to 1.5e-7
        assert bool(((z - want).abs() <= half * 2 * want.abs() + 1.13 * sums + 1e-7 * exact.abs() + tiny).all())


def test_bits_do_not_depend_on_the_shape():
    g = torch.Generator(device=DEV).manual_seed(0)
    x = torch.randn(6000, 1024, generator=g, device=DEV).bfloat16()
    w = (torch.randn(4096, 1024, generator=g, device=DEV) / 32).bfloat16()
    whole = _run(x, w, None, False)
    for rows in (1, 100, 700, 1100, 2200, 3000):
        assert torch.equal(_run(x[:rows], w, None, False), whole[:rows])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("rows,K,N", [
    (24576 + 960, 192, 4096), (24576 + 1025, 64, 4096), (24576, 64, 4096),      # a round of 128 x 128 tiles left, one of 256 x 128, nothing
    (24576 + 2048, 64, 4096), (81920 + 7000, 64, 1000), (27088, 128, 3080), (9887, 192, 4096),      # in 256 x 128
    (13342, 128, 3072), (107523, 128, 384), (54340, 1024, 768),         # left to the estimate: half a round, columns that pad, narrowing
    (19201, 64, 4280), (19200 + 128 * 7, 128, 4224), (81920 + 77, 64, 1000), (294912 + 77, 64, 264),        # columns that are no multiple of a tile
], ids=str)
def test_whole_rounds_and_what_is_left(rows, K, N, dtype):
    """Launches in two tile shapes against the same rows in small launches: bit for bit (every output is one chain of additions)."""
    g = torch.Generator(device=DEV).manual_seed(rows + N)
    x = torch.randn(rows, K, generator=g, device=DEV).to(dtype)
    w = (torch.randn(N, K, generator=g, device=DEV) / K ** 0.5).to(dtype)
    b = torch.randn(N, generator=g, device=DEV).to(dtype)
    got = _run(x, w, b, True)
    assert not bool(got.isnan().any())
    for first in [*range(0, rows, 4000)][-3:] + [0, rows // 2 // 256 * 256]:
        assert torch.equal(_run(x[first:first + 4000], w, b, True), got[first:first + 4000])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@torch.no_grad()
@pytest.mark.parametrize("rows,K,N", [(1, 512, 8), (70, 1024, 512), (129, 640, 136), (257, 4096, 1024), (1596, 4096, 1024), (1024, 2048, 1000)], ids=str)
def test_shares_meet_in_the_residual_step(rows, K, N, dtype):
    g = torch.Generator(device=DEV).manual_seed(rows + K)
    h = torch.randn(rows, K, generator=g, device=DEV).to(dtype)
    w = (torch.randn(N, K, generator=g, device=DEV) / K ** 0.5).to(dtype)
    b, scale, gain, shift = (torch.randn(N, generator=g, device=DEV).to(dtype) for _ in range(4))
    x = torch.randn(rows, N, generator=g, device=DEV).to(dtype)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    code = _lib._DTYPE_CODE[dtype]
    half = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12
    for splits in (2, 4):
        if K // 64 < 4 * splits:
            assert lib.come_linear_split(h.data_ptr(), w.data_ptr(), code, rows, K, N, splits, x.data_ptr(), stream) != 0
            continue
        part = torch.full((splits, rows, N), float("nan"), device=DEV)
        assert lib.come_linear_split(h.data_ptr(), w.data_ptr(), code, rows, K, N, splits, part.data_ptr(), stream) == 0
        exact = h.double() @ w.double().t()
        size = h.abs().float() @ w.abs().float().t()
        assert bool(((part.double().sum(0) - exact).abs() <= K * 2.0 ** -24 * size.double()).all())
        for bias in (b, None):
            total, normed = torch.full_like(x, float("nan")), torch.full_like(x, float("nan"))
            assert lib.come_residual_norm_split(x.data_ptr(), part.data_ptr(), splits, None if bias is None else bias.data_ptr(), scale.data_ptr(),
                                                code, rows, N, gain.data_ptr(), shift.data_ptr(), 1e-5, total.data_ptr(), normed.data_ptr(), stream) == 0
            y = part[0]
            for s in range(1, splits):
                y = y + part[s]
            y = (y if bias is None else bias.float() + y).to(dtype)
            want, want_norm = _lib.host().residual_norm(x, y, scale, True, gain, shift, 1e-5)
            assert torch.equal(total, want) and torch.equal(normed, want_norm)


def test_infinities_and_nan_stay_in_their_rows():
    x = torch.randn(300, 128, device=DEV).bfloat16()
    w = torch.randn(136, 128, device=DEV).bfloat16()
    want = _run(x, w, None, True)
    y = x.clone()
    y[7, 3], y[299, 127] = float("nan"), float("inf")
    got = _run(y, w, None, True)
    assert bool(got[7].isnan().all()) and not bool(got[299].isfinite().all())
    keep = torch.ones(300, dtype=torch.bool, device=DEV)
    keep[[7, 299]] = False
    assert torch.equal(got[keep], want[keep])
    # GELU far out and of infinities, as torch gives it
    big = torch.zeros(5, 64, device=DEV).bfloat16()
    big[:, 0] = torch.tensor([-300.0, -20.0, 20.0, 300.0, float("inf")])
    one = torch.zeros(8, 64, device=DEV).bfloat16()
    one[:, 0] = 1
    assert torch.equal(_run(big[:4], one, None, True), nn.functional.gelu(big[:4, :1].float()).bfloat16().expand(4, 8))
    one.fill_(1)
    assert bool((_run(big, one, None, True)[4] == float("inf")).all())


def test_what_is_left_to_the_module():
    layer = nn.Linear(128, 256, device=DEV, dtype=torch.bfloat16)
    x = torch.randn(200, 128, device=DEV, dtype=torch.bfloat16)
    calls = []
    own = _lib.host().linear

    def plain():
        return own(x, layer.weight, layer.bias, True) is not None

    with torch.no_grad():
        assert plain()
        ref = nn.functional.gelu(layer(x))
        torch.testing.assert_close(harness._linear(layer, x, gelu=True), ref, atol=2 ** -7, rtol=2 ** -7)
        assert torch.equal(harness._linear(layer, x, gelu=True, fuse=False), ref)
        handle = layer.register_forward_hook(lambda *a: calls.append(1))
        assert torch.equal(harness._linear(layer, x, gelu=True), ref) and calls
        handle.remove()
        with torch.autocast("cuda", dtype=torch.float16):
            assert own(x, layer.weight, layer.bias, False) is None
        assert own(x.float(), layer.weight.float(), layer.bias.float(), False) is None
        assert own(x[:, ::2], layer.weight[:, :64], layer.bias, False) is None               # neither is contiguous
        assert own(x.flatten()[1:129].view(1, 128), layer.weight, layer.bias, False) is None  # 2-byte aligned
    assert not plain()                                                                        # gradients are wanted
    harness._linear(layer, x).float().sum().backward()
    assert layer.weight.grad is not None
