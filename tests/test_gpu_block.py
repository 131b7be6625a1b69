"""The block as one native call against the same block operator by operator (same kernels: bit for bit), and what keeps it from
being one call."""

import pytest
import torch
from torch import nn

from come_amd import harness
from come_amd.harness import AggregatorConfig, JaggedBlock

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _setup(dtype, heads=2, dim=128, rows=(37, 90, 64)):
    torch.manual_seed(0)
    with torch.device(DEV):
        block = JaggedBlock(AggregatorConfig(dim=dim, heads=heads, mlp_dim=256, layer_scale=0.7)).to(dtype).eval()
        nxt = nn.LayerNorm(dim, dtype=dtype)
        total = sum(rows)
        x = torch.randn(total, dim, dtype=dtype)
        pos = torch.randint(0, 10, (total, 2))
        cu = torch.tensor([0, *rows]).cumsum(0).to(torch.int32)
        bias = torch.rand(total).to(dtype)
    return block, nxt, (x, pos, 9, cu, max(rows), bias)


def _operators(block, args, attention, **kw):
    """The same forward with the native call switched off."""
    block._native = lambda *a: None
    try:
        return block(*args, attention, harness._default_prologue, **kw)
    finally:
        del block._native


@pytest.mark.parametrize("heads,dim", [(1, 64), (2, 128), (3, 192)], ids=["64", "128", "192"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("fuse", [True, False])
@torch.no_grad()
def test_one_call_equals_the_operators(dtype, fuse, heads, dim):
    block, nxt, args = _setup(dtype, heads, dim)
    native = JaggedBlock._native
    for attention in (harness._default_attention, harness._selection_attention):
        for bias in (args[5], None):
            for normed, after in ((None, nxt), (block.norm1(args[0]), None), (None, None)):
                a = (*args[:5], bias)
                done = native(block, *a, attention, harness._default_prologue, normed, after, fuse)
                assert done is not None
                want = _operators(block, a, attention, normed=normed, next_norm=after, fuse_norm=fuse)
                got = block(*a, attention, harness._default_prologue, normed=normed, next_norm=after, fuse_norm=fuse)
                for g, w in zip(got if after is not None else (got,), want if after is not None else (want,)):
                    assert torch.equal(g, w)


def test_what_is_left_to_the_operators():
    block, nxt, args = _setup(torch.bfloat16)
    rest = (harness._default_attention, harness._default_prologue, None, nxt, True)

    def native(a=args, r=rest):
        return block._native(*a, *r) is not None

    assert not native()                                                       # gradients are wanted
    with torch.no_grad():
        assert native()
        assert not native(r=(lambda *a: None, *rest[1:]))                      # somebody else's attention
        assert not native(r=(rest[0], harness.deferred_q_prologue, *rest[2:]))
        for name in ("norm1", "q_norm", "fc1"):
            seen = []
            hook = getattr(block, name).register_forward_hook(lambda *a: seen.append(1))
            assert not native()
            block(*args, *rest[:2])
            assert seen or name == "q_norm"                                     # (the prologue reads its parameters)
            hook.remove()
        assert native()
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert not native()
        from torch.utils.flop_counter import FlopCounterMode
        with FlopCounterMode(display=False) as flops:
            assert not native()
            block(*args, *rest[:2])
        assert flops.get_total_flops() > 0                                     # the linear layers were seen
        short = list(args)
        short[1] = args[1][:-1]                                                # positions that do not fit: the prologue says so
        with pytest.raises(RuntimeError, match="one \\(y, x\\) pair"):
            block(*short, *rest[:2])
        block.k_norm.eps = 1e-3
        with pytest.raises(RuntimeError, match="same eps"):
            block(*args, *rest[:2])


@pytest.mark.parametrize("form", ["replica", "attributes", "parametrized"])
@torch.no_grad()
def test_weights_that_are_no_registered_parameters(form):
    block, nxt, args = _setup(torch.bfloat16)
    want = _operators(block, args, harness._default_attention, next_norm=nxt)
    if form == "replica":
        def replica(m):                            # what nn.DataParallel makes of a module for another device
            r = m._replicate_for_data_parallel()
            for name, p in m._parameters.items():
                setattr(r, name, p.detach())
            for name, child in m._modules.items():
                setattr(r, name, replica(child))
            return r

        block, nxt = replica(block), replica(nxt)
    elif form == "attributes":
        for m in (block.norm1, block.qkv, block.q_norm, block.fc2, nxt):
            for name in ("weight", "bias"):
                value = getattr(m, name).detach().clone()
                delattr(m, name)
                setattr(m, name, value)
    else:
        nn.utils.parametrize.register_parametrization(block, "ls1", nn.Identity())
    got = block(*args, harness._default_attention, harness._default_prologue, next_norm=nxt)
    for g, w in zip(got, want):
        assert torch.equal(g, w)
    assert block._native(*args, harness._default_attention, harness._default_prologue, None, nxt, True) is not None


@torch.no_grad()
def test_a_default_device_is_no_watching_mode():
    block, nxt, args = _setup(torch.bfloat16)
    rest = (harness._default_attention, harness._default_prologue, None, nxt, True)
    host = harness._lib.host()
    x = args[0]

    def fused():
        return (block._native(*args, *rest) is not None,
                host.residual_norm(x, x, block.ls1, True, nxt.weight, nxt.bias, nxt.eps) is not None,
                host.layer_norm_groups(x[None], nxt.weight, nxt.bias, nxt.eps) is not None,
                host.linear(x, block.fc1.weight, block.fc1.bias, True) is not None)

    class Watcher(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    assert all(fused())
    for device in (DEV, "cpu"):
        with torch.device(device):
            assert all(fused())
            with Watcher():
                assert not any(fused())
        with Watcher(), torch.device(device):
            assert not any(fused())
    torch.set_default_device(DEV)
    try:
        assert all(fused())
    finally:
        torch.set_default_device(None)
    assert all(fused())
