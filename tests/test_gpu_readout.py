"""The fused read-out (row norm and sigmoid gate) against its formula in 64
bits, and the layer's choice between it and torch's kernels."""
from __future__ import annotations

import pytest
import torch

from ramnet_ops import _native as nat
from ramnet_ops.impl import _ops

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
UNIT = {torch.float32: 2.0 ** -24, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _make(rows, C, dtype):
    g = torch.Generator(device=DEV).manual_seed(rows + C)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    return rnd(rows, C), 3 * rnd(rows, C), rnd(C)


def _exact(y, gate, weight, eps):
    y, gate, weight = y.double(), gate.double(), weight.double()
    return torch.sigmoid(gate) * y * weight / (y.square().mean(-1, keepdim=True) + eps).sqrt()


# rounding to the type, and in fp32 the sum of C squares (at most C units, halved by the
# square root), the root, the quotients, the exponential (2 units) and the products
def _bound(C, dtype):
    return 1.01 * UNIT[dtype] + (C / 2 + 10) * UNIT[torch.float32]


@pytest.mark.parametrize("dtype", list(UNIT))
@pytest.mark.parametrize("rows,C", [(1, 8), (3, 16), (17, 24), (63, 40), (64, 64), (65, 128), (1000, 256), (5, 512)])
def test_readout(rows, C, dtype):
    y, gate, weight = _make(rows, C, dtype)
    if C * y.element_size() > 1024:
        assert not _ops.readout_fits(y, gate, weight)
        with pytest.raises(RuntimeError, match="must fit one wave"):
            torch.ops.ramnet_ops.readout(y, gate, weight, 1e-6)
        return
    out = torch.ops.ramnet_ops.readout(y, gate, weight, 1e-6)
    want = _exact(y, gate, weight, 1e-6)
    tiny = 2.0 ** -24 if dtype == torch.float16 else 0.0  # half a unit of fp16's subnormals, rounded up
    assert ((out.double() - want).abs() <= _bound(C, dtype) * want.abs() + tiny).all()


@pytest.mark.parametrize("dtype", list(UNIT))
def test_readout_single_elements(dtype):
    """Rows off the 16-byte grid, at the native entry."""
    rows, C = 21, 37
    y, gate, weight = _make(rows, C, dtype)
    assert not _ops.readout_fits(y, gate, weight)
    out = torch.empty_like(y)
    nat.call("ramnet_readout", y.data_ptr(), gate.data_ptr(), weight.data_ptr(), nat.DTYPE_CODES[dtype], rows, C, 1e-6,
             out.data_ptr(), nat.stream_of(y))
    want = _exact(y, gate, weight, 1e-6)
    assert ((out.double() - want).abs() <= _bound(C, dtype) * want.abs() + 2.0 ** -24).all()


def test_readout_special_values():
    """NaN and infinities stay in their row; a zero row gives zeros."""
    y, gate, weight = _make(4, 128, torch.float32)
    y[0, 3], y[1, 5], y[2] = float("nan"), float("inf"), 0.0
    gate[3, :2] = torch.tensor([float("inf"), float("-inf")])
    out = torch.ops.ramnet_ops.readout(y, gate, weight, 1e-6)
    want = _exact(y, gate, weight, 1e-6)
    assert torch.equal(out.isnan(), want.isnan()) and (out[2] == 0).all() and out[3, 1] == 0
    ok = ~want.isnan()
    assert ((out.double() - want).abs()[ok] <= _bound(128, torch.float32) * want.abs()[ok]).all()


def test_layer_choice():
    """The layer takes the fused form without derivatives or hooks, and the two
    forms agree to the roundings torch's form adds (norm, sigmoid, product)."""
    from ramnet_harness import HarnessConfig
    from ramnet_harness.lm import RamLayer
    cfg = HarnessConfig(d_model=64, heads=4, value_chs=32, addr_order=2, addr_radix=8, top_k=4, embed_num=2)
    torch.manual_seed(0)
    layer = RamLayer(cfg)
    layer.init_weights()
    layer = layer.to(DEV, torch.bfloat16)
    layer.out = torch.nn.Identity()  # the read-out itself
    x = torch.randn(2, 9, 64, device=DEV).to(torch.bfloat16)
    pos = torch.arange(9, device=DEV).view(1, 9).expand(2, 9)
    with torch.no_grad():
        fused, _ = layer(x, (None, None), pos, False)
        calls = []
        handle = layer.out_norm.register_forward_hook(lambda *a: calls.append(1))
        plain, _ = layer(x, (None, None), pos, False)
        handle.remove()
    assert calls == [1]
    assert ((fused.double() - plain.double()).abs() <= 4.1 * UNIT[torch.bfloat16] * plain.double().abs()).all()
    out, _ = layer(x.clone().requires_grad_(), (None, None), pos, False)
    assert out.requires_grad and torch.equal(out, plain)


def _small_layer():
    from ramnet_harness import HarnessConfig
    from ramnet_harness.lm import RamLayer
    cfg = HarnessConfig(d_model=64, heads=4, value_chs=32, addr_order=2, addr_radix=8, top_k=4, embed_num=2)
    torch.manual_seed(1)
    layer = RamLayer(cfg)
    layer.init_weights()
    layer = layer.to(DEV).requires_grad_(False)
    layer.out = torch.nn.Identity()
    x = torch.randn(2, 9, 64, device=DEV)
    pos = torch.arange(9, device=DEV).view(1, 9).expand(2, 9)
    return layer, lambda weight: torch.func.functional_call(layer, {"out_norm.weight": weight},
                                                            (x, (None, None), pos, False))[0]


@pytest.mark.parametrize("grad_mode", [False, True])
def test_layer_keeps_forward_mode(grad_mode):
    """A tangent on the norm's weight alone reaches the output (which is linear
    in the weight), through dual tensors and through torch.func.jvp."""
    layer, call = _small_layer()
    weight, tangent = layer.out_norm.weight.detach() + 0.5, torch.randn(32, device=DEV)
    with torch.set_grad_enabled(grad_mode):
        want = call(tangent)
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(weight, tangent)
            got = torch.autograd.forward_ad.unpack_dual(call(dual)).tangent
        assert got is not None
        torch.testing.assert_close(got, want, atol=1e-6, rtol=1e-5)
        torch.testing.assert_close(torch.func.jvp(call, (weight,), (tangent,))[1], want, atol=1e-6, rtol=1e-5)


def test_layer_keeps_vmap_and_grad_transforms():
    """The norm's weight as a batch of torch.vmap, and as the argument of torch.func.grad."""
    layer, call = _small_layer()
    weights = torch.randn(3, 32, device=DEV)
    with torch.no_grad():
        got = torch.vmap(call)(weights)
        torch.testing.assert_close(got, torch.stack([call(w) for w in weights]), atol=1e-6, rtol=1e-5)
    up = torch.randn(2, 9, 128, device=DEV)
    grad = torch.func.grad(lambda w: (call(w) * up).sum())(weights[0])
    basis = torch.stack([(call(e) * up).sum() for e in torch.eye(32, device=DEV)])
    torch.testing.assert_close(grad, basis, atol=1e-4, rtol=1e-4)


def test_readout_refuses_tangents():
    y, gate, weight = _make(4, 32, torch.float32)
    for at in range(3):
        with torch.autograd.forward_ad.dual_level():
            args = [y, gate, weight]
            args[at] = torch.autograd.forward_ad.make_dual(args[at], torch.ones_like(args[at]))
            with pytest.raises(NotImplementedError, match="forward-mode"):
                torch.ops.ramnet_ops.readout(*args, 1e-6)


# torch's own fp32 values differ by a few units (its sum's order, its root), about 2**-21 of a value, and
# turn a rounding to 16 bits where they straddle a boundary: 2**-21 of the values' spacing, 2**-8 or 2**-11,
# in each of two roundings (a product rounds with them): under 1 in 400 elements, one unit each and its product's
@pytest.mark.parametrize("dtype", list(UNIT))
@pytest.mark.parametrize("rows,C", [(3, 24), (1000, 128), (257, 256)])
def test_readout_stepwise(rows, C, dtype):
    """Rounded step by step, the kernel gives the values of torch's three operators."""
    y, gate, weight = _make(rows, C, dtype)
    out = torch.ops.ramnet_ops.readout(y, gate, weight, 1e-6, stepwise=True)
    want = torch.sigmoid(gate) * torch.nn.functional.rms_norm(y, (C,), weight, 1e-6)
    off = (out.double() - want.double()).abs()
    assert (off <= (4 * UNIT[dtype] if dtype != torch.float32 else _bound(C, dtype)) * want.double().abs() + 2.0 ** -24).all()
    if dtype != torch.float32:
        assert (off != 0).double().mean() <= 1 / 400 + 1 / off.numel()


def test_layer_values_do_not_depend_on_the_form():
    """The layer's fused read-out against its separate operators, which a hook
    or a wanted gradient selects: equal but for single roundings."""
    from ramnet_harness import HarnessConfig
    from ramnet_harness.lm import RamLayer
    cfg = HarnessConfig(d_model=256, heads=8, value_chs=128, addr_order=2, addr_radix=16, top_k=8, embed_num=4)
    torch.manual_seed(2)
    layer = RamLayer(cfg)
    layer.init_weights()
    layer = layer.to(DEV, torch.bfloat16)
    layer.out = torch.nn.Identity()
    x = torch.randn(2, 64, 256, device=DEV).to(torch.bfloat16)
    pos = torch.arange(64, device=DEV).view(1, 64).expand(2, 64)
    with torch.no_grad():
        fused, _ = layer(x, (None, None), pos, False)
        layer.out_norm.register_forward_hook(lambda *a: None)
        plain, _ = layer(x, (None, None), pos, False)
    assert (fused != plain).double().mean() <= 1 / 400
