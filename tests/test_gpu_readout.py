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
