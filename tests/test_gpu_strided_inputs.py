"""Calls on tensors that are not in (B, H, ..., T) memory order: the kernels
read them where they are, and give bit for bit what the same call gives on
contiguous copies (the same arithmetic in the same order, only the addresses
differ). Every route the strides can take: rows in 16-byte pieces, rows with
a digit of fewer logits than the kernel's list, unaligned rows, single logits
at any step, layouts that have to be copied, the workgroup search, and the
level, one-token, paired and slot-range scans.
"""
from __future__ import annotations

import pytest
import torch

from ramnet_ops import _native as nat
from ramnet_ops.impl import _ops  # registers torch.ops.ramnet_ops

pytestmark = pytest.mark.gpu

DEV = "cuda:0"

# how a (B, H, T, *feature) tensor lies in memory
ORDERS = {
    "bth": lambda t: _store(t, (0, 2, 1)),
    "tbh": lambda t: _store(t, (2, 0, 1)),
    "thb": lambda t: _store(t, (2, 1, 0)),
    "sliced": lambda t: _sliced(t),
    "feature_first": lambda t: _store(t, (3, 0, 2, 1)),
}


def _store(t, order):
    """t stored with its first dimensions in `order`, viewed as before."""
    perm = list(order) + [d for d in range(t.dim()) if d not in order]
    inv = [perm.index(d) for d in range(t.dim())]
    return t.permute(perm).contiguous().permute(inv)


def _sliced(t):
    """(B, T, H, ...) rows inside wider rows, one element off their start."""
    flat = t.transpose(1, 2)
    big = t.new_zeros((*flat.shape[:-1], flat.shape[-1] + 3))
    big[..., 1:-2] = flat
    return big[..., 1:-2].transpose(1, 2)


def _inputs(B, H, U, P, T, C, dtype, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    A = P ** U
    return dict(w=rnd(B, H, T, U, P).to(dtype), r=rnd(B, H, T, U, P).to(dtype), x=rnd(B, H, T, C).to(dtype),
                gamma=rnd(B, H, T).to(dtype), slot=rnd(B, H, A, C), mass=torch.rand(B, H, A, generator=g, device=DEV) + 0.1,
                mask=torch.rand(B, T, generator=g, device=DEV) > 0.2)


def _call(op, d, w, r, x, gamma, pos, mask, Kw, Kr, embed, ma):
    return op(w, r, x, gamma, d["slot"], d["mass"], mask, embed, pos, Kw, Kr, 0.5, 0.25, ma, 1e-6)


CASES = [  # B, H, U, P, T, C, Kw, Kr, dtype
    (2, 3, 2, 32, 70, 64, 8, 8, torch.bfloat16),     # whole digits, level scan
    (2, 2, 2, 4, 65, 16, 2, 3, torch.float16),       # an 8-byte digit
    (1, 2, 3, 16, 40, 40, 16, 12, torch.bfloat16),   # three digits, top-K 16
    (2, 2, 2, 24, 67, 36, 6, 5, torch.float16),      # 48-byte digits below the 32 kept
    (2, 2, 2, 12, 33, 20, 5, 4, torch.float32),      # fp32 digits below the 16 kept
    (2, 2, 2, 10, 33, 24, 4, 4, torch.bfloat16),     # 20-byte digits: single logits
    (2, 2, 1, 64, 31, 8, 4, 4, torch.float32),       # one digit, the widest list
    (1, 2, 2, 5, 40, 7, 20, 3, torch.float32),       # the workgroup search, one-token scan
    (1, 1, 2, 100, 9, 16, 4, 4, torch.bfloat16),     # the staircase search
    (1, 1, 3, 32, 33, 16, 4, 4, torch.float32),      # slot ranges, fp32 sums in y
    (1, 2, 3, 32, 33, 16, 4, 4, torch.bfloat16),     # slot ranges, sums in the workspace
    (3, 2, 2, 8, 1, 16, 4, 4, torch.bfloat16),       # one token
]


@pytest.mark.parametrize("order", list(ORDERS))
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v).replace("torch.", "") for v in c))
def test_strided_equals_contiguous(case, order):
    B, H, U, P, T, C, Kw, Kr, dtype = case
    d = _inputs(B, H, U, P, T, C, dtype)
    op = torch.ops.ramnet_ops.ram_attn_forward
    lay = ORDERS[order]
    pos = torch.arange(T, device=DEV).view(1, T) * 3 + torch.arange(B, device=DEV).view(B, 1) * 7 - 5
    logits = lambda t: t.permute(0, 1, 3, 4, 2)  # (B, H, U, P, T)
    for ma, mask, p in ((False, None, pos), (True, d["mask"], pos[:1].expand(B, T))):
        want = _call(op, d, logits(d["w"]).contiguous(), logits(d["r"]).contiguous(), d["x"], d["gamma"],
                     p.to(torch.int32).contiguous(), mask, Kw, Kr, H // 2, ma)
        gamma = _store(d["gamma"], (0, 2, 1))
        got = _call(op, d, logits(lay(d["w"])), logits(_store(d["r"], (0, 2, 1))), lay(d["x"]), gamma, p, mask, Kw, Kr,
                    H // 2, ma)
        for name, a, b in zip(("y", "slot", "mass"), got, want):
            assert torch.equal(a, b), f"{name}: {(a - b).abs().max()}"
    idx, val = torch.ops.ramnet_ops.topk_addr_forward(logits(lay(d["w"])), logits(lay(d["r"])), H // 2, P ** U, pos,
                                                      Kw, Kr, 0.5, 0.25)
    idx0, val0 = torch.ops.ramnet_ops.topk_addr_forward(logits(d["w"]).contiguous(), logits(d["r"]).contiguous(),
                                                        H // 2, P ** U, pos.to(torch.int32), Kw, Kr, 0.5, 0.25)
    assert torch.equal(idx, idx0) and torch.equal(val, val0)


@pytest.mark.parametrize("layout", ["1,8,1,4", "1,8,1,4,1", "2,8,1,4,1,2"])
def test_strided_scan_layouts(monkeypatch, layout):
    """x and y strided in the one-token and paired scans."""
    B, H, U, P, T, C, Kw, Kr = 2, 2, 2, 16, 75, 32, 8, 8
    d = _inputs(B, H, U, P, T, C, torch.bfloat16)
    pos = torch.arange(T, device=DEV).view(1, T).expand(B, T)
    logits = lambda t: t.permute(0, 1, 3, 4, 2)
    op = torch.ops.ramnet_ops.ram_attn_forward
    monkeypatch.setenv("RAMNET_SCAN_LAYOUT", layout)
    want = _call(op, d, logits(d["w"]).contiguous(), logits(d["r"]).contiguous(), d["x"], d["gamma"], pos, d["mask"],
                 Kw, Kr, 1, True)
    got = _call(op, d, logits(d["w"]), logits(d["r"]), _store(d["x"], (0, 2, 1)), d["gamma"], pos, d["mask"], Kw, Kr,
                1, True)
    assert got[0].stride() == _store(d["x"], (0, 2, 1)).stride()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("P,Kw", [(16, 4), (48, 12), (5, 20)], ids=["half", "wave", "general"])
def test_decode_positions(P, Kw):
    """int64 and strided positions in the decode step, the multi-step call
    (one launch, or one a step) and the single decoder."""
    B, H, U, C, S = 3, 2, 2, 16, 3
    d = _inputs(B, H, U, P, S, C, torch.bfloat16)
    w, r = (d[n].permute(2, 0, 1, 3, 4).contiguous() for n in ("w", "r"))
    x, gamma = d["x"].permute(2, 0, 1, 3).contiguous(), d["gamma"].permute(2, 0, 1).contiguous()
    pos = torch.arange(S, device=DEV).view(S, 1) * 5 + torch.arange(B, device=DEV).view(1, B) * 11 - 7
    none = torch.empty(0, dtype=torch.bool, device=DEV)
    ops = torch.ops.ramnet_ops
    outs = []
    # the positions as int32, as int64, as a column-major view and every other word of a wider row
    wide = torch.zeros(S, 2 * B, dtype=torch.int64, device=DEV)
    wide[:, ::2] = pos
    for p in (pos.to(torch.int32), pos, pos.t().contiguous().t(), wide[:, ::2]):
        slot, mass = d["slot"].clone(), d["mass"].clone()
        y = ops.topk_autoregressive_steps_(w, r, x, gamma, slot, mass, none, 1, p, Kw, 3, 0.0, 0.0, True, 1e-6)
        slot1, mass1 = d["slot"].clone(), d["mass"].clone()
        y1 = torch.stack([ops.topk_autoregressive_(w[s], r[s], x[s], gamma[s], slot1, mass1, none, 1, p[s], Kw, 3,
                                                   0.0, 0.0, True, 1e-6) for s in range(S)])
        idx, val = ops.topk_addr_single_forward(w.permute(1, 2, 3, 4, 0), 1, P ** U, p.t(), Kw, 0.5)
        outs.append((y, slot, mass, y1, slot1, mass1, idx, val))
    for other in outs[1:]:
        for a, b in zip(other, outs[0]):
            assert torch.equal(a, b)


@pytest.mark.parametrize("order", list(ORDERS))
@pytest.mark.parametrize("case", [c for c in CASES if c[4] > 1], ids=lambda c: "-".join(str(v).replace("torch.", "") for v in c))
def test_strided_gradients(case, order):
    """Gradients of logits and values in the inputs' layouts: bit for bit those
    of contiguous inputs, fp32 sums rounded once to the inputs' type."""
    B, H, U, P, T, C, Kw, Kr, dtype = case
    d = _inputs(B, H, U, P, T, C, dtype, seed=1)
    lay, ops = ORDERS[order], torch.ops.ramnet_ops
    A = P ** U
    pos = torch.arange(T, device=DEV).view(1, T) * 3 + torch.arange(B, device=DEV).view(B, 1) * 7 - 5
    logits = lambda t: t.permute(0, 1, 3, 4, 2)
    w, r = logits(d["w"]).contiguous(), logits(d["r"]).contiguous()
    idx, val = ops.topk_addr_forward(w, r, H // 2, A, pos, Kw, Kr, 0.5, 0.25)
    dval = torch.randn(val.shape, generator=torch.Generator(device=DEV).manual_seed(2), device=DEV)
    tail = (dval, H // 2, pos, Kw, Kr, 0.5, 0.25, [B, H, U, P, A, T], dtype)
    want = ops.topk_addr_backward(idx, val, w, r, *tail)
    got = ops.topk_addr_backward(idx, val, logits(lay(d["w"])), logits(_store(d["r"], (0, 2, 1))), *tail)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    if nat.segment_saved_bytes(B, H, T, A, C, Kw, Kr, dtype) < 0:
        return
    seg = (d["gamma"], d["slot"], d["mass"])
    y, slot, mass, saved = ops.topk_segment_forward_saved(idx, val, d["x"], *seg, d["mask"], Kw, Kr, True, 1e-6)
    dy = torch.randn(y.shape, generator=torch.Generator(device=DEV).manual_seed(3), device=DEV).to(dtype)
    want = ops.topk_segment_backward_saved(val, d["x"], *seg, saved, dy, None, None, Kw, Kr, True, 1e-6)
    x = lay(d["x"])
    y2, slot2, mass2, saved2 = ops.topk_segment_forward_saved(idx, val, x, *seg, d["mask"], Kw, Kr, True, 1e-6)
    for a, b in zip((y2, slot2, mass2), (y, slot, mass)):
        assert torch.equal(a, b)
    for typed in (False, True):
        got = ops.topk_segment_backward_saved(val, x, *seg, saved2, lay(dy), None, None, Kw, Kr, True, 1e-6, typed)
        assert got[1].dtype == (dtype if typed else torch.float32)
        for k, (a, b) in enumerate(zip(got, want)):
            assert torch.equal(a, b.to(a.dtype)), k


def test_refused_strides():
    """Steps the kernels cannot follow are refused by the native entry."""
    z = torch.zeros(64, device=DEV)
    with pytest.raises(RuntimeError, match="digits must follow"):
        nat.call("ramnet_topk_addr_forward_strided", z.data_ptr(), z.data_ptr(), 0, 1, 1, 2, 2, 2, 0, 4, z.data_ptr(),
                 1, 1, 0.0, 0.0, 1, nat.strides(*(8, 8, 5, 2, 1) * 2, 2, 1), z.data_ptr(), z.data_ptr(), None)
