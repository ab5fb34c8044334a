"""The direct route of ``random_access_memory_attention`` for calls without
broadcasting against the general route: the same outputs, strides of the
state, aliasing and gradients where it is taken, and the same errors where an
argument is wrong.
"""
from __future__ import annotations

import pytest
import torch

import ramnet_ops.ram_attn as api

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
B, H, U, P, C = 2, 3, 2, 4, 8
A = P ** U


def _args(T, dtype=torch.float32, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    return dict(w_addr=rnd(B, T, H, U, P).to(dtype), r_addr=rnd(B, T, H, U, P).to(dtype),
                values=rnd(B, T, H, C).to(dtype), gamma=rnd(B, T, H).to(dtype),
                init_ram=(rnd(B, H, A, C), torch.rand(B, H, A, generator=g, device=DEV) + 0.1),
                position_ids=torch.arange(T, device=DEV).view(1, T).expand(B, T) + 3,
                mask=torch.rand(B, T, generator=g, device=DEV) > 0.3, embed_num=2, top_k=(3, 2),
                top_k_re_norm=(0.5, 0.0), mass_aware=True, eps=1e-6)


FORMS = {
    "full": {},
    "defaults": dict(init_ram=None, position_ids=None, mask=None, top_k=4, top_k_re_norm=0.0),
    "slot_only": lambda a: dict(init_ram=(a["init_ram"][0], None)),
    "mass_only": lambda a: dict(init_ram=(None, a["init_ram"][1])),
    "scalar_mass": lambda a: dict(init_ram=(a["init_ram"][0], 0.25)),
    "scalar_gamma": dict(gamma=-0.5),
    "list_pairs": dict(top_k=[2, 5], top_k_re_norm=[0.25, 1]),
    "int_mask": lambda a: dict(mask=a["mask"].to(torch.int64)),
    "cpu_positions": lambda a: dict(position_ids=a["position_ids"].cpu(), mask=a["mask"].cpu()),
    "double_state": lambda a: dict(init_ram=tuple(t.double() for t in a["init_ram"])),
    "broadcast_batch": lambda a: dict(w_addr=a["w_addr"][:1], position_ids=a["position_ids"][:1]),
    "inplace": dict(inplace=True),
    "grad": "grad",
    "bad_gamma_shape": lambda a: dict(gamma=a["gamma"][:, :, :2]),
    "bad_gamma_dtype": lambda a: dict(gamma=a["gamma"].double()),
    "bad_top_k": dict(top_k=A + 1),
    "zero_top_k": dict(top_k=(0, 1)),
    "bad_re_norm": dict(top_k_re_norm=1.5),
    "bad_embed": dict(embed_num=H + 1),
    "bad_eps": dict(eps=0.0),
    "bad_slots": lambda a: dict(init_ram=(a["init_ram"][0][:, :, :-1], a["init_ram"][1])),
    "bad_mask": lambda a: dict(mask=a["mask"][:, :0]),
    "strided_inplace": lambda a: dict(inplace=True, init_ram=(a["init_ram"][0].transpose(0, 1).contiguous().transpose(0, 1),
                                                              a["init_ram"][1])),
    "half_inplace": lambda a: dict(inplace=True, init_ram=tuple(t.half() for t in a["init_ram"])),
    "empty_batch": lambda a: dict(**{n: a[n][:0] for n in ("w_addr", "r_addr", "values", "gamma", "position_ids", "mask")},
                                  init_ram=tuple(t[:0] for t in a["init_ram"])),
    "double_values": lambda a: {n: a[n].double() for n in ("w_addr", "r_addr", "values", "gamma")},
}


def _outcome(T, form):
    a = _args(T)
    if form == "grad":
        leaves = [a[n].requires_grad_() for n in ("w_addr", "r_addr", "values", "gamma")]
        y, (slot, mass) = api.random_access_memory_attention(**a)
        return [y, slot, mass, *torch.autograd.grad((y.sum() + slot.square().sum() + mass.sum()), leaves)]
    a.update(form(a) if callable(form) else form)
    try:
        y, (slot, mass) = api.random_access_memory_attention(**a)
    except (AssertionError, RuntimeError, ValueError, TypeError) as e:
        return type(e), str(e)
    out = [y, slot, mass]
    if a.get("inplace"):
        assert slot.data_ptr() == a["init_ram"][0].data_ptr() and mass.data_ptr() == a["init_ram"][1].data_ptr()
        out += list(a["init_ram"])
    return out


def _steps(t):
    """Strides of the dimensions that have more than one element."""
    return [s for s, n in zip(t.stride(), t.shape) if n > 1]


@pytest.mark.parametrize("T", [1, 5])
@pytest.mark.parametrize("form", list(FORMS))
def test_plain_equals_general(monkeypatch, form, T):
    got = _outcome(T, FORMS[form])
    monkeypatch.setattr(api, "_plain_call", lambda *a: None)
    want = _outcome(T, FORMS[form])
    assert isinstance(got, type(want)) and len(got) == len(want)
    for a, b in zip(got, want):
        if isinstance(b, torch.Tensor):
            assert a.dtype == b.dtype and a.shape == b.shape and _steps(a) == _steps(b) and torch.equal(a, b)
        else:
            assert a == b
    if form.startswith(("bad", "zero", "strided", "half", "double_values")):
        assert isinstance(want, tuple), "this form is refused"
