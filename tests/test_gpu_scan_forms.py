"""Segment forwards whose form is decided near the edges of LDS, against the
fp64 event loop."""
import pytest
import torch

import oracle
from ram_cases import make_case
from ramnet_ops import _native as nat
from test_gpu_parity import FP32_TOL, _out_tol, _segment_case

pytestmark = pytest.mark.gpu


def _check(B, H, U, P, T, C, Kw, Kr, dtype, masked, mass_aware, seed):
    src, (y, slot, mass), (ry, rslot, rmass) = _segment_case(B, H, U, P, T, C, Kw, Kr, dtype, masked, mass_aware, seed)
    ry = torch.as_tensor(ry)
    if src.mask is not None:
        y, ry = y[:, :, src.mask[0]], ry[:, :, src.mask[0]]
    assert oracle.rel_err(slot, rslot) <= FP32_TOL, "slot state"
    assert oracle.rel_err(mass, rmass) <= FP32_TOL, "mass state"
    err = oracle.rel_err(y, ry)
    assert err <= _out_tol(dtype), f"y rel err {err:.3e}"


@pytest.mark.parametrize("mass_aware", [False, True])
@pytest.mark.parametrize("U,P,K", [(3, 23, 16), (2, 113, 8)])
def test_form_depends_on_mass_aware(U, P, K, mass_aware):
    """Slot spaces that only a call that is not mass-aware holds whole: the
    mass-aware one is scanned in slot ranges, whose fp32 read sums (16-bit y)
    the workspace holds."""
    B, H, T, C, A = 1, 2, 48, 24, P ** U
    form, ranges, _ = nat.segment_call_form(B, H, T, A, C, K, K, torch.bfloat16, mass_aware)
    assert (ranges > 1) == mass_aware
    print(f"A={A} K={K} mass_aware={mass_aware} form {form} ranges {ranges}", flush=True)
    _check(B, H, U, P, T, C, K, K, torch.bfloat16, False, mass_aware, seed=A)


def _run(B, H, U, P, T, C, Kw, Kr, dtype, masked, mass_aware, bias):
    """ram_attn_forward with `bias` (1 or B, H, U, P, 1) added to both logits, against the
    event loop on the decoded events; returns them (idx) and the outputs."""
    ops = torch.ops.ramnet_ops
    src = make_case(B, H, U, P, T, C, dtype=dtype, seed=T + P, masked=masked)
    d = src.to("cuda")
    w, r = ((t.float() + bias.to("cuda")).to(dtype) for t in (d.w_addr, d.r_addr))
    idx, val = ops.topk_addr_forward(w, r, 1, P ** U, d.position_ids, Kw, Kr, 0.0, 0.0)
    out = ops.ram_attn_forward(w, r, d.values, d.gamma, d.init_slot, d.init_mass, d.mask, 1, d.position_ids, Kw, Kr,
                               0.0, 0.0, mass_aware, 1e-12)
    y, slot, mass = (t.cpu() for t in out)
    wi, wv, ri, rv = oracle.split_events(idx.cpu(), val.cpu(), Kw)
    ry, rslot, rmass = oracle.sparse_gsu_f64(wi, wv, ri, rv, src.values.double(), src.gamma.double(), src.init_slot,
                                             src.init_mass, src.mask, mass_aware, 1e-12)
    ok = torch.ones(T, dtype=torch.bool) if src.mask is None else src.mask[0]
    assert oracle.rel_err(slot, rslot) <= FP32_TOL, "slot state"
    assert oracle.rel_err(mass, rmass) <= FP32_TOL, "mass state"
    assert oracle.rel_err(y[:, :, ok], torch.as_tensor(ry)[:, :, ok]) <= _out_tol(dtype), "y"
    return idx, out


def _bias(B, H, U, P, scale):
    return scale * torch.randn(B, H, U, P, 1, generator=torch.Generator().manual_seed(3))


@pytest.mark.parametrize("crowded", [False, True], ids=["spread", "crowded"])
@pytest.mark.parametrize("U,P,K,T,mass_aware", [
    (3, 20, 16, 100, False), (3, 20, 8, 300, True),    # A = 8000: no mass-wave layout beside the level form
    (3, 21, 8, 100, False), (2, 100, 8, 100, True),    # A = 9261, 10000
    (3, 22, 16, 300, False),                           # A = 10648: the widest with a whole one-token layout
    (3, 23, 8, 100, False), (3, 23, 16, 300, True)])   # A = 12167: none, scanned in slot ranges
def test_wide_slot_spaces(U, P, K, T, mass_aware, crowded):
    """Calls of more than 64 tokens where the level-scheduled form fits and the
    forms that take crowded addresses do so only in part, or not at all."""
    print(f"A={P ** U} K={K} T={T} {mass_aware} {crowded} "
          f"{nat.segment_call_form(1, 2, T, P ** U, 64, K, K, torch.bfloat16, mass_aware)}", flush=True)
    _run(1, 2, U, P, T, 64, K, K, torch.bfloat16, False, mass_aware, _bias(1, 2, U, P, 4.0 * crowded))
