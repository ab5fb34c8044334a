"""Segment forwards whose form is decided near the edges of LDS, against the
fp64 event loop."""
import pytest
import torch

import oracle
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
    form, ranges = nat.segment_call_form(B, H, T, A, C, K, K, torch.bfloat16, mass_aware)
    assert (ranges > 1) == mass_aware
    print(f"A={A} K={K} mass_aware={mass_aware} form {form} ranges {ranges}", flush=True)
    _check(B, H, U, P, T, C, K, K, torch.bfloat16, False, mass_aware, seed=A)
