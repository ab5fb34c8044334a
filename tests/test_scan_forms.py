"""The segment forward's choice of form near the edges of LDS, without a GPU
(``ramnet_segment_call_form`` and the size queries do no device work)."""
from __future__ import annotations

import pytest
import torch

from ramnet_ops import _native as nat

B, H, C = 4, 8, 64
# around the widest slot spaces of the forms that hold them whole: 20**3 .. 23**3, 104**2 .. 116**2, and between
SLOTS = sorted({20 ** 3, 21 ** 3, 22 ** 3, 23 ** 3, *(p * p for p in range(86, 117, 3)), *range(7600, 14000, 173)})


@pytest.mark.parametrize("T", [9, 48, 64, 65, 128, 2048, 8192])
@pytest.mark.parametrize("K", [4, 8, 16])
def test_workspace_holds_every_call(K, T):
    """The workspace size, which does not depend on mass_aware, holds the fp32
    read sums of a call scanned in slot ranges, mass-aware or not."""
    for A in SLOTS:
        ws = nat.segment_workspace_bytes(B, H, T, A, C, K, K, torch.bfloat16)
        for mass_aware in (False, True):
            form, ranges, _ = nat.segment_call_form(B, H, T, A, C, K, K, torch.bfloat16, mass_aware)
            sums = B * H * T * C * 4 if ranges > 1 else 0
            assert ws >= nat.scan_workspace_bytes(B, H, T, K, K) + sums, (A, mass_aware, form, ranges)


# what the planner answers where it takes no level-scheduled form: one token a step, in ranges or not
ONE_TOKEN, LEVEL = (0, 1, 2), 3


@pytest.mark.parametrize("mass_aware", [False, True])
@pytest.mark.parametrize("K", [4, 8, 16, 24])
def test_crowded_calls_have_a_form(K, mass_aware):
    """Every call that may leave crowded addresses to another form has one, and
    wider slot spaces than any whole one-token layout are scanned in ranges."""
    for A in SLOTS:
        for T in (65, 100, 300, 1024, 4096):
            form, ranges, crowded = nat.segment_call_form(B, H, T, A, C, K, K, torch.bfloat16, mass_aware)
            assert crowded in ONE_TOKEN, (A, T, form, ranges, crowded)
            assert (ranges == 1) == (A <= 10912), (A, T, form, ranges)


@pytest.mark.skipif(torch.cuda.is_available(), reason="the calls would launch on pointers that are not memory")
@pytest.mark.parametrize("T,C", [(3072, 32), (3072, 64), (4096, 64), (4096, 128)])
def test_noalloc_takes_records_that_fit(T, C):
    """Decoder records that fit the scratch where the other forms' do not: the
    mass-wave form, which needs no more, takes the call (which here ends for
    want of a device, not at the scratch check)."""
    B, H, U, P, K = 8, 16, 2, 32, 16
    assert nat.scan_workspace_bytes(B, H, T, K, K) > 192 << 20
    fake = 0x1000
    rc = nat.lib().ramnet_ram_attn_forward_noalloc(
        fake, fake, fake, fake, 2, None, 8, fake, fake, fake + 64, fake + 128, fake + 192, fake + 256, B, H, U, P, T,
        P ** U, C, K, K, 0.0, 0.0, 0, 1e-12, None)
    message = nat.lib().ramnet_last_error().decode()
    assert rc != nat.RAMNET_EINVAL and "scratch;" not in message, message
