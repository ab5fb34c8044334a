"""The level-scheduled segment scan (csrc/segment_level.hpp) against the fp64
event loop: every compiled layout, forced through RAMNET_SCAN_LAYOUT
(channels per lane, lanes per token, 1, waves, 1, 3), at the sizes where its
chunks, levels and slices end; and its choice of kernel for crowded calls."""
import pytest
import torch

import oracle
from ram_cases import make_case
from test_gpu_parity import FP32_TOL, _out_tol, _segment_case

pytestmark = pytest.mark.gpu
DEV = "cuda"

LAYOUTS = [(v, w) for v in (4, 2, 1) for w in (1, 2, 4)]
# B, H, U, P, T, Kw, Kr, masked, mass_aware: chunks of 32 tokens (T around
# one and two of them), top-K at and below 4, 8 and 16; A = 16 and 27 put
# most events on a late level, up to one per token
CASES = [
    (1, 2, 2, 16, 2, 4, 4, False, False),
    (2, 1, 2, 16, 31, 3, 4, True, True),
    (1, 2, 2, 32, 32, 8, 8, False, False),
    (2, 2, 2, 16, 33, 1, 5, False, True),
    (1, 3, 2, 4, 64, 8, 8, True, False),
    (2, 1, 3, 16, 65, 16, 16, False, False),
    (1, 2, 3, 3, 100, 16, 9, True, True),
    (1, 2, 2, 24, 97, 6, 2, True, False),
]


def _check(case, dtype, C, seed):
    B, H, U, P, T, Kw, Kr, masked, mass_aware = case
    src, got, ref = _segment_case(B, H, U, P, T, C, Kw, Kr, dtype, masked, mass_aware, seed=seed)
    y, slot, mass = got
    ry, rslot, rmass = ref
    ry = torch.as_tensor(ry)
    if src.mask is not None:
        assert bool((y[:, :, ~src.mask[0]] == 0).all()), "masked tokens must read 0"
        y, ry = y[:, :, src.mask[0]], ry[:, :, src.mask[0]]
    assert oracle.rel_err(slot, rslot) <= FP32_TOL, "slot state"
    assert oracle.rel_err(mass, rmass) <= FP32_TOL, "mass state"
    err = oracle.rel_err(y, ry)
    assert err <= _out_tol(dtype), f"y rel err {err:.3e}"


@pytest.mark.parametrize("partial", [False, True], ids=["full_slices", "partial_slice"])
@pytest.mark.parametrize("layout", LAYOUTS, ids=lambda l: "v{}w{}".format(*l))
def test_level_scan_layouts(layout, partial, monkeypatch):
    vec, nw = layout
    monkeypatch.setenv("RAMNET_SCAN_LAYOUT", f"{vec},2,1,{nw},1,3")
    cs = 2 * vec * nw
    C = 2 * cs + ((1 - cs // 2) if partial and cs > 2 else int(partial))
    for i, case in enumerate(CASES):
        if max(case[5], case[6]) > 8 and vec == 4:
            continue  # not compiled
        if 2 * vec * nw > 8 and case[3] ** case[2] == 4096:
            continue  # more than 8 channels of 4096 slots do not fit in LDS
        dtype = (torch.float32, torch.bfloat16, torch.float16)[i % 3]
        print(f"level scan {layout} C={C} {case} {dtype}", flush=True)
        _check(case, dtype, C, seed=i + C)


@pytest.mark.parametrize("case", [(2, 4, 2, 16, 200, 8, 6, True, True), (1, 2, 2, 16, 5000, 8, 8, False, False)],
                         ids=["short", "long"])
def test_level_scan_crowded(case):
    """Spread addresses, and addresses concentrated on a few slots, which leave
    the call to the mass-wave form launched before the level-scheduled one:
    either way the state and y are those of the event loop. (Which form ran, and
    the pre-pass and paired ones: test_gpu_scan_forms.py.)"""
    B, H, U, P, T, Kw, Kr, masked, mass_aware = case
    import ramnet_ops  # noqa: F401
    ops = torch.ops.ramnet_ops
    src = make_case(B, H, U, P, T, 64, seed=T, masked=masked)
    d = src.to(DEV)
    A = P ** U
    bias = 4 * torch.randn(1, H, U, P, 1, generator=torch.Generator().manual_seed(3)).to(DEV)
    for spread in (True, False):
        w, r = (t if spread else t + bias for t in (d.w_addr, d.r_addr))
        print(f"crowded {case} spread={spread}", flush=True)
        idx, val = ops.topk_addr_forward(w, r, 1, A, d.position_ids, Kw, Kr, 0.0, 0.0)
        y, slot, mass = ops.ram_attn_forward(w, r, d.values, d.gamma, d.init_slot, d.init_mass, d.mask, 1,
                                             d.position_ids, Kw, Kr, 0.0, 0.0, mass_aware, 1e-12)
        wi, wv, ri, rv = oracle.split_events(idx.cpu(), val.cpu(), Kw)
        ry, rslot, rmass = oracle.sparse_gsu_f64(wi, wv, ri, rv, src.values.double(), src.gamma.double(),
                                                 src.init_slot, src.init_mass, src.mask, mass_aware, 1e-12)
        assert oracle.rel_err(slot.cpu(), rslot) <= FP32_TOL
        assert oracle.rel_err(mass.cpu(), rmass) <= FP32_TOL
        ok = torch.ones(T, dtype=torch.bool) if src.mask is None else src.mask[0]
        assert oracle.rel_err(y.cpu()[:, :, ok], torch.as_tensor(ry)[:, :, ok]) <= FP32_TOL


def test_level_scan_unaligned_rows():
    """x and the states at addresses aligned to one element only take the
    element-wise path with the same result."""
    ops = torch.ops.ramnet_ops
    B, H, U, P, T, C, K = 1, 2, 2, 16, 70, 64, 8
    d = make_case(B, H, U, P, T, C, dtype=torch.bfloat16, seed=5).to(DEV)
    args = (d.mask, 1, d.position_ids, K, K, 0.0, 0.0, False, 1e-12)
    want = ops.ram_attn_forward(d.w_addr, d.r_addr, d.values, d.gamma, d.init_slot, d.init_mass, *args)

    def shift(t):
        out = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)[1:].view(t.shape)
        return out.copy_(t)

    got = ops.ram_attn_forward(d.w_addr, d.r_addr, shift(d.values), d.gamma, shift(d.init_slot), shift(d.init_mass), *args)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
