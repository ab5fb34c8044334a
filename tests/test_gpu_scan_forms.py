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


def _run(B, H, U, P, T, C, Kw, Kr, dtype, masked, mass_aware, bias, E=1):
    """ram_attn_forward with `bias` (1 or B, H, U, P, 1) added to both logits, against the
    event loop on the decoded events; returns them (idx) and the outputs."""
    ops = torch.ops.ramnet_ops
    src = make_case(B, H, U, P, T, C, dtype=dtype, seed=T + P, masked=masked)
    d = src.to("cuda")
    w, r = ((t.float() + bias.to("cuda")).to(dtype) for t in (d.w_addr, d.r_addr))
    idx, val = ops.topk_addr_forward(w, r, E, P ** U, d.position_ids, Kw, Kr, 0.0, 0.0)
    out = ops.ram_attn_forward(w, r, d.values, d.gamma, d.init_slot, d.init_mass, d.mask, E, d.position_ids, Kw, Kr,
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


def _late_levels(idx, Kw, A):
    """Late levels of each whole 32-token chunk, (B * H, chunks): the largest number of
    earlier writes in the chunk that an event of it waits for."""
    B, H, K, T = idx.shape
    n = T // 32
    slots = (idx % A).view(B * H, K, T)[:, :, :n * 32].reshape(B * H, K, n, 32).permute(0, 2, 3, 1).long()
    written = torch.zeros(B * H, n, 32, A, dtype=torch.int16, device=idx.device).scatter_(3, slots[..., :Kw], 1)
    upto = written.cumsum(2)
    writes, reads = (upto - written).gather(3, slots[..., :Kw]), upto.gather(3, slots[..., Kw:])
    return torch.maximum(writes.amax((2, 3)), reads.amax((2, 3))).float()


MASS_WAVE, GAINS, PAIRED, LEVEL = range(4)


@pytest.mark.parametrize("addresses", ["spread", "crowded", "one_head"])
@pytest.mark.parametrize("B,H,U,P,T,C,Kw,Kr,masked,mass_aware,other", [
    (2, 2, 2, 16, 250, 64, 8, 6, True, True, MASS_WAVE),      # few chunks: each wave counts them
    (1, 6, 3, 14, 333, 32, 16, 16, False, False, MASS_WAVE),  # the same, a part of a chunk and of a window
    (4, 8, 2, 16, 400, 16, 8, 8, False, False, MASS_WAVE),    # more: one workgroup counts
    (2, 8, 3, 16, 300, 128, 8, 8, False, False, PAIRED),
    (2, 8, 3, 16, 300, 128, 16, 9, True, True, PAIRED),
    (1, 4, 3, 20, 300, 64, 8, 8, False, False, GAINS)])
def test_crowded_addresses(B, H, U, P, T, C, Kw, Kr, masked, mass_aware, other, addresses):
    """Spread addresses take the level-scheduled form; crowded ones, also those
    of one head among many, the form beside it. In fp32 the two forms sum a read in
    different orders, so the bits of y say which one ran: the level form's do not
    depend on its layout."""
    A = P ** U
    assert nat.segment_call_form(B, H, T, A, C, Kw, Kr, torch.float32, mass_aware) == (LEVEL, 1, other)
    bias = _bias(1, H, U, P, 8.0).repeat(B, 1, 1, 1, 1)
    if addresses == "spread":
        bias = bias * 0
    elif addresses == "one_head":
        bias[:, :-1], bias[:-1] = 0, 0
    print(f"{(B, H, U, P, T, C, Kw, Kr, masked, mass_aware)} {addresses}", flush=True)
    idx, (y, slot, mass) = _run(B, H, U, P, T, C, Kw, Kr, torch.float32, masked, mass_aware, bias, E=0)
    late = _late_levels(idx, Kw, A).mean(1)
    print(f"late levels a chunk: {late.tolist()}", flush=True)
    assert late.max() <= 5 if addresses == "spread" else late.max() >= 30
    assert (late >= 30).all() == (addresses == "crowded")
    with pytest.MonkeyPatch.context() as env:
        env.setenv("RAMNET_SCAN_LAYOUT", "1,2,1,1,1,3")
        _, (level_y, _, _) = _run(B, H, U, P, T, C, Kw, Kr, torch.float32, masked, mass_aware, bias, E=0)
    assert torch.equal(y, level_y) == (addresses == "spread")


def test_crowded_call_in_place_and_captured():
    """A crowded call that updates its state in place, captured and replayed
    with eager spread calls between the replays: each replay decides by its own
    addresses."""
    ops = torch.ops.ramnet_ops
    B, H, U, P, T, C, K = 2, 8, 3, 16, 300, 128, 8
    d = make_case(B, H, U, P, T, C, seed=2).to("cuda")
    bias = _bias(1, H, U, P, 8.0).to("cuda")
    w, r = d.w_addr.clone(), d.r_addr.clone()
    slot, mass = d.init_slot.clone(), d.init_mass.clone()
    args = (None, 1, d.position_ids, K, K, 0.0, 0.0, False, 1e-12)

    def call(slot, mass):
        return ops.ram_attn_forward_(w, r, d.values, d.gamma, slot, mass, *args)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(slot.clone(), mass.clone())
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = call(slot, mass)
    for replay, scale in enumerate((1.0, 0.0, 1.0, 0.0)):
        w.copy_(d.w_addr + scale * bias)
        r.copy_(d.r_addr + scale * bias)
        slot.copy_(d.init_slot)
        mass.copy_(d.init_mass)
        want_slot, want_mass = slot.clone(), mass.clone()
        want = call(want_slot, want_mass)
        graph.replay()
        torch.cuda.synchronize()
        for name, a, b in zip(("y", "slot", "mass"), (y, slot, mass), (want, want_slot, want_mass)):
            assert torch.equal(a, b), f"replay {replay}: {name}"
