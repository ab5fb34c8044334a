"""Timed workloads of the RAM-Net operators on one GPU.

Each case is a plain dict; ``prepare`` makes its inputs on the GPU, ``run``
makes one pass through the public entry points (``ramnet_ops`` and the layer
of ``ramnet_harness``), ``exact`` restates the same pass in float64 torch.

Kinds of case:
  prefill       random_access_memory_attention over a whole sequence, no gradients
  train         the same with gradients: forward and backward
  decode        one token per sequence, the state updated in place
  decode_graph  consecutive decode calls captured in one HIP graph, replayed
  decode_steps  the multi-step decode operator (replay and verification of known tokens)
  addresses     topk_addr alone
  layer         the language model's RAM layer over a prompt (projections,
                operator, read-out norm, gate, output projection)

Tensors are laid out as a model's projections give them: addresses
(B, T, H, U, P), values (B, T, H, C), gamma (B, T, H), time in dimension 1.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ram-net_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
_EPS = 1e-12


def _case(name, kind, B, T, H, U, P, C, Kw, Kr, dtype, **more):
    case = dict(name=name, kind=kind, B=B, T=T, H=H, U=U, P=P, C=C, Kw=Kw, Kr=Kr, dtype=dtype, embed=H // 2,
                masked=False, mass_aware=False, re_norm=0.0, state="none", shift=0.0)
    case.update(more)
    return case


def listed():
    return [
        # a short single-sequence fp32 call, as in unit-size models and tests: launches and latency
        _case("prefill_small_fp32", "prefill", 1, 256, 4, 2, 16, 64, 4, 4, "fp32"),
        # the main prefill: eight 4096-token prompts, 1024 slots per head, fresh state
        _case("prefill_bf16", "prefill", 8, 4096, 16, 2, 32, 128, 8, 8, "bf16", state="given", shift=-1.0),
        # large slot space: three digits, 4096 slots, top-16, long sequences
        _case("prefill_large_state", "prefill", 4, 8192, 8, 3, 16, 128, 16, 16, "bf16", state="given"),
        # a serving chunk: ragged left-padded batch continuing a live state in place, mass-aware
        # re-normalised reads, unequal top-K, sizes that divide nothing
        _case("prefill_ragged_fp16", "prefill", 3, 1237, 6, 2, 24, 80, 6, 5, "fp16", masked=True, mass_aware=True,
              re_norm=1.0, state="inplace"),
        # eager batch decode
        _case("decode_batch", "decode", 64, 1, 16, 2, 32, 128, 8, 8, "bf16", state="inplace"),
        # one user, the language model's heads: the smallest call there is
        _case("decode_single", "decode", 1, 1, 8, 2, 32, 128, 8, 8, "bf16", state="inplace"),
        # a serving loop: 32 consecutive single-token calls captured once, replayed
        _case("decode_graph", "decode_graph", 64, 32, 16, 2, 32, 128, 8, 8, "bf16", state="inplace"),
        # replay of 64 known tokens per sequence in one call
        _case("decode_steps", "decode_steps", 64, 64, 16, 2, 32, 128, 8, 8, "bf16", state="inplace"),
        # the operator's training step at the main prefill size
        _case("train_bf16", "train", 8, 4096, 16, 2, 32, 128, 8, 8, "bf16", state="given", shift=-1.0),
        # truncated back-propagation over a masked fp32 chunk: gradients through the carried state too
        _case("train_chunk_fp32", "train", 2, 1024, 8, 3, 12, 96, 12, 10, "fp32", masked=True, mass_aware=True,
              re_norm=0.5, state="grad"),
        # address decoding alone (analysis of what a head reads), fp32 logits
        _case("addresses_fp32", "addresses", 4, 2048, 16, 2, 32, 128, 16, 16, "fp32", re_norm=1.0),
        # one RAM layer of the 350M-parameter model over its 16 x 2048 prompt
        _case("layer_bf16", "layer", 16, 2048, 8, 2, 32, 128, 8, 8, "bf16", state="given"),
    ]


def _unnamed(case):
    return {k: v for k, v in case.items() if k != "name"}


def draw(rng):
    """One more case of the same ranges, no dearer than the largest listed one."""
    kind = rng.choice(["prefill", "prefill", "prefill", "train", "train", "decode", "decode_graph", "decode_steps",
                       "addresses", "layer"])

    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    U = rng.choice([2, 2, 3])
    P = rng.choice([16, 32, 32, 64, rng.randint(5, 64)]) if U == 2 else rng.choice([8, 16, rng.randint(4, 16)])
    A = P ** U
    H = rng.choice([4, 8, 16, rng.randint(1, 16)])
    C = rng.choice([64, 128, 128, 8 * rng.randint(4, 24), rng.randint(20, 160)])
    Kw = min(A, rng.choice([4, 8, 8, 16, rng.randint(2, 16)]))
    Kr = Kw if rng.random() < 0.7 else min(A, rng.randint(2, 16))
    more = dict(re_norm=rng.choice([0.0, 0.0, 1.0, 0.5]), mass_aware=rng.random() < 0.25, masked=rng.random() < 0.25,
                embed=rng.choice([0, H // 2, H]), shift=rng.choice([-1.0, 0.0]))
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if kind.startswith("decode"):
        B = spread(1, 96)
        while B * H * A * C > 64 * 16 * 1024 * 128:
            B = max(1, B // 2)
        T = 1 if kind == "decode" else rng.randint(4, 48)
        more["masked"] = False
        return _unnamed(_case("", kind, B, T, H, U, P, C, Kw, Kr, dtype, state="inplace", **more))
    if kind == "layer":
        more.update(masked=False, mass_aware=False, re_norm=0.0, shift=0.0)
        dtype, Kr = "bf16", Kw
        C = max(16, C // 8 * 8)
    T = spread(16, 8192)
    # the main prefill's events and state bound every drawn case
    most = 8 * 16 * 4096 * 16 * 128 // (2 if kind == "train" else 1)
    B = spread(1, 16)
    while B > 1 and (B * H * T * (Kw + Kr) * C > most or B * H * A * C > 8 * 16 * 1024 * 128):
        B //= 2
    while B * H * T * (Kw + Kr) * C > most or (kind == "layer" and B * T > 65536):
        T //= 2
    state = {"prefill": rng.choice(["none", "given", "inplace"]), "train": rng.choice(["given", "grad"]),
             "layer": "given", "addresses": "none"}[kind]
    return _unnamed(_case("", kind, B, T, H, U, P, C, Kw, Kr, dtype, state=state, **more))


# --------------------------------------------------------------------------
# inputs

def _logits(c, n_b, n_t, gen, dev):
    """Write and read address logits (n_b, n_t, H, U, P): q W / sqrt(U), q ~ N(0, 1), W ~ N(0, 1 / d) per head."""
    H, U, P, d = c["H"], c["U"], c["P"], 128
    W = torch.randn(H, d, U * P, generator=gen, device=dev) / math.sqrt(d)
    out = []
    for _ in range(2):
        q = torch.randn(H, n_b * n_t, d, generator=gen, device=dev)
        lg = torch.bmm(q, W) / math.sqrt(U)
        out.append(lg.view(H, n_b, n_t, U, P).permute(1, 2, 0, 3, 4).contiguous().to(_DTYPES[c["dtype"]]))
    return out


def _inputs(c, seed):
    dev = torch.device("cuda")
    dt = _DTYPES[c["dtype"]]
    g = torch.Generator(device=dev).manual_seed(1000003 * (seed + 1) % (2 ** 31))
    B, T, H, P, U, C = c["B"], c["T"], c["H"], c["P"], c["U"], c["C"]
    A = P ** U
    s = {"case": c}
    s["w"], s["r"] = _logits(c, B, T, g, dev)
    s["x"] = torch.randn(B, T, H, C, generator=g, device=dev).to(dt)
    s["gamma"] = torch.sigmoid(torch.randn(B, T, H, generator=g, device=dev) + c["shift"]).to(dt)
    if c["kind"].startswith("decode"):
        s["slot"] = torch.randn(B, H, A, C, generator=g, device=dev).mul_(0.5)
        s["mass"] = torch.rand(B, H, A, generator=g, device=dev) + 1.0 / A
        first = torch.randint(0, 8192, (B, 1), generator=g, device=dev)
        s["pos"] = first + torch.arange(T, device=dev).view(1, T)
        return s
    s["mask"] = None
    s["pos"] = torch.arange(T, device=dev).view(1, T).expand(B, T)
    if c["masked"]:  # left padding of each sequence, up to a quarter of the call
        pad = torch.randint(0, max(2, T // 4), (B, 1), generator=g, device=dev)
        s["mask"] = torch.arange(T, device=dev).view(1, T) >= pad
        s["pos"] = (s["mask"].long().cumsum(-1) - 1).clamp_(min=0)
    if c["state"] in ("inplace", "grad"):  # carried over from the sequence so far
        s["slot"] = torch.randn(B, H, A, C, generator=g, device=dev).mul_(0.5)
        s["mass"] = torch.rand(B, H, A, generator=g, device=dev) + 1.0 / A
    elif c["state"] == "given":  # a new sequence's state
        s["slot"] = torch.zeros(B, H, A, C, device=dev)
        s["mass"] = torch.full((B, H, A), 1.0 / A, device=dev)
    return s


def _layer(c, seed):
    from ramnet_harness.lm import HarnessConfig, RamLayer
    torch.manual_seed(seed + 77)
    cfg = HarnessConfig(layers=1, d_model=1024, heads=c["H"], value_chs=c["C"], addr_order=c["U"], addr_radix=c["P"],
                        top_k=c["Kw"], embed_num=c["embed"])
    with torch.device("cuda"):
        layer = RamLayer(cfg)
        layer.init_weights()
    return layer.to(torch.bfloat16)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "layer":
        dev = torch.device("cuda")
        B, T, A = c["B"], c["T"], c["P"] ** c["U"]
        layer = _layer(c, seed)
        g = torch.Generator(device=dev).manual_seed(seed + 5)
        x = torch.randn(B, T, 1024, generator=g, device=dev).to(torch.bfloat16)
        return {"case": c, "layer": layer, "x": x, "pos": torch.arange(T, device=dev).view(1, T).expand(B, T),
                "slot": torch.zeros(B, c["H"], A, c["C"], device=dev),
                "mass": torch.full((B, c["H"], A), 1.0 / A, device=dev)}
    s = _inputs(c, seed)
    if kind == "addresses":
        s["addr"] = s["w"].permute(0, 2, 3, 4, 1).contiguous()  # topk_addr takes (B, H, U, P, T)
    elif kind == "train":
        for n in ("w", "r", "x", "gamma"):
            s[n].requires_grad_()
        g = torch.Generator(device="cuda").manual_seed(seed + 9)
        s["dy"] = torch.randn(s["x"].shape, generator=g, device="cuda").to(s["x"].dtype)
        if c["state"] == "grad":
            s["slot"].requires_grad_()
            s["mass"].requires_grad_()
            s["dslot"] = 0.1 * torch.randn(s["slot"].shape, generator=g, device="cuda")
            s["dmass"] = 0.1 * torch.randn(s["mass"].shape, generator=g, device="cuda")
    elif kind == "decode_steps":  # step-major, as the operator takes them
        for n in ("w", "r", "x", "gamma"):
            s[n] = s[n].transpose(0, 1).contiguous()
        s["pos"] = s["pos"].transpose(0, 1).contiguous()
        s["no_mask"] = torch.empty(0, dtype=torch.bool, device="cuda")
    elif kind == "decode_graph":
        steps = [{n: s[n][:, t:t + 1].contiguous() for n in ("w", "r", "x", "gamma", "pos")} for t in range(c["T"])]
        slot, mass = s["slot"].clone(), s["mass"].clone()
        with torch.no_grad():
            _attend(c, slot=slot, mass=mass, inplace=True, **steps[0])  # loads the kernels
            del slot, mass
            torch.cuda.synchronize()
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"]):
                s["ys"] = [_attend(c, slot=s["slot"], mass=s["mass"], inplace=True, **st)[0] for st in steps]
        s["steps"] = steps
    return s


# --------------------------------------------------------------------------
# one pass

def _attend(c, w, r, x, gamma, pos, slot=None, mass=None, mask=None, inplace=False):
    from ramnet_ops import random_access_memory_attention
    return random_access_memory_attention(
        w, r, x, gamma, init_ram=None if slot is None else (slot, mass), mask=mask, embed_num=c["embed"],
        position_ids=pos, top_k=(c["Kw"], c["Kr"]), top_k_re_norm=c["re_norm"], mass_aware=c["mass_aware"], eps=_EPS,
        t_dim=1, inplace=inplace)


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "train":
        y, (slot, mass) = _attend(c, s["w"], s["r"], s["x"], s["gamma"], s["pos"], s["slot"], s["mass"], s["mask"])
        ins = [s["w"], s["r"], s["x"], s["gamma"]]
        if c["state"] == "grad":
            grads = torch.autograd.grad((y, slot, mass), ins + [s["slot"], s["mass"]], (s["dy"], s["dslot"], s["dmass"]))
        else:
            grads = torch.autograd.grad(y, ins, s["dy"])
        return [y.detach(), slot.detach(), mass.detach(), *grads]
    with torch.no_grad():
        if kind in ("prefill", "decode"):
            y, (slot, mass) = _attend(c, s["w"], s["r"], s["x"], s["gamma"], s["pos"], s.get("slot"), s.get("mass"),
                                      s.get("mask"), inplace=c["state"] == "inplace")
            return [y, slot, mass]
        if kind == "decode_graph":
            s["graph"].replay()
            return [*s["ys"], s["slot"], s["mass"]]
        if kind == "decode_steps":
            import ramnet_ops  # noqa: F401  (registers the operators)
            y = torch.ops.ramnet_ops.topk_autoregressive_steps_(
                s["w"], s["r"], s["x"], s["gamma"], s["slot"], s["mass"], s["no_mask"], c["embed"], s["pos"], c["Kw"],
                c["Kr"], c["re_norm"], c["re_norm"], c["mass_aware"], _EPS)
            return [y, s["slot"], s["mass"]]
        if kind == "addresses":
            from ramnet_ops import topk_addr
            idx, val = topk_addr(s["addr"], c["embed"], s["pos"], c["Kw"], c["re_norm"])
            return [idx, val]
        y, (slot, mass) = s["layer"](s["x"], (s["slot"], s["mass"]), s["pos"], False)
        return [y, slot, mass]


# --------------------------------------------------------------------------
# what a pass cannot do without

def work(case):
    c = case
    B, T, H, U, P, C = (c[k] for k in ("B", "T", "H", "U", "P", "C"))
    A, n = P ** U, B * T * H
    es = 4 if c["dtype"] == "fp32" else 2
    logits, vals = 2 * n * U * P * es, n * C * es
    tables = B * H * A * (C + 1) * 4
    search = 2 * n * U * P * 4
    rows = n * C * (3 * c["Kw"] + 2 * c["Kr"])
    if c["kind"] == "addresses":
        return {"bytes": logits // 2 + B * T * 8 + n * c["Kw"] * 8, "flops": search // 2}
    if c["kind"] == "layer":
        d = 1024
        wide = H * (2 * U * P + 3 * C + 1)
        return {"bytes": 2 * B * T * d * 2 + wide * d * 2 + 2 * tables, "flops": 2 * B * T * d * wide + search + rows}
    if c["kind"].startswith("decode"):
        # a token moves the rows it writes (read and stored) and the rows it reads
        return {"bytes": logits + 2 * vals + n * (es + 8) + n * (C + 1) * 4 * (2 * c["Kw"] + c["Kr"]),
                "flops": search + rows}
    state_in = 0 if c["state"] == "none" else tables
    fwd = logits + 2 * vals + n * es + B * T * 8 + state_in + tables
    if c["kind"] == "prefill":
        return {"bytes": fwd, "flops": search + rows}
    bwd = logits + vals + n * es + vals  # gradients of the inputs, and dy
    if c["state"] == "grad":
        bwd += 2 * tables
    return {"bytes": fwd + bwd, "flops": 3 * (search + rows)}


def tolerance(case):
    # Measured against exact(): fp32 outputs and gradients 1e-7 to 5e-7 in sequences of 256 to 2000 tokens. 16-bit
    # outputs are one rounding of an fp32 value (rel 1.7e-3 in bf16), so two implementations that select the same
    # slots differ by less than twice that. (Against exact() they show 1e-2 to 3e-2 instead: 16-bit logits tie exactly
    # between candidate slots, and fp32 scores order such ties by their rounding.)
    kind, dt = case["kind"], case["dtype"]
    if kind == "addresses":
        return {"rel": 1e-5, "max": 1e-4, "differ": 1e-3}
    if dt == "fp32":
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 1e-2, "max": 0.1}


# --------------------------------------------------------------------------
# the same pass in float64

def _select(lg, K):
    """Top-K (score desc, content index asc) of (..., U, P) float64 logits: scores and content indices (..., K)."""
    lp = torch.log_softmax(lg, -1)
    U, P = lg.shape[-2:]
    score = content = None
    for u in range(U):
        v, d = torch.sort(lp[..., u, :], dim=-1, descending=True, stable=True)
        v, d = v[..., :K], d[..., :K]
        if score is None:
            score, content = v, d
        else:
            s2 = (score.unsqueeze(-1) + v.unsqueeze(-2)).flatten(-2)
            c2 = (content.unsqueeze(-1) + P ** u * d.unsqueeze(-2)).flatten(-2)
            c2, order = torch.sort(c2, dim=-1)
            s2 = s2.gather(-1, order)
            s2, order = torch.sort(s2, dim=-1, descending=True, stable=True)
            score, content = s2[..., :K], c2.gather(-1, order)[..., :K]
    return score, content


def _weights(lg, content, re_norm):
    """exp(score - re_norm * logsumexp(score)) of given content indices, differentiable in lg."""
    P = lg.shape[-1]
    lp = torch.log_softmax(lg, -1)
    score = sum(lp[..., u, :].gather(-1, content // P ** u % P) for u in range(lg.shape[-2]))
    return torch.exp(score - re_norm * torch.logsumexp(score, -1, keepdim=True))


def _events(c, lg, pos, K):
    lg = lg.detach().double()
    parts = [_select(lg[b:b + 1], K)[1] for b in range(lg.shape[0])]
    content = torch.cat(parts)
    A = c["P"] ** c["U"]
    cape = (torch.arange(c["H"], device=lg.device) < c["embed"]).view(1, 1, -1, 1)
    slot = torch.where(cape, (content - pos.view(*pos.shape, 1, 1)) % A, content)
    return lg, content, slot


def _recur(c, w, r, x, gamma, pos, slot, mass, mask, keep=None):
    """The recurrence over T: y, slot, mass (float64), and per-step tensors in `keep`."""
    B, T, H = x.shape[:3]
    A, C, N = c["P"] ** c["U"], c["C"], x.shape[0] * x.shape[2]
    dev = x.device
    S = torch.zeros(N * A, C, dtype=torch.float64, device=dev) if slot is None else slot.detach().double().reshape(N * A, C)
    S = S.clone()
    # a given scalar or a missing mass is held in the values' type
    M = mass.detach().double().reshape(N * A).clone() if mass is not None else \
        torch.full((N * A,), 1.0 / A, dtype=x.dtype, device=dev).double()
    lw, cw, iw = _events(c, w, pos, c["Kw"])
    lr, cr, ir = _events(c, r, pos, c["Kr"])
    off = (torch.arange(N, device=dev) * A).view(1, B, H, 1)
    iw, ir = iw.transpose(0, 1) + off, ir.transpose(0, 1) + off  # (T, B, H, K)
    vw = torch.cat([_weights(lw[b:b + 1], cw[b:b + 1], c["re_norm"]) for b in range(B)]).transpose(0, 1)
    vr = torch.cat([_weights(lr[b:b + 1], cr[b:b + 1], c["re_norm"]) for b in range(B)]).transpose(0, 1)
    if mask is not None:
        on = mask.transpose(0, 1).view(T, B, 1, 1)
        vw, vr = vw * on, vr * on
    iw, ir, vw, vr = (t.reshape(T, N, -1) for t in (iw, ir, vw, vr))
    q = torch.exp(gamma.detach().double().transpose(0, 1).reshape(T, N, 1))
    den = 1 - vw + q * vw
    alpha = (1 - vw) / den
    xs = x.detach().transpose(0, 1).reshape(T, N, 1, C)
    ys = torch.empty(T, N, C, dtype=torch.float64, device=dev)
    for t in range(T):
        i, v = iw[t], vw[t]
        m0 = M[i]
        m1 = alpha[t] * m0 + v
        M[i] = m1
        g = v / (m1 + _EPS)
        diff = xs[t].double() - S[i]
        S[i] += g.unsqueeze(-1) * diff
        j, e = ir[t], vr[t]
        mr = None
        if c["mass_aware"]:
            mr = M[j]
            e = e.sum(-1, keepdim=True) * (mr * e) / ((mr * e).sum(-1, keepdim=True) + _EPS)
        rows = S[j]
        ys[t] = (e.unsqueeze(-1) * rows).sum(1)
        if keep is not None:
            keep.append((m0, m1, g, diff, mr, e, rows))
    if keep is not None:
        keep.insert(0, (iw, ir, vw, vr, q, den, alpha, xs, lw, cw, lr, cr))
    y = ys.view(T, B, H, C).transpose(0, 1)
    return y, S.view(B, H, A, C), M.view(B, H, A)


def _gradients(c, s, keep):
    """Gradients of w, r, x, gamma (and the initial state) from the recurrence's kept steps."""
    iw, ir, vw, vr, q, den, alpha, xs, lw, cw, lr, cr = keep[0]
    B, T, H, C = s["x"].shape
    A, N = c["P"] ** c["U"], B * H
    dev = xs.device
    f64 = dict(dtype=torch.float64, device=dev)
    DS = s["dslot"].double().reshape(N * A, C).clone() if "dslot" in s else torch.zeros(N * A, C, **f64)
    DM = s["dmass"].double().reshape(N * A).clone() if "dmass" in s else torch.zeros(N * A, **f64)
    dvw, dvr = torch.zeros_like(vw), torch.zeros_like(vr)
    dx, dg = torch.zeros(T, N, C, **f64), torch.zeros(T, N, **f64)
    dys = s["dy"].transpose(0, 1).reshape(T, N, 1, C)
    on = torch.ones(T, N, 1, **f64) if s["mask"] is None else \
        s["mask"].transpose(0, 1).view(T, B, 1).expand(T, B, H).reshape(T, N, 1).double()
    for t in range(T - 1, -1, -1):
        m0, m1, g, diff, mr, e, rows = keep[t + 1]
        dy = dys[t].double() * on[t].unsqueeze(-1)
        d = (dy * rows).sum(-1)
        DS[ir[t]] += e.unsqueeze(-1) * dy
        if mr is not None:
            rsum, nj = vr[t].sum(-1, keepdim=True), mr * vr[t]
            nsum = nj.sum(-1, keepdim=True) + _EPS
            share = (d * nj).sum(-1, keepdim=True) / nsum
            dn = rsum * (d - share) / nsum
            dvr[t] = (share + mr * dn) * on[t]
            DM[ir[t]] += vr[t] * dn
        else:
            dvr[t] = d
        Ds = DS[iw[t]]
        Dg = (Ds * diff).sum(-1)
        dx[t] = (g.unsqueeze(-1) * Ds).sum(1)
        DS[iw[t]] = (1 - g).unsqueeze(-1) * Ds
        dm1 = DM[iw[t]] - Dg * g / (m1 + _EPS)
        da = dm1 * m0
        DM[iw[t]] = alpha[t] * dm1
        dvw[t] = (Dg / (m1 + _EPS) + dm1 - da * q[t] / den[t] ** 2) * on[t]
        dg[t] = (-da * (1 - vw[t]) * q[t] * vw[t] / den[t] ** 2).sum(-1)
    out = []
    for lg, content, dv in ((lw, cw, dvw), (lr, cr, dvr)):
        dv = dv.view(T, B, H, -1).transpose(0, 1)
        parts = []
        for b in range(B):
            leaf = lg[b:b + 1].clone().requires_grad_()
            with torch.enable_grad():
                parts.append(torch.autograd.grad(_weights(leaf, content[b:b + 1], c["re_norm"]), leaf, dv[b:b + 1])[0])
        out.append(torch.cat(parts))
    out.append(dx.view(T, B, H, C).transpose(0, 1))
    out.append(dg.view(T, B, H).transpose(0, 1))
    if c["state"] == "grad":
        out += [DS.view(B, H, A, C), DM.view(B, H, A)]
    return out


@torch.no_grad()
def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "layer":
        # the projections as the layer's own bf16 torch modules give them (inputs of the operator); the rest in float64
        s = prepare(c, seed)
        layer = s["layer"]
        w, r, v, g = layer.op_inputs(s["x"])
        y, slot, mass = _recur(c, w, r, v, g, s["pos"], s["slot"], s["mass"], None)
        y = y / torch.sqrt((y * y).mean(-1, keepdim=True) + layer.cfg.norm_eps) * layer.out_norm.weight.double()
        gate = torch.sigmoid(layer.gate(s["x"]).double())
        return [(gate * y.flatten(-2)) @ layer.out.weight.double().t(), slot, mass]
    if kind == "train":
        s = prepare(c, seed)
        if s["x"].numel() * 16 * (c["Kw"] + c["Kr"]) > 100e9:
            return None
        keep = []
        y, slot, mass = _recur(c, s["w"], s["r"], s["x"], s["gamma"], s["pos"], s["slot"], s["mass"], s["mask"], keep)
        return [y, slot, mass, *_gradients(c, s, keep)]
    s = _inputs(c, seed)
    if kind == "addresses":
        lg, content, slot = _events(c, s["w"], s["pos"], c["Kw"])
        val = torch.cat([_weights(lg[b:b + 1], content[b:b + 1], c["re_norm"]) for b in range(c["B"])])
        off = (torch.arange(c["B"] * c["H"], device=lg.device) * c["P"] ** c["U"]).view(c["B"], 1, c["H"], 1)
        return [(slot + off).permute(0, 2, 3, 1), val.permute(0, 2, 3, 1)]
    y, slot, mass = _recur(c, s["w"], s["r"], s["x"], s["gamma"], s["pos"], s.get("slot"), s.get("mass"), s.get("mask"))
    if kind == "decode_graph":
        return [*(y[:, t:t + 1] for t in range(c["T"])), slot, mass]
    if kind == "decode_steps":
        return [y.transpose(0, 1), slot, mass]
    return [y, slot, mass]
