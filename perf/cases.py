"""The workloads this framework's speed is measured on: the SSSD scan, its backward and the
sub-layer around it, the CHAM memory of the same layer, its Newton-Schulz retraction, and the
whole model's prefill and decode, each through the package's public entry points.

``listed()`` names the cases, ``draw(rng)`` gives more of the same ranges, ``prepare`` makes what
a caller holds before the call, ``run`` is one pass, ``work`` what a pass cannot do without,
``tolerance`` how far another correct implementation may differ and ``exact`` the same outputs in
64 bits as plain torch gives them.
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "verace-v1_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import verace_amd as va  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZE = {"bf16": 2, "fp16": 2, "fp32": 4}
HIDDEN = 1024   # the default model's width, with 8 heads of 128
HOLO = 1024     # and its CHAM dimension


def listed():
    return [
        # One token of one sequence through the SSSD sub-layer, the state updated in place: a
        # single-user generation loop runs this once per layer and token.
        dict(name="attn_step_b1", kind="attn_step", B=1, H=8, dtype="bf16"),
        # The scan of the small fp32 model configuration (2 layers, 4 heads of 64).
        dict(name="scan_small_fp32", kind="scan", B=2, T=128, H=4, D=64, dtype="fp32", init=False),
        # A prompt piece that continues a held state, at a ragged length, in fp16.
        dict(name="scan_continue_fp16", kind="scan", B=3, T=777, H=8, D=128, dtype="fp16", init=True),
        # The operator-level prefill scan that the headline metric is quoted on.
        dict(name="scan_op", kind="scan", B=8, T=4096, H=8, D=128, dtype="bf16", init=False),
        # One very long sequence: few heads, so the work has to be split along time.
        dict(name="scan_long", kind="scan", B=1, T=65536, H=16, D=128, dtype="bf16", init=False),
        # The scan's forward and backward in bf16 at the full model's training shape.
        dict(name="scan_train", kind="scan_train", B=4, T=2048, H=8, D=128, dtype="bf16"),
        # The SSSD sub-layer's training step under bf16 autocast with fp32 weights, as the
        # training loop runs it (the normalised q, k, v reach the scan in fp32 there).
        dict(name="attn_train", kind="attn_train", B=4, T=2048, H=8, dtype="autocast"),
        # The CHAM sub-layer over a fresh prompt at the full model's shape.
        dict(name="cham_prefill", kind="cham", B=4, T=2048, h=HOLO, dtype="bf16", init=False),
        # The CHAM sub-layer over the next piece of a prompt, from the hologram held so far.
        dict(name="cham_continue", kind="cham", B=4, T=512, h=HOLO, dtype="bf16", init=True),
        # The retraction of held holograms (done once when decode states are loaded).
        dict(name="ns_retraction", kind="ns", B=4, h=HOLO),
        # A whole model (of two layers, as the small configuration has, so that roundings do not
        # pile up over twelve; every layer does the same work) over a batch of prompts: logits.
        dict(name="model_prefill", kind="model_prefill", B=4, T=2048, L=2, dtype="bf16"),
        # One token for 64 sequences through such a model, replayed from its captured graph.
        dict(name="model_decode", kind="model_decode", B=64, L=2, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["attn_step", "scan_small", "scan", "scan", "scan_train", "attn_train",
                       "cham", "cham", "ns", "model_prefill", "model_decode"])
    if kind == "attn_step":
        return dict(kind=kind, B=_log(rng, 1, 256), H=rng.choice([4, 8, 16]),
                    dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]))
    if kind == "scan_small":  # fp32, the head sizes the small configurations and tests use
        return dict(kind="scan", B=rng.randint(1, 4), T=_log(rng, 8, 2048), H=rng.randint(2, 8),
                    D=rng.choice([16, 24, 64, 64, 128, 128]), dtype="fp32", init=rng.random() < 0.5)
    if kind == "scan":        # 16-bit, up to a quarter of the long sequence's tokens
        B, H = _log(rng, 1, 16), rng.choice([4, 8, 8, 16])
        T = _log(rng, 32, max(64, 262144 // (B * H)))
        return dict(kind=kind, B=B, T=T, H=H, D=128, dtype=rng.choice(["bf16", "bf16", "fp16"]),
                    init=rng.random() < 0.5)
    if kind == "scan_train":
        B, H = rng.randint(1, 4), rng.choice([4, 8])
        return dict(kind=kind, B=B, T=_log(rng, 64, 2048), H=H, D=rng.choice([64, 128, 128]),
                    dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]))
    if kind == "attn_train":
        return dict(kind=kind, B=rng.randint(1, 4), T=_log(rng, 64, 2048), H=8, dtype="autocast")
    if kind == "cham":
        init = rng.random() < 0.5
        return dict(kind=kind, B=rng.randint(1, 4), T=_log(rng, 24, 1024 if init else 2048),
                    h=rng.choice([256, 512, HOLO, HOLO]), dtype=rng.choice(["bf16", "bf16", "fp16"]),
                    init=init)
    if kind == "ns":
        return dict(kind=kind, B=_log(rng, 1, 8), h=rng.choice([128, 256, 512, 1000, HOLO]))
    if kind == "model_prefill":
        return dict(kind=kind, B=rng.randint(1, 4), T=_log(rng, 32, 2048), L=rng.randint(1, 3),
                    dtype="bf16")
    return dict(kind=kind, B=_log(rng, 1, 64), L=rng.randint(1, 3), dtype="bf16")


# ------------------------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _scan_inputs(c, seed):
    """Unit q, k, v and delta = 0.1 sigmoid(.), as the sub-layer's projections give them."""
    g, dt = _gen(seed), DTYPES[c["dtype"]]
    shape = (c["B"], c["T"], c["H"], c["D"])
    q, k, v = (F.normalize(_randn(g, *shape), dim=-1).to(dt) for _ in range(3))
    delta = (0.1 * torch.sigmoid(_randn(g, *shape[:3]))).to(dt)
    return g, q, k, v, delta


def _orthogonal(g, n, d, count=24):
    """n orthogonal d x d states, the identity times ``count`` random reflections (a held state
    is the identity times the factors of the tokens so far)."""
    s = torch.eye(d, device="cuda").expand(n, d, d).contiguous()
    for _ in range(count):
        w = F.normalize(_randn(g, n, d), dim=-1)
        s -= 2.0 * w.unsqueeze(2) * (w.unsqueeze(1) @ s)
    return s


def _unitary(g, n, h, count=8):
    """n unitary h x h holograms (real, imaginary), made the same way."""
    r = torch.eye(h, device="cuda").expand(n, h, h).contiguous()
    i = torch.zeros_like(r)
    for _ in range(count):
        w = F.normalize(_randn(g, n, 2 * h), dim=-1)
        wr, wi = w[:, :h], w[:, h:]
        ar = wr.unsqueeze(1) @ r + wi.unsqueeze(1) @ i       # w^H H
        ai = wr.unsqueeze(1) @ i - wi.unsqueeze(1) @ r
        r -= 2.0 * (wr.unsqueeze(2) * ar - wi.unsqueeze(2) * ai)
        i -= 2.0 * (wr.unsqueeze(2) * ai + wi.unsqueeze(2) * ar)
    return r, i


def _module(cls, seed, dtype, *args):
    torch.manual_seed(seed)
    with torch.device("cuda"):
        return cls(*args).to(dtype)


def _attn(c, seed, dtype):
    return _module(va.SSSDAttention, seed, dtype, HIDDEN, c["H"], 128)


def _attn_train_inputs(c, seed):
    g = _gen(seed)
    x = _randn(g, c["B"], c["T"], HIDDEN)
    return _attn(c, seed, torch.float32), x, _randn(g, *x.shape).to(torch.bfloat16)


def _cham_inputs(c, seed):
    dt = DTYPES[c["dtype"]]
    g = _gen(seed)
    m = _module(va.ContinuousHolographicMemory, seed, dt, HIDDEN, c["h"])
    x = _randn(g, c["B"], c["T"], HIDDEN).to(dt)
    return m, x, _unitary(g, c["B"], c["h"]) if c["init"] else None


def _ns_inputs(c, seed):
    g = _gen(seed)
    hr, hi = _unitary(g, c["B"], c["h"])
    eps = 0.02 / math.sqrt(c["h"])   # rounding and input error of a held state
    return hr + eps * _randn(g, *hr.shape), hi + eps * _randn(g, *hi.shape)


def _model(c, seed):
    """Random weights, but routers as decided as a trained one's: an untrained router's logits lie
    so close together that one bf16 rounding changes the selected components, and with them
    everything after."""
    cfg = va.VeraceV1Config(vocab_size=32000, num_layers=c["L"])
    m = _module(va.VeraceV1Model, seed, DTYPES[c["dtype"]], cfg).requires_grad_(False)
    for layer in m.layers:
        layer.mcmoe.router.weight.mul_(8.0)
    return m


def prepare(case, seed):
    c = case
    kind = c["kind"]
    if kind == "attn_step":
        dt, g = DTYPES[c["dtype"]], _gen(seed)
        m = _attn(c, seed, dt)
        x = _randn(g, c["B"], 1, HIDDEN).to(dt)
        state = _orthogonal(g, c["B"] * c["H"], 128).view(c["B"], c["H"], 128, 128)
        return dict(kind=kind, m=m, x=x, state=state)
    if kind == "scan":
        g, q, k, v, delta = _scan_inputs(c, seed)
        init = None
        if c["init"]:
            init = _orthogonal(g, c["B"] * c["H"], c["D"]).view(c["B"], c["H"], c["D"], c["D"])
        return dict(kind=kind, args=(q, k, v, delta, init))
    if kind == "scan_train":
        g, q, k, v, delta = _scan_inputs(c, seed)
        ins = [t.requires_grad_() for t in (q, k, v, delta)]
        return dict(kind=kind, ins=ins, d_out=_randn(g, *q.shape).to(q.dtype))
    if kind == "attn_train":
        m, x, dy = _attn_train_inputs(c, seed)
        return dict(kind=kind, m=m, x=x.requires_grad_(), dy=dy)
    if kind == "cham":
        m, x, holo = _cham_inputs(c, seed)
        return dict(kind=kind, m=m, x=x, holo=holo)
    if kind == "ns":
        return dict(kind=kind, args=_ns_inputs(c, seed))
    m = _model(c, seed)
    g = _gen(seed)
    if kind == "model_prefill":
        ids = torch.randint(0, 32000, (c["B"], c["T"]), generator=g, device="cuda")
        return dict(kind=kind, m=m, ids=ids)
    st = va.DecodeState([va.LayerDecodeState(
        _orthogonal(g, c["B"] * 8, 128, 8).view(c["B"], 8, 128, 128), _unitary(g, c["B"], HOLO, 4))
        for _ in range(c["L"])])
    ids = torch.randint(0, 32000, (c["B"], 1), generator=g, device="cuda")
    with torch.no_grad():
        return dict(kind=kind, state=st, ids=ids, graph=va.DecodeGraph(m, st, c["B"]), m=m)


# ---------------------------------------------------------------------------------- one pass

def run(state):
    s = state
    kind = s["kind"]
    if kind == "scan":
        return va.launch_sssd_hip_scan(*s["args"])
    if kind == "scan_train":
        o, psi = va.sssd_scan(*s["ins"])
        return (o.detach(), psi.detach(), *torch.autograd.grad(o, s["ins"], s["d_out"]))
    if kind == "attn_train":
        m, x = s["m"], s["x"]
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y, psi = m(x, return_state=True)
        return (y.detach(), psi.detach(), *torch.autograd.grad(y, [x, *m.parameters()], s["dy"]))
    with torch.no_grad():
        if kind == "attn_step":
            return s["m"].step_(s["x"], s["state"]), s["state"]
        if kind == "cham":
            y, (hr, hi) = s["m"](s["x"], initial_hologram=s["holo"])
            return y, hr, hi
        if kind == "ns":
            return va.newton_schulz_unitary_retraction(*s["args"], steps=3)
        if kind == "model_prefill":
            return s["m"](s["ids"], use_adaptive_depth=False)
        logits = s["graph"].step(s["ids"])
        return (logits, [(l.sssd, l.cham[0], l.cham[1]) for l in s["state"].layers])


# -------------------------------------------------------------------------------------- work

def _attn_params(H):
    return 4 * HIDDEN * H * 128 + HIDDEN * H


def _scan_work(B, T, H, D, es, init):
    """q, k, v, out and delta once, the state out (and in); 10 D^2 per token and head: two
    column sums, a rank-2 update and a readout."""
    n = B * T * H
    return n * (4 * D + 1) * es + B * H * D * D * 4 * (2 if init else 1), 10 * D * D * n


def _cham_flops(B, T, h):
    """Per token two complex column sums with real k, v, a rank-2 complex update, and the
    readout's real part."""
    return B * T * (8 + 8 + 4) * h * h


def _mcmoe_work(n):
    """Base GLU of width 2 x hidden, 64 components of rank 32 with 8 selected, router, sigma."""
    d = HIDDEN
    return 2 * n * (6 * d * d + 64 * d + 2048 * d + 2 * 8 * 32 * d)


_LAYER_PARAMS = _attn_params(8) + 4 * HIDDEN * HOLO + HIDDEN \
    + 6 * HIDDEN * HIDDEN + 64 * HIDDEN + 3 * 2048 * HIDDEN


def work(case):
    c = case
    kind = c["kind"]
    if kind == "attn_step":
        es, p, st = SIZE[c["dtype"]], _attn_params(c["H"]), c["B"] * c["H"] * 128 * 128
        return dict(bytes=p * es + 2 * st * 4 + 2 * c["B"] * HIDDEN * es,
                    flops=2 * c["B"] * p + 10 * st)
    if kind == "scan":
        b, f = _scan_work(c["B"], c["T"], c["H"], c["D"], SIZE[c["dtype"]], c["init"])
        return dict(bytes=b, flops=f)
    if kind == "scan_train":
        es = SIZE[c["dtype"]]
        b, f = _scan_work(c["B"], c["T"], c["H"], c["D"], es, False)
        # d_out in, dq, dk, dv, d_delta out; two products for each of the forward's
        return dict(bytes=b + c["B"] * c["T"] * c["H"] * (4 * c["D"] + 1) * es, flops=3 * f)
    if kind == "attn_train":
        n, p = c["B"] * c["T"], _attn_params(c["H"])
        _, f = _scan_work(c["B"], c["T"], c["H"], 128, 4, False)
        # x, weights, dy in; y, dx, dw out; three products per projection
        return dict(bytes=n * HIDDEN * (4 + 2 + 2 + 4) + 2 * p * 4 + c["B"] * c["H"] * 128 * 128 * 4,
                    flops=6 * n * p + 3 * f)
    if kind == "cham":
        n, h, es = c["B"] * c["T"], c["h"], SIZE[c["dtype"]]
        p = 4 * HIDDEN * h + HIDDEN
        st = c["B"] * h * h * 8
        f = 2 * n * p + _cham_flops(c["B"], c["T"], h)
        return dict(bytes=2 * n * HIDDEN * es + p * es + st * (2 if c["init"] else 1), flops=f)
    if kind == "ns":  # Gram and product, four real products each, three steps
        return dict(bytes=16 * c["B"] * c["h"] ** 2, flops=48 * c["B"] * c["h"] ** 3)
    head = 32000 * HIDDEN
    if kind == "model_prefill":
        n = c["B"] * c["T"]
        per = 2 * n * (_attn_params(8) + 4 * HIDDEN * HOLO + HIDDEN) + 10 * 128 * 128 * 8 * n \
            + _cham_flops(c["B"], c["T"], HOLO) + _mcmoe_work(n)
        return dict(bytes=2 * (c["L"] * _LAYER_PARAMS + head + n * 32000),
                    flops=c["L"] * per + 2 * n * head)
    B = c["B"]
    st = B * (8 * 128 * 128 + 2 * HOLO * HOLO) * 4
    return dict(bytes=2 * (c["L"] * _LAYER_PARAMS + head + B * 32000) + c["L"] * 2 * st,
                flops=c["L"] * (2 * B * (_attn_params(8) + 4 * HIDDEN * HOLO) + _mcmoe_work(B)
                                + 10 * B * 8 * 128 * 128 + _cham_flops(B, 1, HOLO)) + 2 * B * head)


# --------------------------------------------------------------------------------- tolerance

def tolerance(case):
    """About four times the largest relative difference from the 64-bit results (whole models:
    between two op sequences of this package) measured over the ranges; each is what the types
    give: fp32 sums, one 16-bit rounding of an output, 16-bit operands of a product."""
    kind, dt = case["kind"], case.get("dtype")
    if kind == "ns":
        return dict(rel=4e-6)
    if kind == "scan":
        return dict(rel={"fp32": 6e-6, "fp16": 2.5e-3, "bf16": 7e-3}[dt])
    if kind == "scan_train":
        return dict(rel=6e-6 if dt == "fp32" else 1.7e-2)
    if kind == "attn_train":
        return dict(rel=2.8e-2)
    if kind == "attn_step":
        return dict(rel=1e-5 if dt == "fp32" else 1.2e-2)
    if kind == "cham":
        return dict(rel=1.5e-2)
    return dict(rel=0.05 * case["L"])   # a router's near tie that falls the other way, per layer


# ------------------------------------------------------------------------------------- exact

def _cayley_apply(k, v, delta, psi):
    """(I + X)^-1 (I - X) psi for X = (delta/2)(k v^T - v k^T): X^3 = -m^2 X gives the closed
    form I + c(X^2 - X), c = 2 / (1 + m^2)."""
    h = (0.5 * delta).unsqueeze(-1)
    kk, vv, kv = (k * k).sum(-1, True), (v * v).sum(-1, True), (k * v).sum(-1, True)
    c = 2.0 / (1.0 + h * h * (kk * vv - kv * kv))
    a = (k.unsqueeze(-2) @ psi).squeeze(-2)
    b = (v.unsqueeze(-2) @ psi).squeeze(-2)
    ak = c * (-h * b + h * h * (kv * b - vv * a))
    av = c * (h * a + h * h * (kv * a - kk * b))
    return psi + torch.stack((k, v), -1) @ torch.stack((ak, av), -2)


def _scan64(q, k, v, delta, psi):
    """[B, T, H, D] double inputs -> (o, psi)."""
    out = []
    for t in range(q.shape[1]):
        psi = _cayley_apply(k[:, t], v[:, t], delta[:, t], psi)
        out.append((psi @ q[:, t].unsqueeze(-1)).squeeze(-1))
    return torch.stack(out, 1), psi


def _eye64(B, H, D):
    return torch.eye(D, device="cuda", dtype=torch.double).expand(B, H, D, D).contiguous()


def _scan64_grad(q, k, v, delta, d_out, piece=64):
    """(o, psi, dq, dk, dv, d_delta) by autograd over pieces of the sequence, last piece first."""
    B, T, H, D = q.shape
    starts, outs, psi = [], [], _eye64(B, H, D)
    with torch.no_grad():
        for t in range(0, T, piece):
            starts.append(psi)
            sl = slice(t, t + piece)
            o, psi = _scan64(q[:, sl], k[:, sl], v[:, sl], delta[:, sl], psi)
            outs.append(o)
    d_psi, grads = torch.zeros_like(psi), []
    with torch.enable_grad():
        for i in reversed(range(len(starts))):
            sl = slice(i * piece, (i + 1) * piece)
            ins = [t[:, sl].detach().requires_grad_() for t in (q, k, v, delta)]
            ins.append(starts[i].detach().requires_grad_())
            g = torch.autograd.grad(_scan64(*ins), ins, (d_out[:, sl], d_psi))
            grads.append(g[:4])
            d_psi = g[4]
    return (torch.cat(outs, 1), psi, *(torch.cat(x, 1) for x in zip(*reversed(grads))))


def _rms64(x, w, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w


def _attn64(p, x, H):
    """The sub-layer's projections in 64 bits: unit q, k, v and delta."""
    B, T, _ = x.shape
    q, k, v = (F.normalize((x @ p[n].t()).view(B, T, H, 128), dim=-1)
               for n in ("w_q.weight", "w_k.weight", "w_v.weight"))
    return q, k, v, 0.1 * torch.sigmoid(x @ p["w_delta.weight"].t())


_EPS32 = torch.finfo(torch.float32).eps   # what nn.RMSNorm adds by default


def _params64(m):
    return {n: t.detach().double() for n, t in m.named_parameters()}


def _ns64(r, i):
    h = torch.complex(r.double(), i.double())
    eye = 3.0 * torch.eye(h.shape[-1], device="cuda", dtype=h.dtype)
    for _ in range(3):
        h = 0.5 * (h @ (eye - h.mH @ h))
    return h


def _cham64(m, x, holo):
    p = _params64(m)
    x = x.double()
    B, T, _ = x.shape
    q, k = (F.normalize(x @ p[n].t(), dim=-1) for n in ("w_q.weight", "w_k.weight"))
    v = F.normalize(F.silu(x @ p["w_v.weight"].t()), dim=-1)
    g = 0.05 * torch.sigmoid(x @ p["w_gamma.weight"].t())          # gamma / 2, [B, T, 1]
    kk, vv, kv = (k * k).sum(-1, True), (v * v).sum(-1, True), (k * v).sum(-1, True)
    scale = 2.0 / torch.complex(1.0 + g * g * (kk * vv - kv * kv), -2.0 * g * kv)
    nkk, nvv = scale * (-g * g * vv), scale * (-g * g * kk)
    nkv = scale * torch.complex(g * g * kv, g)
    h = q.shape[-1]
    # raw state, and beside it the readout state NS_3(H) = (product of the factors) NS_3(H_0)
    if holo is None:
        st = [torch.eye(h, device="cuda", dtype=torch.complex128).expand(B, h, h).contiguous()]
    else:
        st = [torch.complex(holo[0].double(), holo[1].double()), _ns64(*holo)]
    N = torch.stack((torch.cat((nkk, nkv), -1), torch.cat((nkv, nvv), -1)), -2)   # [B, T, 2, 2]
    W = torch.stack((k, v), -1).to(torch.complex128)                              # [B, T, h, 2]
    out = []
    for t in range(T):
        for s in st:
            s.baddbmm_(W[:, t], N[:, t] @ (W[:, t].mT.contiguous() @ s))
        out.append((st[-1] @ q[:, t].unsqueeze(-1).to(torch.complex128)).squeeze(-1).real)
    y = torch.stack(out, 1) @ p["w_out.weight"].t()
    return _rms64(y, p["norm.weight"], _EPS32), st[0].real.contiguous(), st[0].imag.contiguous()


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind == "scan":
        s = prepare(c, seed)
        q, k, v, delta, init = s["args"]
        psi = _eye64(c["B"], c["H"], c["D"]) if init is None else init.double()
        with torch.no_grad():
            return _scan64(q.double(), k.double(), v.double(), delta.double(), psi)
    if kind == "scan_train":
        s = prepare(c, seed)
        return _scan64_grad(*(t.detach().double() for t in s["ins"]), s["d_out"].double())
    if kind == "attn_step":
        s = prepare(c, seed)
        p = _params64(s["m"])
        with torch.no_grad():
            q, k, v, delta = _attn64(p, s["x"].double(), c["H"])
            o, psi = _scan64(q, k, v, delta, s["state"].double())
            o = _rms64(o, p["head_rmsnorm.weight"], _EPS32).reshape(c["B"], 1, -1)
            return o @ p["w_out.weight"].t(), psi
    if kind == "attn_train":
        m, x, dy = _attn_train_inputs(c, seed)
        p = {n: t.requires_grad_() for n, t in _params64(m).items()}
        x = x.double().requires_grad_()
        with torch.enable_grad():
            ins = _attn64(p, x, c["H"])
            leaf = torch.zeros(c["B"], c["T"], c["H"], 128, device="cuda", dtype=torch.double)
            with torch.no_grad():
                o, _ = _scan64(*ins, _eye64(c["B"], c["H"], 128))
            leaf = o.detach().requires_grad_()
            y = _rms64(leaf, p["head_rmsnorm.weight"], _EPS32).reshape(c["B"], c["T"], -1) \
                @ p["w_out.weight"].t()
            g = torch.autograd.grad(y, [leaf, p["head_rmsnorm.weight"], p["w_out.weight"]], dy.double())
            _, psi, *d_ins = _scan64_grad(*(t.detach() for t in ins), g[0])
            names = ["w_q.weight", "w_k.weight", "w_v.weight", "w_delta.weight"]
            gi = torch.autograd.grad(ins, [x] + [p[n] for n in names], d_ins)
        grads = dict(zip(names, gi[1:]))
        grads["head_rmsnorm.weight"], grads["w_out.weight"] = g[1], g[2]
        return (y.detach(), psi, gi[0], *(grads[n] for n, _ in m.named_parameters()))
    if kind == "cham":
        with torch.no_grad():
            return _cham64(*_cham_inputs(c, seed))
    if kind == "ns":
        h = _ns64(*_ns_inputs(c, seed))
        return h.real.contiguous(), h.imag.contiguous()
    return None   # whole models: a change of one rounding travels through every later layer
