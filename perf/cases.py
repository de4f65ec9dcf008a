"""What is measured: the calls that users of the package make, over the sizes they make them at.

``listed()`` holds the fixed cases and ``draw(rng)`` makes further ones of the same ranges.
``prepare`` builds what a program has in hand before a call, ``run`` makes one pass through the
package's public entry points, ``work`` states the bytes and operations the pass cannot do
without, ``exact`` computes the same outputs in 64 bits with plain torch, and ``tolerance`` says
how far a correct implementation at the same precision may be from another.
"""

from __future__ import annotations

import math

import torch
from torch.nn import functional as F

from mamba3_amd import Mamba3, ops

TWO_PI = 2.0 * math.pi
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZE = {"bf16": 2, "f16": 2, "f32": 4}
DEVICE = "cuda"


def listed():
    return [
        # one token of a served model at batch 1 (the decode configuration's widths, 12 layers):
        # launches, weight streaming and latency
        dict(name="decode_b1", kind="decode", d_model=2048, d_state=128, rank=1, depth=12, batch=1,
             dtype="bf16"),
        # the decode step of one layer at full serving batch: the FP32 state streamed once
        dict(name="step_b256", kind="step", d_model=2048, d_state=128, rank=1, batch=256,
             dtype="bf16"),
        # the same layer with rank-4 MIMO at a middle batch
        dict(name="step_mimo_b64", kind="step", d_model=2048, d_state=128, rank=4, batch=64,
             dtype="bf16"),
        # the SISO prefill scan of the benchmark's headline
        dict(name="prefill_siso", kind="scan", d_model=1024, d_state=128, rank=1, batch=8,
             length=8192, dtype="bf16", cache=False, reverse=False),
        # rank-4 MIMO prefill, leaving the decode cache
        dict(name="prefill_mimo", kind="scan", d_model=1024, d_state=128, rank=4, batch=8,
             length=4096, dtype="bf16", cache=True, reverse=False),
        # one user's prompt of ordinary, ragged length before decoding at batch 1
        dict(name="prompt_b1", kind="scan", d_model=2048, d_state=128, rank=1, batch=1,
             length=1777, dtype="bf16", cache=True, reverse=False),
        # one long document, the state carried over a thousand blocks
        dict(name="long_document", kind="scan", d_model=768, d_state=128, rank=1, batch=1,
             length=65536, dtype="bf16", cache=False, reverse=False),
        # FP32 scan at the small reference configuration's width
        dict(name="scan_fp32", kind="scan", d_model=256, d_state=128, rank=1, batch=2,
             length=1024, dtype="f32", cache=True, reverse=False),
        # a state width that is no power of two, ragged length
        dict(name="scan_state96", kind="scan", d_model=512, d_state=96, rank=1, batch=4,
             length=1500, dtype="bf16", cache=False, reverse=False),
        # the reference's scan hook: normed q / k, FP32 dt / adt and a given phase, rank 2
        dict(name="hook_rank2", kind="hook", d_model=1024, d_state=128, rank=2, batch=4,
             length=2048, dtype="bf16", state=True),
        # a bidirectional encoder, whole: two layers over a batch of sequences under autocast
        dict(name="encoder", kind="model", d_model=768, d_state=128, rank=1, depth=2, batch=8,
             length=2000, causal=False),
        # the residual add and RMSNorm between two mixers of a prefill
        dict(name="residual_norm", kind="norm", rows=65536, dim=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "step", "step", "scan", "scan", "scan", "scan", "hook", "model",
                       "norm"])
    if kind == "decode":
        return dict(kind=kind, d_model=rng.choice([1024, 2048]), d_state=128,
                    rank=rng.choice([1, 1, 4]), depth=rng.randint(4, 12), batch=_log(rng, 1, 64),
                    dtype=rng.choice(["bf16", "bf16", "f16"]))
    if kind == "step":
        return dict(kind=kind, d_model=rng.choice([512, 768, 1024, 2048]),
                    d_state=rng.choice([64, 128, 128]), rank=rng.choice([1, 1, 2, 4]),
                    batch=_log(rng, 1, 256), dtype=rng.choice(["bf16", "bf16", "f16", "f32"]))
    if kind == "norm":
        return dict(kind=kind, rows=_log(rng, 1, 65536), dim=rng.choice([256, 512, 768, 1024, 2048]))
    if kind == "model":
        batch = _log(rng, 1, 8)
        return dict(kind=kind, d_model=rng.choice([256, 512, 768]), d_state=128,
                    rank=rng.choice([1, 1, 4]), depth=rng.randint(1, 2), batch=batch,
                    length=_log(rng, 100, 16000 // batch), causal=rng.random() < 0.4)
    # scans: from a short prompt to a long batch; ragged lengths; at most the headline's heads
    # times tokens (FP32 and the rarer state widths at most an eighth of it)
    if kind == "hook":
        d_model, d_state = rng.choice([512, 768, 1024]), rng.choice([64, 128, 128])
        rank, dtype = rng.choice([1, 2, 4]), rng.choice(["bf16", "bf16", "f32"])
    else:
        d_model = rng.choice([256, 512, 768, 1024, 2048])
        d_state = rng.choice([64, 96, 128, 128, 128, 128])
        rank = rng.choice([1, 1, 1, 2, 4])
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
    heads = d_model // 32
    most = 65536 * 32 // (heads * rank)
    if dtype == "f32" or d_state != 128 or kind == "hook":
        most //= 8
    tokens = _log(rng, 200, min(65536, most))
    batch = _log(rng, 1, min(16, tokens // 100))
    length = min(tokens // batch, 2048 if d_state == 96 else 65536)
    case = dict(kind=kind, d_model=d_model, d_state=d_state, rank=rank, batch=batch, length=length,
                dtype=dtype)
    if kind == "hook":
        return dict(case, state=rng.random() < 0.5)
    cache = rng.random() < 0.6
    return dict(case, cache=cache, reverse=not cache and rng.random() < 0.4)


# ------------------------------------------------------------------ inputs


def _sizes(c):
    inner = 2 * c["d_model"]
    p = math.gcd(inner, 64)
    return inner, inner // p, p, c["d_state"], c["rank"], int(c["d_state"] * 0.5) // 2


def _trained(model):
    """Spread the constant initial values, as training does (norm weights, biases, D, MIMO)."""
    with torch.no_grad():
        for name, w in model.named_parameters():
            if not name.endswith(("in_proj.weight", "out_proj.weight", "dt_bias")):
                w.add_(0.1 * torch.randn_like(w))
    return model


def _model(c, dtype):
    with torch.device(DEVICE):
        model = Mamba3(c["d_model"], c["d_state"], c.get("depth", 1), c["rank"],
                       causal=c.get("causal", True))
    return _trained(model).to(dtype).eval()


def _cache(c, mixer, batch, dtype):
    inner, h, p, n, r, s = _sizes(c)
    return ((torch.rand(batch, h, s, device=DEVICE) * 2 - 1) * 6.28,
            torch.randn(batch, h, p, n, device=DEVICE) * 0.5,
            torch.randn(batch, h, r, n, device=DEVICE).to(dtype),
            torch.randn(batch, h, p, device=DEVICE).to(dtype) * 0.6)


@torch.no_grad()
def prepare(case, seed):
    c = case
    torch.manual_seed(seed)
    torch.cuda.manual_seed(seed)
    kind = c["kind"]
    if kind == "norm":
        return dict(case=c, x=torch.randn(c["rows"], c["dim"], device=DEVICE) * 2,
                    add=torch.randn(c["rows"], c["dim"], device=DEVICE).to(torch.bfloat16),
                    weight=1 + 0.1 * torch.randn(c["dim"], device=DEVICE))
    if kind == "model":
        # FP32 master weights, run under bf16 autocast
        return dict(case=c, model=_model(c, torch.float32),
                    x=torch.randn(c["batch"], c["length"], c["d_model"], device=DEVICE))
    dtype = DTYPES[c["dtype"]]
    inner, h, p, n, r, s = _sizes(c)
    if kind == "hook":
        b, l = c["batch"], c["length"]
        q, k = (F.rms_norm(torch.randn(b, l, 1, r, n, device=DEVICE), (n,)).to(dtype)
                for _ in range(2))
        v, z = (0.6 * torch.randn(b, l, h, p, device=DEVICE).to(dtype) for _ in range(2))
        dt = F.softplus(0.6 * torch.randn(b, l, h, device=DEVICE) - 4)
        phase = torch.cumsum(dt.unsqueeze(-1) * torch.randn(b, l, 1, s, device=DEVICE), 1)
        st = dict(case=c, q=q, k=k, value=v, gate=z, dt=dt,
                  adt=-dt * (0.5 + torch.rand(b, l, h, device=DEVICE)),
                  trap=torch.randn(b, l, h, device=DEVICE).to(dtype),
                  D=1 + 0.1 * torch.randn(h, device=DEVICE), phase=torch.fmod(phase, TWO_PI),
                  q_bias=1 + 0.1 * torch.randn(h, r, n, device=DEVICE),
                  k_bias=1 + 0.1 * torch.randn(h, r, n, device=DEVICE))
        st.update({m: (1 / r if m != "mimo_z" else 1) + 0.1 * torch.randn(h, r, p, device=DEVICE)
                   if r > 1 else None for m in ("mimo_x", "mimo_z", "mimo_out")})
        st["state"] = torch.randn(b, h, p, n, device=DEVICE) * 0.5 if c["state"] else None
        return st
    if kind == "decode":
        model = _model(c, dtype)
        decoder = model.cuda_graph(c["batch"])
        with torch.inference_mode():
            decoder.load_cache([_cache(c, layer.mixer, c["batch"], dtype) for layer in model.layers])
        return dict(case=c, model=model, decoder=decoder,
                    x=torch.randn(c["batch"], 1, c["d_model"], device=DEVICE).to(dtype))
    # one layer's scan or step from its in_proj output: bf16 / FP16 rows of an autocast prefill
    # with FP32 parameters, or the decode step with 16-bit weights
    model = _model(c, dtype if kind == "step" else torch.float32)
    mixer = model.layers[0].mixer
    rows = c["batch"] * c.get("length", 1)
    x = torch.randn(rows, c["d_model"], device=DEVICE).to(dtype)
    proj = F.linear(x, mixer.in_proj.weight.to(dtype)).view(c["batch"], c.get("length", 1), -1)
    cache = _cache(c, mixer, c["batch"], dtype) if kind == "step" else None
    return dict(case=c, mixer=mixer, proj=proj, cache=cache)


# ------------------------------------------------------------------ the calls


@torch.inference_mode()
def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "norm":
        return ops.rms_norm(state["x"], state["weight"], add=state["add"], keep_sum=True,
                            out_dtype=torch.bfloat16)
    if kind == "model":
        with torch.autocast("cuda", torch.bfloat16):
            return state["model"](state["x"])
    if kind == "hook":
        return ops.mamba3_scan(
            state["q"], state["k"], state["value"], state["gate"], state["adt"], state["dt"],
            state["trap"], state["D"], mimo_x=state["mimo_x"], mimo_z=state["mimo_z"],
            mimo_out=state["mimo_out"], initial_state=state["state"], phase=state["phase"],
            mimo_rotation=c["rank"] > 1, q_bias=state["q_bias"], k_bias=state["k_bias"])
    if kind == "decode":
        return state["decoder"](state["x"]), state["decoder"].cache
    if kind == "step":
        return ops.step_projection(state["proj"], state["mixer"], state["cache"], inplace=True)
    return [t for t in ops.scan_projection(state["proj"], state["mixer"], want_cache=c["cache"],
                                           reverse=c["reverse"]) if t is not None]


# ------------------------------------------------------------------ what a pass needs


def work(case):
    c = case
    kind = c["kind"]
    if kind == "norm":
        # x and add read, the sum and the normed rows written
        return {"bytes": c["rows"] * c["dim"] * (4 + 2 + 4 + 2), "flops": 5 * c["rows"] * c["dim"]}
    inner, h, p, n, r, s = _sizes(c)
    proj = 2 * inner + 2 * n * r + 3 * h + s
    rows = c["batch"] * c.get("length", 1)
    ssm = 4 * rows * h * r * n * p          # state update and readout of every (token, head)
    state = 4 * c["batch"] * h * p * n      # one FP32 state
    if kind == "model":
        d, depth, ways = c["d_model"], c["depth"], 1 if c["causal"] else 2
        weights = 4 * depth * d * (proj + inner)
        return {"bytes": weights + 8 * rows * d,
                "flops": depth * (2 * rows * d * (proj + ways * inner) + ways * ssm)}
    es = SIZE[c["dtype"]]
    cache = 2 * (state + c["batch"] * h * (4 * s + es * (r * n + p)))  # read and written
    if kind == "step":
        return {"bytes": cache + es * rows * (proj + inner), "flops": ssm}
    if kind == "decode":
        d, depth = c["d_model"], c["depth"]
        return {"bytes": depth * (es * d * (proj + inner) + cache) + 2 * es * rows * d,
                "flops": depth * (2 * rows * d * (proj + inner) + ssm)}
    if kind == "hook":
        per = es * (3 * inner + 2 * n * r + h) + 4 * (2 * h + h * s)
        return {"bytes": rows * per + state * (2 if c["state"] else 1), "flops": ssm}
    return {"bytes": es * rows * (proj + inner) + state, "flops": ssm}


# rel: about four times the largest error against exact() that the outputs showed when the cases
# were written (decode at most 3e-2: twelve layers of 16-bit rounding)
_REL = {("decode", "bf16"): 3e-2, ("decode", "f16"): 4e-3, ("step", "bf16"): 1.4e-2,
        ("step", "f16"): 1.8e-3, ("step", "f32"): 1e-5, ("scan", "bf16"): 1.4e-2,
        ("scan", "f16"): 1.8e-3, ("scan", "f32"): 1e-5, ("hook", "bf16"): 1.4e-2,
        ("hook", "f32"): 1e-5}


def tolerance(case):
    kind = case["kind"]
    if kind == "norm":
        return {"rel": 7e-3}
    if kind == "model":
        return {"rel": 2.6e-2}
    return {"rel": _REL[kind, case["dtype"]]}


# ------------------------------------------------------------------ the same in 64 bits


def _d(t):
    return None if t is None else t.detach().double()


def _norm64(x, weight, eps=1e-5):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight


def _split64(proj, m, c):
    """The in_proj output's slices: z, x, k, q, dt, adt, trap and pi tanh(angle)."""
    inner, h, p, n, r, s = _sizes(c)
    lead = proj.shape[:-1]
    z, x, k, q, ddt, da, trap, ang = torch.split(proj.double(), (inner, inner, n * r, n * r, h, h,
                                                                 h, s), -1)
    k = _norm64(k.reshape(*lead, 1, r, n), _d(m.B_norm.weight)) + _d(m.B_bias)
    q = _norm64(q.reshape(*lead, 1, r, n), _d(m.C_norm.weight)) + _d(m.C_bias)
    u = ddt + _d(m.dt_bias)
    dt = torch.where(u > 20, u, torch.log1p(torch.exp(u.clamp(max=20))))
    heavy = torch.where(da >= 0, 1 + da, 1 / (1 - da.clamp(max=0)))
    adt = -heavy.clamp(min=1e-4) * dt
    return (z.reshape(*lead, h, p), x.reshape(*lead, h, p), k, q, dt, adt,
            torch.sigmoid(trap), math.pi * torch.tanh(ang))


def _rotate64(t, phase, rank):
    """Rotate [..., H, R, N] by phase [..., H, S]: adjacent pairs, or quarters 0 and 2 (MIMO)."""
    s = phase.shape[-1]
    cos, sin = torch.cos(phase).unsqueeze(-2), torch.sin(phase).unsqueeze(-2)
    t = t.clone()
    i = torch.arange(s, device=t.device)
    ia, ib = (2 * i, 2 * i + 1) if rank == 1 else (i, 2 * s + i)
    a, b = t[..., ia], t[..., ib]
    t[..., ia], t[..., ib] = a * cos - b * sin, a * sin + b * cos
    return t


def _ssm64(k, q, v, z, dt, adt, trap, D, mimo, state, k0=None, v0=None):
    """The recurrence token by token: k, q [B, L, H, R, N] rotated, v, z [B, L, H, P]."""
    b, l, h, r, n = k.shape
    p = v.shape[-1]
    mx, mz, mo = (1.0 if t is None else _d(t) for t in mimo)
    vr, zr = v.unsqueeze(-2) * mx, z.unsqueeze(-2) * mz
    k0 = torch.zeros_like(k[:, 0]) if k0 is None else k0
    v0 = torch.zeros_like(vr[:, 0]) if v0 is None else v0.unsqueeze(-2) * mx
    alpha = torch.exp(adt)
    beta, gamma = (1 - trap) * dt * alpha, trap * dt
    kk = torch.cat((torch.cat((k0.unsqueeze(1), k[:, :-1]), 1), k), 3)
    vv = torch.cat((torch.cat((v0.unsqueeze(1), vr[:, :-1]), 1) * beta[..., None, None],
                    vr * gamma[..., None, None]), 3).transpose(-1, -2)
    kk, vv, qt = (t.transpose(0, 1).reshape(l, b * h, *t.shape[3:]).contiguous()
                  for t in (kk, vv, q.transpose(-1, -2)))
    al = alpha.transpose(0, 1).reshape(l, b * h, 1, 1)
    st = state.reshape(b * h, p, n).clone()
    ys = torch.empty(l, b * h, p, r, dtype=torch.float64, device=k.device)
    for t in range(l):
        st.mul_(al[t]).baddbmm_(vv[t], kk[t])
        torch.bmm(st, qt[t], out=ys[t])
    y = ys.transpose(-1, -2).reshape(l, b, h, r, p).transpose(0, 1)
    y = (y + _d(D)[:, None, None] * vr) * (zr * torch.sigmoid(zr)) * mo
    return y.sum(-2), st.view(b, h, p, n)


def _scan64(proj, m, c, block=512):
    """One mixer's scan from its in_proj output, in blocks of tokens."""
    inner, h, p, n, r, s = _sizes(c)
    b, l = proj.shape[:2]
    state = torch.zeros(b, h, p, n, dtype=torch.float64, device=proj.device)
    phase, k0, v0, ys = 0.0, None, None, []
    for t in range(0, l, block):
        z, x, k, q, dt, adt, trap, ang = _split64(proj[:, t:t + block], m, c)
        ph = phase + torch.cumsum(ang.unsqueeze(-2) * dt.unsqueeze(-1), 1)
        k, q = _rotate64(k, ph, r), _rotate64(q, ph, r)
        y, state = _ssm64(k, q, x, z, dt, adt, trap, m.D, (m.mimo_x, m.mimo_z, m.mimo_out), state,
                          k0, v0)
        ys.append(y)
        phase, k0, v0 = torch.fmod(ph[:, -1:], TWO_PI), k[:, -1], x[:, -1]
    return torch.cat(ys, 1), state, k0


def _step64(proj, m, c, cache):
    z, x, k, q, dt, adt, trap, ang = _split64(proj, m, c)
    ph = _d(cache[0]).unsqueeze(1) + ang.unsqueeze(-2) * dt.unsqueeze(-1)
    k, q = _rotate64(k, ph, c["rank"]), _rotate64(q, ph, c["rank"])
    y, state = _ssm64(k, q, x, z, dt, adt, trap, m.D, (m.mimo_x, m.mimo_z, m.mimo_out),
                      _d(cache[1]), _d(cache[2]), _d(cache[3]))
    return y, state, k[:, 0], x[:, 0]


@torch.no_grad()
def exact(case, seed):
    c = case
    st = prepare(c, seed)
    kind = c["kind"]
    if kind == "norm":
        total = st["x"].double() + st["add"].double()
        return _norm64(total, _d(st["weight"])), total
    if kind == "hook":
        inner, h, p, n, r, s = _sizes(c)
        k, q = (_rotate64(_d(st[t]) + _d(st[t + "_bias"]), st["phase"].double(), r)
                for t in ("k", "q"))
        state = (torch.zeros(c["batch"], h, p, n, dtype=torch.float64, device=DEVICE)
                 if st["state"] is None else _d(st["state"]))
        return _ssm64(k, q, _d(st["value"]), _d(st["gate"]), _d(st["dt"]), _d(st["adt"]),
                      torch.sigmoid(_d(st["trap"])), st["D"],
                      (st["mimo_x"], st["mimo_z"], st["mimo_out"]), state)
    if kind == "scan":
        proj = st["proj"].flip(1) if c["reverse"] else st["proj"]
        y, state, k = _scan64(proj, st["mixer"], c)
        y = y.flip(1) if c["reverse"] else y
        # the final phase is known up to whole turns only
        return [y, state, None, k] if c["cache"] else [y, state]
    if kind == "step":
        y, state, k, v = _step64(st["proj"], st["mixer"], c, st["cache"])
        return y[:, 0], (None, state, k, v)
    h = _d(st["x"])
    model, caches = st["model"], []
    for i, layer in enumerate(model.layers):
        m = layer.mixer
        proj = _norm64(h, _d(layer.norm.weight)) @ _d(m.in_proj.weight).T
        out = _d(m.out_proj.weight).T
        if kind == "decode":
            y, state, k, v = _step64(proj, m, c, st["decoder"].cache[i])
            caches.append((None, state, k, v))
            mixed = y.flatten(-2) @ out
        else:
            mixed = _scan64(proj, m, c)[0].flatten(-2) @ out
            if not c["causal"]:
                back = _scan64(proj.flip(1), m, c)[0].flip(1).flatten(-2) @ out
                blend = torch.sigmoid(_d(m.direction_logit))
                mixed = mixed * blend + back * (1 - blend)
        h = h + mixed
    h = _norm64(h, _d(model.norm_f.weight))
    return (h, caches) if kind == "decode" else h
