"""The calls whose speed this repository is measured by.

A case is one call a serving engine makes per layer, through the package's
public entry points: the whole MoE layer (`ops.MoeForward`) in each weight
format and at each batch size an engine has in its hands (one token, a few
sequences decoding together, a draft being verified, a ragged prompt chunk, a
full prompt), the fused combine + residual + RMSNorm behind it, the
ingestion of a layer's GPTQ checkpoint tensors, and the tiered NVFP4 experts.

Sizes are those of `grimoire_amd.configs` and `bench.py` where a case has one
there; the others are the same layers at other batch sizes.  Weights, router,
activations and popularity follow `grimoire_amd.configs` (activations are
bf16 values held as fp32, as the engine's residual stream has them after its
norm).
"""
from __future__ import annotations

import math

import torch

from grimoire_amd import _abi, ingest, ops, tiered
from grimoire_amd.weights import MAKERS, MoeLayer

DEV = "cuda"


def _layer(name, fmt, T, H, E, K, I, **kw):
    c = dict(kind="layer", fmt=fmt, T=T, H=H, E=E, K=K, I=I, route="softmax", zipf=0.0,
             shared=False, gate=False, n_group=0, topk_group=0, scaling=1.0)
    c.update(kw)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one sequence decoding: latency and launches
        _layer("decode_1_int4", "int4", 1, 2048, 128, 8, 768),
        # the INT8 model of the prefill cases decoding three sequences
        _layer("decode_3_int8", "int8", 3, 2048, 512, 10, 512, zipf=1.2, shared=True, gate=True),
        # eight sequences decoding on MXFP4 experts with skewed popularity,
        # rows of 2880 elements (no whole number of memory lines)
        _layer("decode_8_mxfp4", "mxfp4", 8, 2880, 128, 4, 2880, zipf=1.1),
        # sixteen sequences decoding on GPTQ experts
        _layer("decode_16_int4", "int4", 16, 2048, 64, 4, 1024),
        # a speculative draft verified on a large group-routed layer (6 GB of experts)
        _layer("verify_32_mxfp4", "mxfp4", 32, 7168, 256, 8, 2048, route="group", shared=True,
               n_group=8, topk_group=4, scaling=2.5),
        # a ragged last chunk of a prompt on the INT8 model
        _layer("chunk_201_int8", "int8", 201, 2048, 512, 10, 512, zipf=1.2, shared=True, gate=True),
        # unquantised experts: sequences decoding together and prompt chunks mixed in one batch
        _layer("mixed_150_bf16", "bf16", 150, 2048, 64, 4, 1024, route="sigmoid", scaling=1.5),
        # a prompt chunk on the decode_8 model
        _layer("prefill_1000_mxfp4", "mxfp4", 1000, 2880, 128, 4, 2880, zipf=1.1),
        # a full prompt on the INT8 model
        _layer("prefill_4096_int8", "int8", 4096, 2048, 512, 10, 512, zipf=1.2, shared=True, gate=True),
        # what follows the experts of a long, odd prompt: combine, residual, next norm
        dict(name="combine_norm_3001", kind="norm", T=3001, H=2048, K=10, shared=True),
        # loading a layer: the GPTQ tensors of 128 experts into the stacked layout
        dict(name="ingest_gptq_128", kind="ingest", E=128, H=2048, I=768, group=128, f16=False),
        # experts behind a block table (all resident), two sequences decoding
        dict(name="tiered_2_nvfp4", kind="tiered", T=2, H=2048, I=768, K=8, E=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(c):
    w = work(c)
    return w["bytes"] / 4e12 + w["flops"] / 0.5e15


def draw(rng):
    """A case of the same kinds: any batch size up to the largest listed one
    of its format, layer sizes around the listed ones."""
    top = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["int4", "int8", "int8", "mxfp4", "mxfp4", "bf16", "norm", "ingest", "tiered"])
        if kind == "norm":
            c = dict(kind="norm", T=_log(rng, 1, 8192), H=4 * _log(rng, 256, 2048),
                     K=rng.choice([2, 4, 6, 8, 10]), shared=rng.random() < 0.5)
        elif kind == "ingest":
            c = dict(kind="ingest", E=_log(rng, 8, 160), H=128 * rng.randint(6, 24), I=128 * rng.randint(3, 12),
                     group=rng.choice([64, 128]), f16=rng.random() < 0.5)
        elif kind == "tiered":
            c = dict(kind="tiered", T=rng.randint(1, 8), H=128 * rng.randint(8, 32), I=128 * rng.randint(3, 12),
                     K=rng.choice([2, 4, 6, 8, 10]), E=rng.randint(16, 128))
        else:
            E = rng.choice({"int4": [32, 64, 96, 128, 160], "int8": [64, 128, 256, 384, 512],
                            "mxfp4": [32, 64, 128, 256], "bf16": [16, 32, 64]}[kind])
            K = rng.choice([2, 4, 6, 8] + ([10] if kind == "int8" else []))
            step = 128 if kind == "int4" else 64
            H = step * rng.randint(1024 // step, 4096 // step)
            I = step * rng.randint(512 // step, 2048 // step if kind != "mxfp4" else 3072 // step)
            # INT4 experts are served up to two routes per expert (or 64 routes)
            most = max(64, 2 * E) // K if kind == "int4" else {"int8": 4096, "mxfp4": 2048, "bf16": 1024}[kind]
            route = rng.choice(["softmax", "softmax", "sigmoid", "group"])
            if route == "group" and (E < 64 or K > 4 * (E // 8)):
                route = "softmax"
            sh = rng.random() < 0.5
            c = _layer("", kind, _log(rng, 1, most), H, E, K, I, route=route,
                       zipf=rng.choice([0.0, 1.1]) if route == "softmax" else 0.0, shared=sh,
                       gate=sh and rng.random() < 0.5, scaling=1.0 if route == "softmax" else 2.5,
                       n_group=8 if route == "group" else 0, topk_group=4 if route == "group" else 0)
        if _cost(c) <= top:
            return c


# ------------------------------------------------------------------ inputs

ROUTES = {"softmax": _abi.ROUTE_SOFTMAX, "sigmoid": _abi.ROUTE_SIGMOID, "group": _abi.ROUTE_GROUP}


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _popularity(E, K, s):
    """Share of the tokens that route to the expert of each popularity rank:
    min(1, lam * (rank + 1)^-s), summing to K (uniform for s = 0)."""
    p = (torch.arange(E, dtype=torch.float64) + 1.0) ** -s
    lo, hi = 0.0, float(K) / float(p[-1])
    for _ in range(80):
        lam = 0.5 * (lo + hi)
        lo, hi = (lo, lam) if float(torch.clamp(lam * p, max=1.0).sum()) > K else (lam, hi)
    return torch.clamp(lo * p, max=1.0)


def _make_layer(c, seed):
    mk, E, H, I, K = MAKERS[c["fmt"]], c["E"], c["H"], c["I"], c["K"]
    g = _gen(seed * 16 + 1)
    router = torch.randn((E, H), generator=g, device=DEV) * 0.02
    sgu = sdn = sgw = None
    if c["shared"]:
        sgu, sdn = mk(2 * I, H, device=DEV, seed=seed * 16 + 4), mk(H, I, device=DEV, seed=seed * 16 + 5)
        if c["gate"]:
            sgw = (torch.randn((H,), generator=g, device=DEV) * 0.02).bfloat16().view(torch.int16)
    bias = None
    if c["route"] == "softmax" and c["zipf"] > 0:
        # the bias under which normally distributed logits pass a common
        # threshold as often as each rank's popularity says
        q = _popularity(E, K, c["zipf"]).clamp(1e-6, 1 - 1e-4)
        b = (0.02 * math.sqrt(H) * torch.special.ndtri(q)).float()
        bias = b.to(DEV)[torch.randperm(E, generator=g, device=DEV)].contiguous()
    elif c["route"] == "sigmoid":
        bias = (torch.randn((E,), generator=g, device=DEV) * 1e-2).bfloat16().view(torch.int16)
    elif c["route"] == "group":
        bias = torch.randn((E,), generator=g, device=DEV) * 1e-3
    L = MoeLayer(H, I, E, K, mk(E * 2 * I, H, device=DEV, seed=seed * 16 + 2),
                 mk(E * H, I, device=DEV, seed=seed * 16 + 3), router, sgu, sdn, sgw, True)
    x = torch.randn((c["T"], H), generator=g, device=DEV).bfloat16().float()
    return L, bias, x


def _norm_inputs(c, seed):
    T, H, K = c["T"], c["H"], c["K"]
    g = _gen(seed * 16 + 1)
    rw = torch.rand((T, K), device=DEV, generator=g) + 0.05
    return dict(
        h=torch.randn((T, H), device=DEV, generator=g),
        routed=torch.randn((T * K, H), device=DEV, generator=g).bfloat16().view(torch.int16),
        inverse=torch.randperm(T * K, device=DEV, generator=g).int(),
        rw=rw / rw.sum(1, keepdim=True),
        shared=torch.randn((T, H), device=DEV, generator=g) if c["shared"] else None,
        w=(torch.randn((H,), device=DEV, generator=g) * 0.1).bfloat16().view(torch.int16))


def _ingest_inputs(c, seed):
    E, H, I, grp = c["E"], c["H"], c["I"], c["group"]
    g = _gen(seed * 16 + 1)

    def rand32(*shape):
        return torch.randint(-2 ** 31, 2 ** 31 - 1, shape, dtype=torch.int32, device=DEV, generator=g)

    def proj(out, inn):
        return ingest.gptq(rand32(inn // 8, out), rand32(inn // grp, out // 8),
                           (torch.rand((inn // grp, out), device=DEV, generator=g) * 0.02 + 1e-4).half()
                           .view(torch.int16), grp)
    return [(proj(I, H), proj(I, H), proj(H, I)) for _ in range(E)]


def _tiered_inputs(c, seed):
    T, H, I, K, E = c["T"], c["H"], c["I"], c["K"], c["E"]
    lay = tiered.layout(H, I)
    g = _gen(seed * 16 + 1)
    b = torch.randint(0, 256, (E, lay.bytes), dtype=torch.uint8, device=DEV, generator=g)
    for lo, hi in ((lay.gu_s, lay.dn_p), (lay.dn_s, lay.gsc)):
        b[:, lo:hi] = 0x30 + (b[:, lo:hi] & 15)                  # E4M3 scales 0.5 .. 1.875
    s = torch.rand((E, 4), device=DEV, generator=g) * 0.02 + 0.01    # projection scales
    b[:, lay.gsc:lay.gsc + 16] = s.view(torch.uint8)
    ex = torch.stack([torch.randperm(E, device=DEV, generator=g)[:K] for _ in range(T)]).int()
    w = torch.rand((T, K), device=DEV, generator=g) + 0.05
    x = torch.randn((T, H), device=DEV, generator=g).bfloat16().float()
    return lay, b, ex, (w / w.sum(1, keepdim=True)).contiguous(), x


def prepare(case, seed):
    c, T = case, case.get("T", 0)
    if c["kind"] == "layer":
        L, bias, x = _make_layer(c, seed)
        rp = _abi.RouteParams(mode=ROUTES[c["route"]], n_group=c["n_group"], topk_group=c["topk_group"],
                              scaling=c["scaling"], bias=bias.data_ptr() if bias is not None else None)
        return dict(kind="layer", fwd=ops.MoeForward(L, T, rp), bias=bias, x=x,
                    y=torch.empty((T, c["H"]), device=DEV),
                    oe=torch.empty((T, c["K"]), dtype=torch.int32, device=DEV),
                    ow=torch.empty((T, c["K"]), device=DEV))
    if c["kind"] == "norm":
        s = _norm_inputs(c, seed)
        return dict(kind="norm", c=c, out=torch.empty((T, c["H"]), device=DEV),
                    out_bf=torch.empty((T, c["H"]), dtype=torch.bfloat16, device=DEV), **s)
    if c["kind"] == "ingest":
        return dict(kind="ingest", experts=_ingest_inputs(c, seed), f16=c["f16"])
    lay, b, ex, w, x = _tiered_inputs(c, seed)
    return dict(kind="tiered", L=tiered.TieredLayer(c["H"], c["I"], c["K"], list(b), DEV), ex=ex, w=w, x=x,
                h=torch.empty((T, c["K"] * c["I"]), device=DEV), y=torch.empty((T, c["H"]), device=DEV))


# ------------------------------------------------------------------ one pass

def run(state):
    s = state
    if s["kind"] == "layer":
        s["fwd"](s["x"], s["y"], s["oe"], s["ow"])
        return {"y": s["y"], "experts": s["oe"], "weights": s["ow"]}
    if s["kind"] == "norm":
        c = s["c"]
        ops.launch_rmsnorm_moe_residual_batched(s["h"], s["routed"], s["inverse"], s["rw"], s["shared"], s["w"],
                                                s["out"], s["out_bf"], c["T"], c["K"], c["H"], 1e-6)
        return {"h": s["h"], "out": s["out"], "out_bf": s["out_bf"]}
    if s["kind"] == "ingest":
        gu, dn = ingest.ingest_experts(s["experts"], DEV, exact_scales=s["f16"])
        return {k: [w.payload, w.scales, w.zeros] for k, w in (("gate_up", gu), ("down", dn))}
    s["L"].gate_up(s["ex"], s["x"], s["h"])
    s["L"].down(s["ex"], s["w"], s["h"], s["y"])
    return {"h": s["h"], "y": s["y"]}


# ------------------------------------------------------------------ what a pass cannot do without

def _row_bytes(fmt, K):
    """One weight row of K elements with its scales."""
    return {"int4": K / 2 + K / 128 * 2, "mxfp4": K / 2 + K / 32, "int8": K + 4, "bf16": 2 * K}[fmt]


def work(case):
    c, T = case, case.get("T", 0)
    if c["kind"] == "norm":
        H, K = c["H"], c["K"]
        n = T * K * (2 * H + 8) + T * H * (8 + (4 if c["shared"] else 0) + 4 + 2) + 2 * H
        return {"bytes": n, "flops": T * H * (2 * K + 5)}
    E, H, I, K = c["E"], c["H"], c["I"], c.get("K", 0)
    if c["kind"] == "ingest":
        elems, groups = 3 * E * H * I, 3 * E * H * I // c["group"]
        return {"bytes": elems / 2 * 2 + groups * (2 + 0.5 + 2 + 1), "flops": 0}
    if c["kind"] == "tiered":
        touched = E * (1 - (1 - K / E) ** T)
        per = 2 * I * (H / 2 + H / 16) + H * (I / 2 + I / 16)
        return {"bytes": touched * per + T * (8 * H + 8 * K + 4 * K * I), "flops": 6 * T * K * H * I}
    q = _popularity(E, K, c["zipf"])
    touched = float((1 - (1 - q) ** T).sum())
    per = 2 * I * _row_bytes(c["fmt"], H) + H * _row_bytes(c["fmt"], I)
    sh = 1 if c["shared"] else 0
    return {"bytes": (touched + sh) * per + 4 * E * H + 8 * T * H + 8 * T * K,
            "flops": 6 * T * (K + sh) * H * I + 2 * T * E * H}


def tolerance(case):
    """Four times the error against the same in 64 bits that was measured
    over the listed and drawn sizes (relative 2-norm), 1e-5 for fp32 sums."""
    if case["kind"] == "ingest":
        return "exact"
    if case["kind"] == "norm":
        return {"rel": 2e-3, "max": 2e-2}      # one output is rounded to bf16 (1.7e-3)
    if case["kind"] == "tiered":
        return {"rel": 1e-5}
    # INT8 prompts: activations as two int8 limbs under one scale per row
    # (9.8e-5); MXFP4 batches: three e4m3 limbs under one scale per 32
    # elements (3.5e-5); otherwise h as two bf16 halves (3.5e-6).  A near tie
    # may route a token elsewhere.
    rel = {"int8": 4e-4, "mxfp4": 1.5e-4, "int4": 1.5e-5, "bf16": 1.5e-5}[case["fmt"]]
    return {"rel": rel, "differ": 1e-3}


# ------------------------------------------------------------------ the same in 64 bits

E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _nibbles(p):
    return torch.stack((p & 15, p >> 4), -1).reshape(p.shape[0], -1)


def _e2m1(p):
    t = torch.tensor(E2M1 + [-v for v in E2M1], dtype=torch.float64, device=p.device)
    return t[_nibbles(p).long()]


def _dense(w, r0, n):
    """Rows [r0, r0 + n) of a packed weight, fp64."""
    p = w.payload[r0:r0 + n]
    s = None if w.scales is None else w.scales[r0:r0 + n]
    if w.fmt == _abi.FMT_BF16:
        return p.contiguous().view(torch.bfloat16).double()
    if w.fmt == _abi.FMT_INT8:
        return p.view(torch.int8).double() * s.double()[:, None]
    if w.fmt == _abi.FMT_MXFP4:
        return _e2m1(p) * torch.exp2(s.double() - 127).repeat_interleave(32, 1)
    return (_nibbles(p).double() - 8) * s.view(torch.float16).double().repeat_interleave(128, 1)


def _ffn(x, gu, dn):
    g, u = (x @ gu.T).chunk(2, 1)
    return (torch.nn.functional.silu(g) * u) @ dn.T


def _exact_layer(c, seed):
    L, bias, x = _make_layer(c, seed)
    E, H, I, K, T = c["E"], c["H"], c["I"], c["K"], c["T"]
    x = x.double()
    logits = x @ L.router.double().T
    if c["route"] == "softmax":
        sel = logits if bias is None else logits + bias.double()
        top, ids = torch.sort(sel, dim=1, descending=True, stable=True)
        ids = ids[:, :K]
        w = torch.softmax(top[:, :K], 1)
    else:
        score = torch.sigmoid(logits)
        sel = score + (bias.view(torch.bfloat16) if c["route"] == "sigmoid" else bias).double()
        if c["route"] == "group":
            per = sel.view(T, c["n_group"], -1)
            best = per.topk(2, 2).values.sum(2)
            keep = torch.zeros_like(best, dtype=torch.bool)
            keep.scatter_(1, torch.sort(best, dim=1, descending=True, stable=True).indices[:, :c["topk_group"]], True)
            sel = per.masked_fill(~keep[:, :, None], -math.inf).view(T, E)
        ids = torch.sort(sel, dim=1, descending=True, stable=True).indices[:, :K]
        w = score.gather(1, ids)
        w = w / w.sum(1, keepdim=True) * c["scaling"]
    y = torch.zeros((T, H), dtype=torch.float64, device=DEV)
    for e in torch.unique(ids).tolist():
        t, k = torch.where(ids == e)
        out = _ffn(x[t], _dense(L.gate_up, e * 2 * I, 2 * I), _dense(L.down, e * H, H))
        y.index_add_(0, t, out * w[t, k][:, None])
    if c["shared"]:
        out = _ffn(x, _dense(L.shared_gate_up, 0, 2 * I), _dense(L.shared_down, 0, H))
        if c["gate"]:
            out = out * torch.sigmoid(x @ L.shared_gate_w.view(torch.bfloat16).double())[:, None]
        y += out
    return {"y": y, "experts": ids.int(), "weights": w}


def _exact_norm(c, seed):
    s = _norm_inputs(c, seed)
    T, H = c["T"], c["H"]
    h = s["h"].double() + (s["shared"].double() if c["shared"] else 0.0)
    for k in range(c["K"]):
        rows = s["inverse"].view(T, -1)[:, k].long()
        h += s["rw"].double()[:, k, None] * s["routed"][rows].view(torch.bfloat16).double()
    out = h * torch.rsqrt(h.square().mean(1, keepdim=True) + 1e-6) * (1.0 + s["w"].view(torch.bfloat16).double())
    return {"h": h, "out": out, "out_bf": out}


def _exact_tiered(c, seed):
    lay, b, ex, w, x = _tiered_inputs(c, seed)
    T, H, I, K = c["T"], c["H"], c["I"], c["K"]

    def dense(blk, p, s, rows, cols, g):
        q = _e2m1(blk[p:p + rows * cols // 2].view(rows, -1))
        sc = blk[s:s + rows * cols // 16].view(torch.float8_e4m3fn).double().view(rows, -1)
        return q * sc.repeat_interleave(16, 1) * g
    h = torch.zeros((T, K, I), dtype=torch.float64, device=DEV)
    y = torch.zeros((T, H), dtype=torch.float64, device=DEV)
    for t in range(T):
        for k in range(K):
            blk = b[int(ex[t, k])]
            gs = blk[lay.gsc:lay.gsc + 16].view(torch.float32).double()
            gu = dense(blk, lay.gu_p, lay.gu_s, 2 * I, H, 1.0)
            hk = torch.nn.functional.silu(gu[:I] @ x[t].double() * gs[0]) * (gu[I:] @ x[t].double() * gs[1])
            h[t, k] = hk
            y[t] += w[t, k].double() * (dense(blk, lay.dn_p, lay.dn_s, H, I, gs[2]) @ hk)
    return {"h": h.view(T, -1), "y": y}


def exact(case, seed):
    if case["kind"] == "layer":
        return _exact_layer(case, seed)
    if case["kind"] == "norm":
        return _exact_norm(case, seed)
    if case["kind"] == "tiered":
        return _exact_tiered(case, seed)
    return None     # bytes: compared exactly
