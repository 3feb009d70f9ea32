"""The register-weight expert products (grimoire_moe_forward on MXFP4, bf16
and INT4 batches) against the oracle where their tiles can go wrong: row
counts around the 16 / 32 / 64 / 128-row blocks, one expert with every token
and experts with none, K and N with half-filled last segments, scale rows
whose last window is read early, signed and missing INT4 zero points,
activations that need their low halves, both INT4 scale formats, every routing
mode in the dispatch launch, and a shared expert."""
import dataclasses

import pytest
import torch

from oracle import oracle as O
from grimoire_amd import _abi, configs, ops
from grimoire_amd.weights import Weight
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu

# x and the weights are exact in bf16; h is a bf16 pair (2^-17 relative per
# element) and the sums are fp32: 2^-17 plus a few fp32 roundings of sums of
# a few thousand terms, far below 2e-5.
TOL = 2e-5


def _run(gpu, cfg, seed, zeros=None, fp32_x=False, regime=0):
    wl = configs.make_workload(cfg, "cpu", seed=seed)
    L, x = wl.layer, wl.x
    if zeros is not None:
        g = torch.Generator().manual_seed(seed)
        for name in ("gate_up", "down", "shared_gate_up", "shared_down"):
            w = getattr(L, name)
            if w is not None:
                z = torch.randint(0, 16, w.scales.shape, dtype=torch.uint8, generator=g)
                z[torch.rand(z.shape, generator=g) < zeros] = 0xFF       # signed codes
                setattr(L, name, Weight(w.fmt, w.N, w.K, w.payload, w.scales, z, w.row_scales))
    if fp32_x:
        rows = torch.arange(cfg.T) % 3 == 1
        x = torch.where(rows[:, None], torch.randn(x.shape, generator=torch.Generator().manual_seed(5)), x).contiguous()
    # expert 0 takes every token, the last one none
    bias = torch.zeros(cfg.E)
    bias[0], bias[-1] = 50.0, -50.0
    Lg = L.to(gpu)
    bg = bias.to(gpu)
    fwd = ops.MoeForward(Lg, cfg.T, configs.route_params(cfg, bg), regime)
    xg = x.to(gpu)
    y = torch.full((cfg.T, cfg.H), float("nan"), device=gpu)
    oe = torch.empty(cfg.T, cfg.K, dtype=torch.int32, device=gpu)
    ow = torch.empty(cfg.T, cfg.K, device=gpu)
    fwd(xg, y, oe, ow)
    torch.cuda.synchronize()
    oe, ow = oe.cpu(), ow.cpu()
    assert (oe[:, 0] == 0).all() and (oe != cfg.E - 1).all()
    gate = None
    if L.has_shared and L.shared_gate_w is not None:
        gw = (L.shared_gate_w.to(torch.int32) << 16).view(torch.float32)
        gate = torch.sigmoid(x.double() @ gw.double()).float().contiguous()
    want = O.moe_forward(L.struct(), oe, ow, gate, x)
    err = rel_l2(y.cpu(), want)
    assert err <= TOL, err


@pytest.mark.parametrize("T", [1, 16, 17, 32, 33, 64, 65, 128, 129, 193])
@pytest.mark.parametrize("fmt", ["mxfp4", "bf16"])
def test_row_blocks(gpu, fmt, T):
    print(f"wreg {fmt} T={T}", flush=True)
    _run(gpu, configs.Config("t", T, 576, 6, 3, 704, fmt, shared=T % 2 == 1, shared_gate=T % 4 == 1), seed=T, regime=2)


@pytest.mark.parametrize("H,I", [(512, 576), (2112, 512), (2880, 1024), (4096, 640)])
def test_mxfp4_scale_windows(gpu, H, I):
    """Scale rows of 16, 18, 20, 66, 90 and 128 bytes: whole, early and
    several chunks of windows."""
    print(f"wreg mxfp4 H={H} I={I}", flush=True)
    _run(gpu, configs.Config("t", 40, H, 5, 2, I, "mxfp4"), seed=H, regime=2)


@pytest.mark.parametrize("H,I", [(512, 640), (2176, 512), (2688, 896)])
@pytest.mark.parametrize("zeros,fp32_x", [(None, False), (0.5, False), (0.0, True), (None, True)])
def test_int4(gpu, H, I, zeros, fp32_x):
    print(f"wreg int4 H={H} I={I} zeros={zeros} fp32_x={fp32_x}", flush=True)
    _run(gpu, configs.Config("t", 35, H, 36, 2, I, "int4", shared=True), seed=H, zeros=zeros, fp32_x=fp32_x)


@pytest.mark.parametrize("fmt,T,regime", [("int4", 35, 0), ("bf16", 150, 2), ("mxfp4", 1500, 2)])
def test_shards_sum_to_the_layer(gpu, fmt, T, regime):
    """Shards of 12 of 36 experts (routes elsewhere are -1), both dispatch
    routes: each y is the layer's part, the sum the whole layer."""
    print(f"wreg shards {fmt} T={T}", flush=True)
    cfg = configs.Config("t", T, 512, 36, 6 if T > 1000 else 2, 640, fmt)
    Lg = configs.make_workload(cfg, "cpu", seed=T).layer.to(gpu)
    x = configs.make_x(cfg, "cpu", seed=T).to(gpu)
    rp = configs.route_params(cfg, None)
    y = torch.empty(T, cfg.H, device=gpu)
    ops.MoeForward(Lg, T, rp, regime)(x, y)
    total = torch.zeros(T, cfg.H, dtype=torch.float64, device=gpu)
    for b in (0, 12, 24):
        ys = torch.full((T, cfg.H), float("nan"), device=gpu)
        ops.MoeForward(Lg.shard(b, 12, shared=False), T, rp, regime).shard(x, ys, b, 12)
        total += ys.double()
    torch.cuda.synchronize()
    assert torch.isfinite(total).all()
    assert rel_l2(total.float().cpu(), y.cpu()) <= TOL


@pytest.mark.parametrize("fmt,T,regime", [("int4", 16, 0), ("int4", 35, 0), ("bf16", 150, 2), ("mxfp4", 1500, 2)])
def test_graph_replays(gpu, fmt, T, regime):
    """Captured once, replayed on new inputs between eager calls: the bits of
    the eager call."""
    print(f"wreg graph {fmt} T={T}", flush=True)
    # T = 16: the rule on bytes (55 MB of slot reads), top-k in the dispatch launch
    cfg = configs.Config("t", T, 2048 if T == 16 else 512, 36, 6 if T > 1000 else 2, 640, fmt, shared=T != 16)
    Lg = configs.make_workload(cfg, "cpu", seed=T).layer.to(gpu)
    fwd = ops.MoeForward(Lg, T, configs.route_params(cfg, None), regime)
    xs = [configs.make_x(cfg, "cpu", seed=s).to(gpu) for s in (1, 2)]
    x, y, ye = xs[0].clone(), torch.empty(T, cfg.H, device=gpu), torch.empty(T, cfg.H, device=gpu)
    fwd(x, y)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        fwd(x, y, stream=s)
    for rep in range(3):
        for xi in xs:
            fwd(xi, ye)
            x.copy_(xi)
            y.fill_(float("nan"))
            torch.cuda.synchronize()
            with torch.cuda.stream(s):
                g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, ye), f"replay {rep}"


def _widen(w):
    """The weight with 16 bytes of other rows' codes behind each row."""
    p = torch.cat((w.payload, w.payload.flip(0)[:, :16]), 1).contiguous()
    return Weight(w.fmt, w.N, w.K, p, w.scales, w.zeros, w.row_scales)


def test_int4_rows_with_a_stride(gpu):
    """Up to 64 routes such rows give the packed rows' values (16 tokens: the
    rule on bytes): the same products, but rows of whole kilobytes start their
    K walk at another place per column tile, so the fp32 sums of 2048 terms
    run in another order (a bound as for the oracle); above, no path but this one could take them and the call
    ends in the format error it always had."""
    cfg = configs.Config("t", 35, 2048, 36, 2, 768, "int4")
    L = configs.make_layer(cfg, "cpu", seed=3).to(gpu)
    wide = dataclasses.replace(L, gate_up=_widen(L.gate_up), down=_widen(L.down))
    x = configs.make_x(cfg, "cpu", seed=3).to(gpu)
    rp = configs.route_params(cfg, None)
    y, yw = torch.empty(16, cfg.H, device=gpu), torch.empty(16, cfg.H, device=gpu)
    ops.MoeForward(L, 16, rp)(x[:16], y)
    ops.MoeForward(wide, 16, rp)(x[:16], yw)
    assert rel_l2(yw.cpu(), y.cpu()) <= TOL
    y = torch.empty(35, cfg.H, device=gpu)
    ops.MoeForward(L, 35, rp)(x, y)
    with pytest.raises(_abi.GrimoireError):
        ops.MoeForward(wide, 35, rp)(x, y)
    torch.cuda.synchronize()


@pytest.mark.parametrize("H,I", [(512, 640), (2688, 896)])
@pytest.mark.parametrize("zeros", [None, 0.0, 0.5])
def test_int4_bf16_scales(gpu, H, I, zeros):
    """The format that ingestion writes by default: bf16 scales, a zero point
    per group (some 0xFF: signed codes), or none (zero point 0)."""
    print(f"wreg int4 bf16 scales H={H} I={I} zeros={zeros}", flush=True)
    cfg = configs.Config("t", 35, H, 36, 2, I, "int4", shared=True)
    wl = configs.make_workload(cfg, "cpu", seed=H)
    L, g = wl.layer, torch.Generator().manual_seed(H)
    for name in ("gate_up", "down", "shared_gate_up", "shared_down"):
        w = getattr(L, name)
        z = None
        if zeros is not None:
            z = torch.randint(0, 16, w.scales.shape, dtype=torch.uint8, generator=g)
            z[torch.rand(z.shape, generator=g) < zeros] = 0xFF
        sc = w.scales.view(torch.float16).bfloat16().view(torch.int16)
        setattr(L, name, Weight(_abi.FMT_INT4, w.N, w.K, w.payload, sc, z, w.row_scales))
    y = torch.full((cfg.T, H), float("nan"), device=gpu)
    oe = torch.empty(cfg.T, cfg.K, dtype=torch.int32, device=gpu)
    ow = torch.empty(cfg.T, cfg.K, device=gpu)
    ops.MoeForward(L.to(gpu), cfg.T, configs.route_params(cfg, None))(wl.x.to(gpu), y, oe, ow)
    torch.cuda.synchronize()
    assert rel_l2(y.cpu(), O.moe_forward(L.struct(), oe.cpu(), ow.cpu(), None, wl.x)) <= TOL


@pytest.mark.parametrize("route", [_abi.ROUTE_SOFTMAX, _abi.ROUTE_SIGMOID, _abi.ROUTE_GROUP])
@pytest.mark.parametrize("fmt,T,regime", [("int4", 16, 0), ("int4", 11, 0), ("bf16", 13, 2), ("mxfp4", 1, 2)])
def test_topk_in_the_dispatch_launch(gpu, fmt, T, regime, route):
    """Up to 16 tokens the top-k runs in the dispatch launch: its experts and
    weights are the bits of the slot path's top-k, in each routing mode."""
    print(f"wreg route fmt={fmt} T={T} route={route}", flush=True)
    cfg = configs.Config("t", T, 2048, 64, 4, 896, fmt, route=route, bias_std=0.05, scaling=2.5,
                         n_group=8 if route == _abi.ROUTE_GROUP else 0, topk_group=3 if route == _abi.ROUTE_GROUP else 0)
    wl = configs.make_workload(cfg, "cpu", seed=T + route)
    bias = None if wl.route_bias is None else wl.route_bias.to(gpu)
    L, x = wl.layer.to(gpu), wl.x.to(gpu)
    got = []
    for r in (regime, 3):
        y = torch.full((T, cfg.H), float("nan"), device=gpu)
        oe = torch.empty(T, cfg.K, dtype=torch.int32, device=gpu)
        ow = torch.empty(T, cfg.K, device=gpu)
        ops.MoeForward(L, T, configs.route_params(cfg, bias), r)(x, y, oe, ow)
        got.append((y, oe, ow))
    torch.cuda.synchronize()
    assert torch.equal(got[0][1], got[1][1]) and torch.equal(got[0][2], got[1][2])
    want = O.moe_forward(wl.layer.struct(), got[0][1].cpu(), got[0][2].cpu(), None, wl.x)
    assert rel_l2(got[0][0].cpu(), want) <= TOL
