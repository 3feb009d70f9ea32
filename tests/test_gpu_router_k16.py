"""The K-split router for 33 tokens up to one round of its tiles: logits
against the oracle at ragged token / expert / K-part edges (K parts of unequal
length, waves without any), x that is not bf16 valued in some units, both tile
widths and just past the last one, and the kernels behind it; and the forward's routing, which adds the
two K halves in the top-k, from the same bits."""
import pytest
import torch

from oracle import oracle as O
from grimoire_amd import configs, ops
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,H", [(33, 1, 32), (47, 17, 96), (64, 64, 1024), (65, 33, 1056), (129, 130, 2912),
                                   (256, 512, 160), (257, 512, 160), (520, 512, 64), (1024, 128, 2048)])
@pytest.mark.parametrize("kind", ["bf16", "mixed"])
def test_router_k16(gpu, T, E, H, kind):
    print(f"router k16 T={T} E={E} H={H} {kind}", flush=True)
    g = torch.Generator().manual_seed(T + E + H)
    W = torch.randn(E, H, generator=g) * 0.02
    x = torch.randn(T, H, generator=g).bfloat16().float()
    bias = torch.randn(E, generator=g)
    if kind == "mixed":
        x[T // 2, H // 2] += 2.0 ** -12
        x[::37] = torch.randn(x[::37].shape, generator=g)
    out = torch.full((T, E), float("nan"), device=gpu)
    ops.router_logits(W.to(gpu), x.to(gpu), out)
    torch.cuda.synchronize()
    # three limbs keep 24 bits of each operand; sums of H products in fp32
    assert rel_l2(out.cpu(), x.double() @ W.double().T) < 1e-6


@pytest.mark.parametrize("T,E,H", [(4200, 64, 128), (40, 4200, 256), (4161, 65, 96), (97, 2070, 100)])
def test_router_past_one_round(gpu, T, E, H):
    """More tiles than CUs and no K long enough for the split of long
    prompts: the 64 x 64 tiles, and H that is no whole number of K tiles."""
    print(f"router past one round T={T} E={E} H={H}", flush=True)
    g = torch.Generator().manual_seed(T)
    W = torch.randn(E, H, generator=g) * 0.02
    x = torch.randn(T, H, generator=g)
    out = torch.full((T, E), float("nan"), device=gpu)
    ops.router_logits(W.to(gpu), x.to(gpu), out)
    torch.cuda.synchronize()
    assert rel_l2(out.cpu(), x.double() @ W.double().T) < 1e-6


@pytest.mark.parametrize("T,E,H", [(40, 64, 512), (150, 64, 2048), (100, 512, 576)])
def test_forward_routing_from_split_halves(gpu, T, E, H):
    print(f"router k16 forward T={T} E={E} H={H}", flush=True)
    cfg = configs.Config("t", T, H, E, 4, 512, "mxfp4", zipf=1.1)
    wl = configs.make_workload(cfg, "cpu", seed=T)
    Lg = wl.layer.to(gpu)
    bias = wl.route_bias.to(gpu)
    fwd = ops.MoeForward(Lg, T, configs.route_params(cfg, bias), 2)
    xg = wl.x.to(gpu)
    y = torch.empty(T, H, device=gpu)
    oe = torch.empty(T, 4, dtype=torch.int32, device=gpu)
    ow = torch.empty(T, 4, device=gpu)
    fwd(xg, y, oe, ow)
    lg = torch.empty(T, E, device=gpu)
    ops.router_logits(Lg.router, xg, lg)
    torch.cuda.synchronize()
    we, ww = O.topk_softmax((lg.cpu() + wl.route_bias).contiguous(), 4, True)
    assert torch.equal(oe.cpu(), we) and torch.equal(ow.cpu(), ww)
