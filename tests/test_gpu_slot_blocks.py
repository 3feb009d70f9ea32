"""The slot kernels where a work-group takes several row blocks: enough tokens
that the items are grouped, row counts that leave a last group and a last
block partly filled, rows of one and of several chunk batches, a shared
expert; the layer against the oracle (INT8 and bf16 experts, one and several
tokens)."""
import pytest
import torch

from oracle import oracle as O
from grimoire_amd import configs, ops
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,tol", [("int8", 2e-6), ("bf16", 2e-5)])   # h in fp32; as a bf16 pair
@pytest.mark.parametrize("T,H,I,E,K,shared", [(1, 2048, 512, 16, 10, True), (3, 2064, 520, 12, 10, True),
                                              (8, 1048, 1544, 6, 6, False), (5, 4096, 264, 8, 8, True),
                                              (13, 1032, 1048, 8, 4, False)])
def test_slot_blocks(gpu, fmt, tol, T, H, I, E, K, shared):
    print(f"slot blocks {fmt} T={T} H={H} I={I} E={E} K={K} shared={shared}", flush=True)
    if fmt == "int8":
        H, I = (H + 15) // 16 * 16, (I + 15) // 16 * 16
    cfg = configs.Config("t", T, H, E, K, I, fmt, shared=shared, shared_gate=shared)
    wl = configs.make_workload(cfg, "cpu", seed=T + H)
    Lg = wl.layer.to(gpu)
    fwd = ops.MoeForward(Lg, T, configs.route_params(cfg, None), 1)
    y = torch.full((T, H), float("nan"), device=gpu)
    oe = torch.empty(T, K, dtype=torch.int32, device=gpu)
    ow = torch.empty(T, K, device=gpu)
    fwd(wl.x.to(gpu), y, oe, ow)
    torch.cuda.synchronize()
    oe, ow = oe.cpu(), ow.cpu()
    gate = None
    if shared:
        gw = (wl.layer.shared_gate_w.to(torch.int32) << 16).view(torch.float32)
        gate = torch.sigmoid(wl.x.double() @ gw.double()).float().contiguous()
    want = O.moe_forward(wl.layer.struct(), oe, ow, gate, wl.x)
    assert rel_l2(y.cpu(), want) <= tol


@pytest.mark.parametrize("fmt", ["int8", "bf16"])
@pytest.mark.parametrize("T,H,I,E,K,shared", [(3, 1008, 512, 16, 10, True), (8, 960, 1040, 12, 6, False),
                                              (6, 912, 272, 8, 8, True)])
def test_grouped_blocks_same_bits(gpu, fmt, T, H, I, E, K, shared):
    """Several row blocks an item (all tokens in a call) and one (each token
    in a call of its own, too few blocks to group): the same bits."""
    print(f"slot bits {fmt} T={T} H={H} I={I} E={E} K={K} shared={shared}", flush=True)
    cfg = configs.Config("t", T, H, E, K, I, fmt, shared=shared, shared_gate=shared)
    wl = configs.make_workload(cfg, "cpu", seed=T + H)
    Lg, x = wl.layer.to(gpu), wl.x.to(gpu)
    y, y1 = torch.empty(T, H, device=gpu), torch.empty(T, H, device=gpu)
    oe = torch.empty(T, K, dtype=torch.int32, device=gpu)
    ow = torch.empty(T, K, device=gpu)
    ops.MoeForward(Lg, T, configs.route_params(cfg, None), 1)(x, y, oe, ow)
    h, gate = torch.empty(1, K + shared, I, device=gpu), torch.empty(1, device=gpu)
    for t in range(T):
        s = slice(t, t + 1)
        if shared:
            ops.launch_moe_shared_rows(Lg, Lg.shared_gate_w, oe[s], ow[s], x[s], h, gate, y1[s], 1)
        else:
            ops.launch_moe_gate_up_batched(Lg, oe[s], x[s], h, 1)
            ops.launch_moe_down_batched(Lg, oe[s], ow[s], h, y1[s], 1)
    torch.cuda.synchronize()
    assert torch.equal(y, y1)


@pytest.mark.parametrize("fmt,K,I", [("bf16", 16, 2256), ("bf16", 8, 4512), ("int8", 16, 2368)])
def test_fills_lds(gpu, fmt, K, I):
    """Activations that leave no LDS for the dots of a second row block, with
    enough tokens to group."""
    print(f"slot lds {fmt} K={K} I={I}", flush=True)
    cfg = configs.Config("t", 8, 1024, K, K, I, fmt)
    wl = configs.make_workload(cfg, "cpu", seed=I)
    y = torch.full((8, 1024), float("nan"), device=gpu)
    oe = torch.empty(8, K, dtype=torch.int32, device=gpu)
    ow = torch.empty(8, K, device=gpu)
    ops.MoeForward(wl.layer.to(gpu), 8, configs.route_params(cfg, None), 1)(wl.x.to(gpu), y, oe, ow)
    torch.cuda.synchronize()
    want = O.moe_forward(wl.layer.struct(), oe.cpu(), ow.cpu(), None, wl.x)
    assert rel_l2(y.cpu(), want) <= 2e-5
