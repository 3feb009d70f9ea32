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
