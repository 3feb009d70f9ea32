"""Tiered NVFP4 experts with the activations staged in LDS, against the oracle
where the staged kernels' items can go wrong: enough tokens that a work-group
takes several row blocks, a last group and a last block partly filled, 1, 2
and 4 x 4 slots over four and eight waves, rows of several chunk iterations,
skipped slots; and a down too wide to stage.  Outputs within 1e-5 of the
largest (fp32 sums in another order); a token's bits do not depend on the
batch, and so not on the kernel or the row blocks per work-group."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from grimoire_amd import tiered
from tests.test_oracle_tiered import make_block

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,I,K,E,M", [(128, 128, 1, 2, 1), (640, 384, 4, 5, 70), (2176, 128, 8, 9, 9),
                                       (384, 2176, 9, 10, 3), (4224, 256, 16, 17, 2), (256, 1536, 14, 15, 2)])
def test_tmoe_staged(gpu, H, I, K, E, M):
    print(f"tmoe staged H={H} I={I} K={K} E={E} M={M}", flush=True)
    lay = O.tmoe_layout(H, I)
    rng = np.random.default_rng(H + I)
    blocks_np = [make_block(lay, rng) for _ in range(E)]
    layer = tiered.TieredLayer(H, I, K, [torch.from_numpy(b).to(gpu) for b in blocks_np], gpu)
    ex = np.stack([rng.permutation(E + 1)[:K] - 1 for _ in range(M)]).astype(np.int32)   # -1: skipped
    w = rng.random((M, K)).astype(np.float32)
    w[-1, 0] = 0.0
    x = rng.standard_normal((M, H)).astype(np.float32)
    exd, wd, xd = (torch.from_numpy(a).to(gpu) for a in (ex, w, x))
    h = torch.full((M, K * I), float("nan"), device=gpu)
    y = torch.full((M, H), float("nan"), device=gpu)
    layer.gate_up(exd, xd, h)
    layer.down(exd, wd, h, y)
    torch.cuda.synchronize()
    hc = h.cpu().numpy()
    for got, want in ((hc, O.tmoe_gate_up(blocks_np, H, I, K, ex, x, M)),
                      (y.cpu().numpy(), O.tmoe_down(blocks_np, H, I, K, ex, w, hc, M))):
        assert np.abs(got - want).max() <= 1e-5 * max(np.abs(want).max(), 1e-30)


@pytest.mark.parametrize("H,I,K,E,M", [(1280, 1152, 4, 6, 7), (1280, 1152, 16, 20, 4), (1024, 384, 8, 9, 40),
                                       (2048, 768, 9, 12, 5), (384, 2176, 2, 4, 600)])
def test_tmoe_bits_do_not_depend_on_the_batch(gpu, H, I, K, E, M):
    """One token takes other row blocks per work-group than M do, and at 1280
    x 1152, 4 slots, the unstaged down."""
    print(f"tmoe batch bits H={H} I={I} K={K} E={E} M={M}", flush=True)
    rng = np.random.default_rng(H + I + M)
    lay = O.tmoe_layout(H, I)
    layer = tiered.TieredLayer(H, I, K, [torch.from_numpy(make_block(lay, rng)).to(gpu) for _ in range(E)], gpu)
    ex = torch.from_numpy(np.stack([rng.permutation(E)[:K] for _ in range(M)]).astype(np.int32)).to(gpu)
    w = torch.from_numpy(rng.random((M, K)).astype(np.float32)).to(gpu)
    x = torch.from_numpy(rng.standard_normal((M, H)).astype(np.float32)).to(gpu)

    def run(lo, hi):
        h = torch.full((hi - lo, K * I), float("nan"), device=gpu)
        y = torch.full((hi - lo, H), float("nan"), device=gpu)
        layer.gate_up(ex[lo:hi], x[lo:hi], h)
        layer.down(ex[lo:hi], w[lo:hi], h, y)
        return h, y
    h, y = run(0, M)
    for t in sorted({0, M // 2, M - 1}):
        h1, y1 = run(t, t + 1)
        assert torch.equal(h1[0], h[t]) and torch.equal(y1[0], y[t]), t
