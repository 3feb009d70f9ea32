"""The one-work-group dispatch (batches of up to 8192 routes over up to 512
experts) against a stable sort, at the sizes where its waves, batches of 64
routes and expert bits end, and just past its limits, where the launches of
the larger batches take over: counts, offsets, rows, token map and tile table
exactly, with skipped routes."""
import pytest
import torch

from grimoire_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,K,E", [(1, 1, 1), (1, 16, 512), (63, 1, 3), (65, 1, 257), (128, 8, 512), (205, 5, 64),
                                   (1000, 4, 128), (1024, 8, 512), (1025, 8, 512), (500, 2, 513)])
def test_dispatch_one(gpu, T, K, E):
    print(f"dispatch one T={T} K={K} E={E}", flush=True)
    g = torch.Generator().manual_seed(T + E)
    ids = torch.randint(0, E, (T, K), generator=g)
    ids = torch.where(torch.rand((T, K), generator=g) < 0.3, torch.zeros_like(ids), ids)     # one popular expert
    ids = torch.where(torch.rand((T, K), generator=g) < 0.05, torch.full_like(ids, -1), ids)   # skipped
    R, mc = T * K, 4
    tmax = E + R // mc + 3
    i32 = lambda n: torch.full((n,), -7, dtype=torch.int32, device=gpu)
    counts, offsets, inverse, perm, te, tm = i32(E), i32(E), i32(R), i32(R), i32(tmax), i32(tmax)
    ops.launch_moe_route_grouped(None, ids.int().to(gpu), None, None, counts, offsets, inverse, te, tm, tmax, T, 8, E,
                                 mc, K, perm_token=perm)
    torch.cuda.synchronize()
    flat = ids.flatten()
    valid = flat >= 0
    want_counts = torch.bincount(flat[valid], minlength=E)
    order = torch.argsort(torch.where(valid, flat, torch.full_like(flat, E)), stable=True)[:int(valid.sum())]
    want_inv = torch.full((R,), -1, dtype=torch.int64)
    want_inv[order] = torch.arange(order.numel())
    assert torch.equal(counts.cpu().long(), want_counts)
    assert torch.equal(offsets.cpu().long(), torch.cumsum(want_counts, 0) - want_counts)
    assert torch.equal(inverse.cpu().long(), want_inv)
    assert torch.equal(perm.cpu().long()[:order.numel()], order // K)
    tiles = [(e, b) for e in range(E) for b in range((int(want_counts[e]) + mc - 1) // mc)]
    tiles += [(-1, 0)] * (tmax - len(tiles))
    assert list(zip(te.cpu().tolist(), tm.cpu().tolist())) == tiles
