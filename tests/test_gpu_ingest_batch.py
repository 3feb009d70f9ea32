"""GPTQ ingestion of many projections at once (grimoire_moe_ingest_projections):
byte-exact against the oracle around the batch of one launch and the edges of
its transpose tiles (64 words) and of its scale blocks (256 items)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from grimoire_amd import _abi, ingest
from tests.test_gpu_ingest import _gptq_src

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,out,inn,group", [(1, 8, 32, 32), (127, 8, 64, 32), (128, 16, 512, 32), (129, 16, 32, 32),
                                             (3, 64, 512, 128), (3, 72, 544, 32), (2, 256, 1056, 96)])
def test_batches(gpu, n, out, inn, group):
    print(f"gptq ingest n={n} out={out} in={inn} g={group}", flush=True)
    made = [_gptq_src(out, inn, group, 7 + i, gpu) for i in range(n)]
    dst = ingest.stacked(ingest.target_format(_abi.SRC_GPTQ), (n + 1) * out, inn, group, gpu)
    dst.payload.fill_(0x5A); dst.scales.fill_(0x1234); dst.zeros.fill_(0xA5)
    # the projections in reverse order, the first rows left alone
    rows = [(n - i) * out for i in range(n)]
    ingest.ingest_projections([m[0] for m in made], dst, rows)
    torch.cuda.synchronize()
    pay, scl, zer = dst.payload.cpu().numpy(), dst.scales.cpu().numpy(), dst.zeros.cpu().numpy()
    for (_, src), r in zip(made, rows):
        p, s, z = O.gptq_repack(*src, inn, out, group, keep_f16=False)
        assert np.array_equal(pay[r:r + out], p)
        assert np.array_equal(scl[r:r + out], s)
        assert np.array_equal(zer[r:r + out], z)
    assert (pay[:out] == 0x5A).all() and (scl[:out] == 0x1234).all() and (zer[:out] == 0xA5).all()
