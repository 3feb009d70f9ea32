"""The slot kernels group row blocks only where their LDS allows it: a layer
whose activations fill a work-group's LDS runs as it does with one block an
item, up to the same size.  Host checks only."""
import ctypes as C
import os

import pytest

from grimoire_amd import _abi
from tests.test_workspace_need import _layer

pytestmark = pytest.mark.skipif(os.path.exists("/dev/kfd"), reason="made-up device addresses: no GPU may see them")


@pytest.mark.parametrize("T", [1, 8])
@pytest.mark.parametrize("K,shared,most", [(2, False, 18192), (4, False, 9088), (8, False, 4544), (8, True, 4032),
                                           (16, False, 2272), (16, True, 2128)])
def test_bf16_limit(K, shared, most, T):
    """`most`: the largest inter (a multiple of 16) of which (K + shared) rows
    and one block's dots fit 160 KiB."""
    lib = _abi.lib()
    rp, a = _abi.RouteParams(mode=_abi.ROUTE_SOFTMAX), 1 << 12
    for inter, fits in ((most - 16, True), (most + 16, False)):
        L = _layer(_abi.FMT_BF16, 4096, inter, 64, K, shared)
        n = int(lib.grimoire_moe_forward_workspace_bytes(C.byref(L), T))
        r = lib.grimoire_moe_forward(None, C.byref(L), C.byref(rp), None, a, a, T, None, None, 1, a, n)
        # a HIP error: past the checks, to the first launch (no device here)
        assert (r > 0) if fits else (r == _abi.ERR_SHAPE), (inter, r)
