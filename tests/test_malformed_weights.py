"""A layer whose weights do not cover what its configuration says (too few
rows, null scales or payload, a payload off its alignment, another K) is
refused with the slot kernels' error before anything is launched, also where
the call would take the register-weight products: host checks only."""
import ctypes as C
import os

import pytest

from grimoire_amd import _abi
from tests.test_workspace_need import _layer

# (an intact layer's call would reach a launch)
pytestmark = pytest.mark.skipif(os.path.exists("/dev/kfd"), reason="made-up device addresses: no GPU may see them")

BREAK = {
    "rows": (lambda w: setattr(w, "N", w.N - 1), _abi.ERR_SHAPE),
    "k": (lambda w: setattr(w, "K", w.K - 128), _abi.ERR_SHAPE),
    "payload": (lambda w: setattr(w, "payload", None), _abi.ERR_ARG),
    "aligned": (lambda w: setattr(w, "payload", (1 << 20) + 8), _abi.ERR_ARG),
    "scales": (lambda w: setattr(w, "scales", None), _abi.ERR_ARG),
}


def _forward(L, T, shard=0):
    lib = _abi.lib()
    rp, a = _abi.RouteParams(mode=_abi.ROUTE_SOFTMAX), 1 << 12
    n = int(lib.grimoire_moe_forward_workspace_bytes(C.byref(L), T))
    if shard:
        return lib.grimoire_moe_forward_shard(None, C.byref(L), C.byref(rp), None, a, a, T, None, None, 0, 0, shard, a, n)
    return lib.grimoire_moe_forward(None, C.byref(L), C.byref(rp), None, a, a, T, None, None, 0, a, n)


@pytest.mark.parametrize("what", BREAK)
@pytest.mark.parametrize("name", ["gate_up", "down", "shared_gate_up", "shared_down"])
def test_int4_refused(name, what):
    # 12 tokens x top-4: INT4 batches that the rule on bytes moves off the slot kernels
    L = _layer(_abi.FMT_INT4, 4096, 2048, 64, 4, shared=True)
    brk, want = BREAK[what]
    brk(getattr(L, name))
    assert _forward(L, 12) == want


def test_shard_counts_its_own_rows():
    """A shard's weights hold its own experts' rows: 8 of 64 are enough for a
    shard of 8, not for one of 16."""
    L = _layer(_abi.FMT_INT4, 4096, 2048, 64, 4)
    L.gate_up.N, L.down.N = 8 * 2 * 2048, 8 * 4096
    assert _forward(L, 12, shard=16) == _abi.ERR_SHAPE
    assert _forward(L, 12, shard=8) > 0       # past the checks, to the first launch (no device here)
