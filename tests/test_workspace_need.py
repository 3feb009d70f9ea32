"""The smallest workspace that grimoire_moe_forward accepts does not depend
on whether the call takes the register-weight products: it is that of the
slot or grouped plan of the same call (what a caller with a size of its own
had).  Host checks only: an unknown route mode ends every call that passes
the size check before anything is launched."""
import ctypes as C

import pytest

from grimoire_amd import _abi


def _layer(fmt, H, I, E, K, shared=False):
    L = _abi.MoeLayer()
    L.cfg.hidden, L.cfg.inter, L.cfg.num_experts, L.cfg.top_k, L.cfg.norm_topk = H, I, E, K, 1
    L.router = 1 << 12
    bits = {_abi.FMT_INT4: 4, _abi.FMT_MXFP4: 4, _abi.FMT_BF16: 16}[fmt]
    ws = [(L.gate_up, E * 2 * I, H), (L.down, E * H, I)]
    if shared:
        L.has_shared = 1
        L.cfg.shared_inter = I
        ws += [(L.shared_gate_up, 2 * I, H), (L.shared_down, H, I)]
    for w, n, k in ws:
        w.fmt, w.N, w.K, w.row_bytes = fmt, n, k, k * bits // 8
        w.row_scales = {_abi.FMT_INT4: k // 128, _abi.FMT_MXFP4: k // 32, _abi.FMT_BF16: 0}[fmt]
        w.payload = w.scales = w.zeros = 1 << 20
    return L


def _need(L, T, regime):
    """Smallest workspace_bytes not refused as too small."""
    lib = _abi.lib()
    rp = _abi.RouteParams(mode=99)

    def fits(n):
        r = lib.grimoire_moe_forward(None, C.byref(L), C.byref(rp), None, 1 << 12, 1 << 12, T, None, None, regime,
                                     1 << 12, n)
        assert r in (_abi.ERR_WORKSPACE, _abi.ERR_SHAPE, _abi.ERR_ARG)
        return r != _abi.ERR_WORKSPACE

    lo, hi = 0, int(lib.grimoire_moe_forward_workspace_bytes(C.byref(L), T))
    assert fits(hi)
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if fits(mid) else (mid, hi)
    return hi


@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("T", [1, 17, 200, 1000])
@pytest.mark.parametrize("fmt,H,I", [(_abi.FMT_MXFP4, 2880, 2880), (_abi.FMT_MXFP4, 2048, 768),
                                     (_abi.FMT_BF16, 2048, 1024)])
def test_gemm_regime_need(fmt, H, I, T, shared):
    # regime 4 never takes the register-weight products, regime 2 does
    L = _layer(fmt, H, I, 64, 4, shared)
    assert _need(L, T, 2) == _need(L, T, 4)


@pytest.mark.parametrize("T", [2, 8, 9, 16])
def test_int4_slots_need(T):
    # regime 3: the slot kernels for any T they cover
    L = _layer(_abi.FMT_INT4, 4096, 2048, 64, 4)
    assert _need(L, T, 0) == _need(L, T, 3)
