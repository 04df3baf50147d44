"""Meson-meson contraction (k_mesmes): edges of its 16-site tiles against the
CPU oracle -- spatial volumes below a tile, not a multiple of 16 and odd --
and two views with preparations of their own fused into the staging.
Tolerances: FP64 1e-12 normwise, mixed 1e-6 (the FP32 path's bound)."""
import pytest

from oracle import oracle as O
from plegma_amd import capi

import gpu_util as G

pytestmark = pytest.mark.gpu

LATTICES = [[2, 2, 2, 4], [3, 3, 3, 4], [6, 6, 2, 4], [5, 5, 5, 4], [4, 4, 4, 4]]


@pytest.mark.parametrize("lat", range(len(LATTICES)))
def test_mesmes_partial_tiles(lat):
    L, src, totalT, q2 = LATTICES[lat], [1, 1, 0, 2], 4, 1
    G.torch_cuda()
    print(f"\n[gpu] plg_init {L}", flush=True)
    capi.init(L, 0)
    try:
        t1, v1 = G.make_prop(L, 31, 1 + lat, src[3], 0.5)
        t2, v2 = G.make_prop(L, 31, 21 + lat, src[3], 1.2)
        k1, f1 = G.cast_f32(t1, v1, scaled=True)
        k2, f2 = G.cast_f32(t2, v2, scaled=True)
        R = G.oracle_H(O.MESON_MESON, L, src, totalT, q2, G.host(t1), G.host(t2))
        for mode, a, b, tol in ((capi.MODE_F64, v1, v2, 1e-12), (capi.MODE_MIXED, f1, f2, 1e-6)):
            H = G.shaped(G.run_correlator(capi.MESON_MESON, 0, a, b, src, totalT, q2, mode=mode), capi.MESON_MESON, 0,
                         src, totalT, q2)
            err = G.rel_err(H, R)
            print(f"[gpu] mode={mode} err {err:.2e}", flush=True)
            assert err < tol
        del k1, k2
    finally:
        capi.finalize()


@pytest.mark.parametrize("mode", ["f64", "mixed"])
def test_mesmes_prepared(mode):
    L, src, totalT, q2 = [5, 3, 5, 6], [0, 2, 1, 4], 5, 2
    torch = G.torch_cuda()
    capi.init(L, 0)
    try:
        outs, keep = [], []
        for fused in (True, False):
            views = []
            for stream, lam, rot, bc in ((1, 0.5, 1, 3), (2, 0.8, -1, 5)):
                t, v = G.make_prop(L, 7, stream, src[3], lam)
                if mode == "mixed":
                    keep.append(t)
                    t, v = G.cast_f32(t, v)
                if fused:
                    v.rotate_sign, v.bc_t0 = rot, bc
                else:
                    capi.prop_rotate_physical(v, rot)
                    capi.prop_apply_boundaries(v, bc)
                keep.append(t)
                views.append(v)
            m = capi.MODE_F64 if mode == "f64" else capi.MODE_MIXED
            outs.append(G.shaped(G.run_correlator(capi.MESON_MESON, 0, views[0], views[1], src, totalT, q2, mode=m),
                                 capi.MESON_MESON, 0, src, totalT, q2))
            torch.cuda.synchronize()
        assert G.rel_err(outs[0], outs[1]) < (1e-12 if mode == "f64" else 1e-6)
    finally:
        capi.finalize()
