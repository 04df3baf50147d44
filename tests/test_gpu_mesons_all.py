"""contractMesonsAll (k_meson_all): edges of its 16-site rows against the CPU
oracle -- spatial volumes below a row, odd, one over a workgroup -- and views
with rotations and boundary signs of their own fused into the load against
prepared copies.  Tolerances: FP64 1e-12 normwise, mixed 1e-6 (the FP32 path's
bound)."""
import pytest

from oracle import oracle as O
from plegma_amd import capi

import gpu_util as G

pytestmark = pytest.mark.gpu

LATTICES = [[2, 2, 2, 4], [3, 3, 3, 4], [13, 5, 1, 4], [4, 4, 4, 4]]


@pytest.mark.parametrize("lat", range(len(LATTICES)))
def test_mesons_all_partial_rows(lat):
    L, src, totalT, q2 = LATTICES[lat], [1, 1, 0, 2], 4, 1
    G.torch_cuda()
    print(f"\n[gpu] plg_init {L}", flush=True)
    capi.init(L, 0)
    try:
        t1, v1 = G.make_prop(L, 37, 1 + lat, src[3], 0.5)
        t2, v2 = G.make_prop(L, 37, 21 + lat, src[3], 0.9)
        k1, f1 = G.cast_f32(t1, v1, scaled=True)
        k2, f2 = G.cast_f32(t2, v2, scaled=True)
        R = G.oracle_H(O.MESONS_ALL, L, src, totalT, q2, G.host(t1), G.host(t2))
        for mode, a, b, tol in ((capi.MODE_F64, v1, v2, 1e-12), (capi.MODE_MIXED, f1, f2, 1e-6)):
            H = G.shaped(G.run_correlator(capi.MESONS_ALL, 0, a, b, src, totalT, q2, mode=mode), capi.MESONS_ALL, 0,
                         src, totalT, q2)
            assert G.rel_err(H, R) < tol, mode
        del k1, k2
    finally:
        capi.finalize()


@pytest.mark.parametrize("mode,tol", [("f64", 1e-12), ("mixed", 1e-6)])
@pytest.mark.parametrize("rots", [(1, -1), (0, 1), (-1, 0)])
def test_mesons_all_prepared(mode, tol, rots):
    L, src, totalT, q2 = [5, 3, 5, 6], [0, 2, 1, 4], 5, 2
    torch = G.torch_cuda()
    capi.init(L, 0)
    try:
        outs, keep = [], []
        for fused in (True, False):
            views = []
            for stream, lam, rot, bc in ((1, 0.5, rots[0], 3), (2, 0.8, rots[1], 5)):
                t, v = G.make_prop(L, 7, stream, src[3], lam)
                if mode == "mixed":
                    keep.append(t)
                    t, v = G.cast_f32(t, v)
                if fused:
                    v.rotate_sign, v.bc_t0 = rot, bc
                else:
                    if rot:
                        capi.prop_rotate_physical(v, rot)
                    capi.prop_apply_boundaries(v, bc)
                keep.append(t)
                views.append(v)
            outs.append(G.shaped(G.run_correlator(capi.MESONS_ALL, 0, *views, src, totalT, q2,
                                                  mode=capi.MODE_F64 if mode == "f64" else capi.MODE_MIXED),
                                 capi.MESONS_ALL, 0, src, totalT, q2))
            torch.cuda.synchronize()
        assert G.rel_err(outs[0], outs[1]) < tol
    finally:
        capi.finalize()
