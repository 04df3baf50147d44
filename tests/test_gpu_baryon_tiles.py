"""Baryon contraction (k_baryon): edges of its 16-site tiles against the CPU
oracle.

A tile is staged in 16-byte units (two FP32 sites), a partial last tile
entry by entry; one wave contracts a diquark class of a dataset.  The lattices
have a spatial volume below one tile, one not a multiple of 16 and an odd one
(27 and 125 sites: FP32 site pairs off 16-byte boundaries), and every group mask
on one and two propagators, with and without the fused preparation.
Tolerances: FP64 1e-12 (27 648 products per proton site at 1.1e-16, normwise),
mixed 1e-6 (the FP32 path's bound), per group, dataset, row and channel.
"""
import numpy as np
import pytest

from oracle import oracle as O
from plegma_amd import capi

import gpu_util as G

pytestmark = pytest.mark.gpu

MASKS = {"nucl": capi.G_NUCL, "delta": capi.G_DELTAPP_ALL, "all": capi.G_NUCL | capi.G_DELTAPP_ALL}
LATTICES = [[2, 2, 2, 4], [3, 3, 3, 4], [6, 6, 2, 4], [5, 5, 5, 4], [4, 4, 4, 4]]


def _omask(mask):
    return sum(O.G_DELTA32[k] for k in range(3) if mask & (capi.G_DELTAPP_11 << k)) + \
        (O.G_NUCL if mask & capi.G_NUCL else 0)


@pytest.mark.parametrize("mask", sorted(MASKS))
@pytest.mark.parametrize("lat", range(len(LATTICES)))
def test_baryons_partial_tiles(lat, mask):
    L, src, totalT, q2 = LATTICES[lat], [1, 0, 1, 3], 3, 1
    G.torch_cuda()
    print(f"\n[gpu] plg_init {L} mask {mask}", flush=True)
    capi.init(L, 0)
    try:
        t1, v1 = G.make_prop(L, 99, 1 + lat, src[3], 0.5)
        t2, v2 = G.make_prop(L, 99, 11 + lat, src[3], 0.7)
        k1, f1 = G.cast_f32(t1, v1, scaled=True)
        k2, f2 = G.cast_f32(t2, v2, scaled=True)
        h1, h2 = G.host(t1), G.host(t2)
        for two in (False, True):
            R = G.oracle_H(O.BARYONS, L, src, totalT, q2, h1, h2 if two else h1, mask=_omask(MASKS[mask]))
            for mode, a, b, tol in ((capi.MODE_F64, v1, v2, 1e-12), (capi.MODE_MIXED, f1, f2, 1e-6)):
                H = G.shaped(G.run_correlator(capi.BARYONS, MASKS[mask], a, b if two else a, src, totalT, q2, mode=mode),
                             capi.BARYONS, MASKS[mask], src, totalT, q2)
                err = G.rel_err(H, R)
                print(f"[gpu] two={two} mode={mode} err {err:.2e}", flush=True)
                assert err < tol
        # mesons + baryons on one propagator (the mixed path's fused kernel)
        M = G.oracle_H(O.MESONS16, L, src, totalT, q2, h1, h1)[:, :1]
        B = G.oracle_H(O.BARYONS, L, src, totalT, q2, h1, h1, mask=_omask(MASKS[mask]))[:, :1]
        H = G.shaped(G.run_correlator(capi.TWOPT, MASKS[mask], f1, f1, src, totalT, q2, mode=capi.MODE_MIXED),
                     capi.TWOPT, MASKS[mask], src, totalT, q2)
        assert G.rel_err(H, np.concatenate([M, B], 0)) < 1e-6
        del k1, k2
    finally:
        capi.finalize()


@pytest.mark.parametrize("mode", ["f64", "mixed"])
def test_baryons_two_flavours_prepared(mode):
    """rotation and boundary signs of two views, each with its own, fused into
    the staging, against propagators prepared in place"""
    L, src, totalT, q2 = [5, 5, 3, 6], [0, 2, 1, 4], 5, 2
    torch = G.torch_cuda()
    capi.init(L, 0)
    try:
        outs = []
        for fused in (True, False):
            views = []
            keep = []
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
            mask = MASKS["all"]
            outs.append(G.shaped(G.run_correlator(capi.BARYONS, mask, views[0], views[1], src, totalT, q2, mode=m),
                                 capi.BARYONS, mask, src, totalT, q2))
            torch.cuda.synchronize()
        assert G.rel_err(outs[0], outs[1]) < (1e-12 if mode == "f64" else 1e-6)
    finally:
        capi.finalize()
