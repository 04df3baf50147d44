"""The fused two-point kernel with every set of baryon groups -- none, the
proton, the Deltas, both -- in both precisions, on volumes below, beside and
above its 16-site tiles, against the CPU oracle.  Tolerances as in the baryon
tiles' test: FP64 1e-12, mixed 1e-6, per group, row and channel."""
import numpy as np
import pytest

from oracle import oracle as O
from plegma_amd import capi

import gpu_util as G

pytestmark = pytest.mark.gpu

MASKS = {"none": 0, "nucl": capi.G_NUCL, "delta": capi.G_DELTAPP_ALL, "all": capi.G_NUCL | capi.G_DELTAPP_ALL}
LATTICES = [[2, 2, 2, 4], [3, 3, 3, 4], [6, 6, 2, 4], [5, 5, 5, 4], [4, 4, 4, 4]]


@pytest.mark.parametrize("mask", sorted(MASKS))
@pytest.mark.parametrize("lat", range(len(LATTICES)))
def test_twopt_masks(lat, mask):
    L, src, totalT, q2 = LATTICES[lat], [1, 0, 1, 3], 3, 1
    G.torch_cuda()
    print(f"\n[gpu] plg_init {L} mask {mask}", flush=True)
    capi.init(L, 0)
    try:
        t, v = G.make_prop(L, 98, 21 + lat, src[3], 0.5)
        keep, f = G.cast_f32(t, v, scaled=True)
        h = G.host(t)
        R = G.oracle_H(O.MESONS16, L, src, totalT, q2, h, h)[:, :1]
        if MASKS[mask]:
            om = (O.G_NUCL if MASKS[mask] & capi.G_NUCL else 0) + \
                sum(O.G_DELTA32[k] for k in range(3) if MASKS[mask] & (capi.G_DELTAPP_11 << k))
            R = np.concatenate([R, G.oracle_H(O.BARYONS, L, src, totalT, q2, h, h, mask=om)[:, :1]], 0)
        for rot, bc in ((0, 0), (1, 3)):
            if rot:   # the preparation fused into the staging against a prepared copy
                v.rotate_sign, v.bc_t0, f.rotate_sign, f.bc_t0 = rot, bc, rot, bc
                u, w = G.make_prop(L, 98, 21 + lat, src[3], 0.5)
                capi.prop_rotate_physical(w, rot)
                capi.prop_apply_boundaries(w, bc)
                R = G.shaped(G.run_correlator(capi.TWOPT, MASKS[mask], w, w, src, totalT, q2), capi.TWOPT, MASKS[mask],
                             src, totalT, q2)
            for mode, view, tol in ((capi.MODE_F64, v, 1e-12), (capi.MODE_MIXED, f, 1e-6)):
                H = G.shaped(G.run_correlator(capi.TWOPT, MASKS[mask], view, view, src, totalT, q2, mode=mode),
                             capi.TWOPT, MASKS[mask], src, totalT, q2)
                err = G.rel_err(H, R)
                print(f"[gpu] mode={mode} rot={rot} err {err:.2e}", flush=True)
                assert H.shape == R.shape and err < tol
        del keep
    finally:
        capi.finalize()
