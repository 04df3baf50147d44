"""Four-propagator tables: edges of the walk's 16-site tiles (k_tetra), of its
blocks of 16 operators (32 per launch) and of its steps --
operators without terms, duplicate terms, one term, every spin quad -- and
large irregular tables, which go term by term (k_tetra_terms), against the CPU
oracle.  Tolerances: FP64 1e-12 normwise, mixed 1e-6 (the paths' bounds)."""
import numpy as np
import pytest

from oracle import oracle as O
from plegma_amd import capi

import gpu_util as G

pytestmark = pytest.mark.gpu

PATTERNS = [(0, 2, 1, 3, 2, 0, 3, 1), (0, 3, 1, 2, 3, 0, 2, 1), (0, 2, 1, 3, 3, 0, 2, 1), (0, 3, 1, 2, 2, 0, 3, 1),
            (0, 2, 1, 3, 3, 1, 2, 0), (0, 3, 1, 2, 3, 1, 2, 0)]
COEFS = [1, -1, 2, 1j, -0.5, 0.25 + 0.5j]
# lattice, operators, terms of an operator, real coefficients only
CASES = [([2, 2, 2, 4], 1, 1, True), ([3, 3, 3, 4], 16, 30, True), ([17, 1, 1, 4], 17, 12, False),
         ([4, 4, 1, 4], 33, 9, False), ([5, 3, 3, 4], 64, 8, False), ([3, 3, 3, 4], 3, 900, False),
         ([3, 3, 3, 4], 7, 1500, False), ([5, 1, 1, 4], 16, 700, False)]  # these term by term


@pytest.mark.parametrize("case", range(len(CASES)))
def test_tetra_edges(case):
    torch = G.torch_cuda()
    L, nops, nterm, real = CASES[case]
    src, totalT, q2 = [1, 0, 0, 3], 3, 1
    rng = np.random.default_rng(100 + case)
    idxs, cols, vals, counts = [], [], [], []
    for k in range(nops):
        n = 0 if nops > 2 and k % 5 == 2 else nterm
        counts.append(n)
        for i in range(n):
            if i % 7 == 3:  # a duplicate: the coefficients add
                idxs.append(idxs[-1])
                cols.append(cols[-1])
            else:
                idxs.append(rng.integers(0, 4, size=8))
                cols.append(PATTERNS[rng.integers(len(PATTERNS))])
            v = complex(COEFS[rng.integers(3 if real else len(COEFS))])
            vals.append([v.real, v.imag])
    idxs, cols = np.array(idxs, dtype=np.int16), np.array(cols, dtype=np.int16)
    vals, counts = np.array(vals, dtype=np.float32), np.array(counts, dtype=np.int16)
    print(f"\n[gpu] plg_init {L} operators {nops} terms {len(idxs)}", flush=True)
    capi.init(L, 0)
    try:
        moms = capi.momlist(q2)
        P = [G.make_prop(L, 17, 50 + i, src[3], 0.4 + 0.2 * i) for i in range(4)]
        v64 = vals[:, 0].astype(np.float64) + 1j * vals[:, 1].astype(np.float64)
        ref = O.tetra_correlator(L, src, totalT, q2, [G.host(t) for t, _ in P], idxs, cols, v64, counts)
        cast = [G.cast_f32(t, v, scaled=True) for t, v in P]
        for mode, views, tol in ((capi.MODE_F64, [v for _, v in P], 1e-12),
                                 (capi.MODE_MIXED, [v for _, v in cast], 1e-6)):
            out = torch.full((nops * totalT * len(moms), 2), float("nan"), dtype=torch.float64, device="cuda")
            capi.tetraquark_table(*views, idxs, cols, vals, counts, src, totalT, moms, mode, capi.MOMENTUM_SPACE,
                                  capi.F64, out)
            torch.cuda.synchronize()
            got = torch.view_as_complex(out.cpu()).numpy().reshape(ref.shape)
            assert G.rel_err(got, ref, axis=-1) < tol, mode
    finally:
        capi.finalize()
