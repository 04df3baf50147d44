"""Four-propagator tables: the choice between the walk over distinct products
(k_tetra) and the terms one by one (k_tetra_terms) by the table and the number
of workgroups.

A large irregular table goes term by term where its sites fill the chip and by
the walk where they do not: a call over all slices against calls of one slice
each, the walk itself being held to the oracle elsewhere.  Both hold it to
1e-12 (FP64) and 1e-6 (mixed) normwise, so they agree within twice that, and
not bit for bit."""
import time

import numpy as np
import pytest

from plegma_amd import capi

import gpu_util as G

pytestmark = pytest.mark.gpu

DIRECT = [(0, 2, 1, 3, 2, 0, 3, 1), (0, 3, 1, 2, 3, 0, 2, 1)]
MIXED = DIRECT + [(0, 2, 1, 3, 3, 0, 2, 1), (0, 3, 1, 2, 2, 0, 3, 1)]
SWAPPED = DIRECT + [(0, 2, 1, 3, 3, 1, 2, 0), (0, 3, 1, 2, 3, 1, 2, 0)]   # both pairings: two sets


def _table(rng, nops, nterm, patterns):
    n = nops * nterm
    idxs = rng.integers(0, 4, size=(n, 8)).astype(np.int16)
    cols = np.array(patterns, dtype=np.int16)[rng.integers(len(patterns), size=n)]
    vals = rng.integers(1, 4, size=(n, 2)).astype(np.float32)
    return idxs, cols, vals, np.full(nops, nterm, dtype=np.int16)


def _views(torch, f64, V3, T):
    g = torch.Generator(device="cuda")
    g.manual_seed(2)
    keep = [torch.randn((144, T * V3, 2), dtype=torch.float64 if f64 else torch.float32, device="cuda", generator=g)
            for _ in range(4)]
    return keep, [capi.plg_prop(t.data_ptr(), capi.F64 if f64 else capi.F32, 0, T, 0, T * V3) for t in keep]


@pytest.mark.parametrize("mode", ["f64", "mixed"])
@pytest.mark.parametrize("shape", [(16, 768, DIRECT), (7, 1500, MIXED), (33, 500, SWAPPED)],
                         ids=["direct", "mixed", "swapped"])
def test_both_forms_agree(shape, mode):
    torch = G.torch_cuda()
    f64 = mode == "f64"
    nops, nterm, patterns = shape
    L, T = [16, 16, 16, 8], 8
    V3 = 4096
    tab = _table(np.random.default_rng(nops), nops, nterm, patterns)
    m = capi.MODE_F64 if f64 else capi.MODE_MIXED
    print(f"\n[gpu] plg_init {L} {nops} x {nterm} {mode}", flush=True)
    capi.init(L, 0)
    try:
        keep, views = _views(torch, f64, V3, T)

        def call(t0, n):
            out = torch.full((nops * n * V3, 2), float("nan"), dtype=torch.float64, device="cuda")
            capi.tetraquark_table(*views, *tab, [0, 0, 0, t0], n, [], m, capi.POSITION_SPACE, capi.F64, out)
            torch.cuda.synchronize()
            return torch.view_as_complex(out.cpu()).numpy().reshape(nops, n, V3)

        whole = call(0, T)
        slices = np.concatenate([call(t, 1) for t in range(T)], 1)
        assert np.isfinite(whole.view(np.float64)).all()
        assert not np.array_equal(whole, slices)
        assert G.rel_err(whole, slices, axis=-1) < (2e-12 if f64 else 2e-6)
        assert np.array_equal(call(0, T), whole)    # each form kept and found again
        assert np.array_equal(call(3, 1)[:, 0], slices[:, 3])
        del keep
    finally:
        capi.finalize()


def test_small_tables_on_small_lattices_take_the_walk():
    """64 operators of 40 irregular terms on 8^3 x 8 sites: 0.18 ms by the
    walk, 1.6 ms term by term; the limit lies between"""
    torch = G.torch_cuda()
    L, T = [8, 8, 8, 8], 8
    tab = _table(np.random.default_rng(1), 64, 40, MIXED)
    capi.init(L, 0)
    try:
        moms = capi.momlist(1)
        for f64 in (True, False):
            keep, views = _views(torch, f64, 512, T)
            out = torch.empty((64 * T * len(moms), 2), dtype=torch.float64, device="cuda")
            best = 1.0
            for _ in range(20):
                t0 = time.perf_counter()
                capi.tetraquark_table(*views, *tab, [0, 0, 0, 0], T, moms, capi.MODE_F64 if f64 else capi.MODE_MIXED,
                                      capi.MOMENTUM_SPACE, capi.F64, out)
                best = min(best, time.perf_counter() - t0)
            print(f"[gpu] f64={f64}: {best * 1e3:.2f} ms", flush=True)
            assert best < 0.6e-3
            del keep
    finally:
        capi.finalize()
