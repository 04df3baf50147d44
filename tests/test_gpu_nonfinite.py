"""Entries that are not finite, and products that overflow, in the table
contractions whose operator sums run on the matrix cores (k_tetra,
k_udsc_all): they reach the operators that have a term with them, at their
site, and nothing else.  The other operators and sites keep the bits they have
with a finite entry in that place."""
import numpy as np
import pytest

from plegma_amd import capi, gen_udsc

import gpu_util as G

pytestmark = pytest.mark.gpu

PATTERNS = [(0, 2, 1, 3, 2, 0, 3, 1), (0, 3, 1, 2, 3, 0, 2, 1), (0, 2, 1, 3, 3, 0, 2, 1), (0, 3, 1, 2, 2, 0, 3, 1),
            (0, 2, 1, 3, 3, 1, 2, 0), (0, 3, 1, 2, 3, 1, 2, 0)]
L, SRC, T = [3, 3, 3, 2], [0, 0, 0, 0], 2
V3 = 27
# site, time slice, spin pair (some operators of uds, udc, usc and dsc lack it) and colour pair of the bad entry
SITE, SLICE, SPINS, COLOUR = 20, 1, (0, 1), 5
BAD = {"nan": float("nan"), "inf": float("inf"), "huge": 3e38}


def _view(t, f64):
    return capi.plg_prop(t.data_ptr(), capi.F64 if f64 else capi.F32, 0, T, 0, T * V3)


def _props(torch, n, f64):
    g = torch.Generator(device="cuda")
    g.manual_seed(4)
    return [torch.randn((144, T * V3, 2), dtype=torch.float64 if f64 else torch.float32, device="cuda", generator=g)
            for _ in range(n)]


def _check(clean, bad, hit, must):
    """clean, bad: [operator][slice][site]; hit: the operators with the entry"""
    there = np.zeros(clean.shape, bool)
    there[hit, SLICE, SITE] = True
    assert np.isfinite(clean.view(np.float64)).all()
    assert np.array_equal(bad[~there], clean[~there])
    lost = ~(np.isfinite(bad[there].real) & np.isfinite(bad[there].imag))
    assert lost.all() if must else lost.any()


@pytest.mark.parametrize("value", sorted(BAD))
@pytest.mark.parametrize("mode", ["f64", "mixed"])
@pytest.mark.parametrize("nops", [7, 20, 40])
def test_tetra_walk(nops, mode, value):
    torch = G.torch_cuda()
    f64 = mode == "f64"
    rng = np.random.default_rng(nops)
    idxs = rng.integers(0, 4, size=(nops * 8, 8)).astype(np.int16)
    cols = np.array(PATTERNS, dtype=np.int16)[rng.integers(len(PATTERNS), size=nops * 8)]
    vals = np.stack([rng.integers(1, 4, size=nops * 8), rng.integers(0, 3, size=nops * 8)], 1).astype(np.float32)
    vals[: nops * 4, 1] = 0   # the first half of the operators real
    hit = np.array([bool((idxs[8 * k:8 * k + 8, :2] == SPINS).all(1).any()) for k in range(nops)])
    assert 0 < hit.sum() < nops
    print(f"\n[gpu] plg_init {L} operators {nops} {mode} {value}", flush=True)
    capi.init(L, 0)
    try:
        P = _props(torch, 4, f64)
        outs = []
        for v in (0.25, BAD[value] if not (f64 and value == "huge") else 1e308):
            P[0].view(4, 4, 9, T, V3, 2)[SPINS[0], SPINS[1], COLOUR, SLICE, SITE, 0] = v
            out = torch.full((nops * T * V3, 2), float("nan"), dtype=torch.float64, device="cuda")
            capi.tetraquark_table(*[_view(p, f64) for p in P], idxs, cols, vals, np.full(nops, 8, dtype=np.int16), SRC, T,
                                  [], capi.MODE_F64 if f64 else capi.MODE_MIXED, capi.POSITION_SPACE, capi.F64, out)
            torch.cuda.synchronize()
            outs.append(torch.view_as_complex(out.cpu()).numpy().reshape(nops, T, V3))
        _check(outs[0], outs[1], hit, value != "huge")
    finally:
        capi.finalize()


def _operators_with(prod, table, flavour):
    """per operator of a product: a term with the bad spin pair at the flavour's
    propagator, terms that differ by an exchange of equal flavours being one"""
    hit = []
    for _, t in table:
        merged = {}
        for m, v in t.items():
            pairs = [(prod[i], m[2 * i], m[2 * i + 1]) for i in range(3)]
            key = tuple(sorted(pairs))
            merged[key] = merged.get(key, 0) + v
        hit.append(any(v != 0 and (flavour, *SPINS) in key for key, v in merged.items()))
    return hit


@pytest.mark.parametrize("value", sorted(BAD))
@pytest.mark.parametrize("mode", ["f64", "mixed"])
@pytest.mark.parametrize("flavour", ["s", "c"])
def test_udsc_products(flavour, mode, value):
    torch = G.torch_cuda()
    f64 = mode == "f64"
    tables = dict(gen_udsc.products())
    hits = [_operators_with(prod, tables[prod], flavour) for prod, _ in capi.udsc_products()]
    assert any(0 < sum(h) < len(h) for h in hits)   # operators that differ within a product
    hit = np.array([x for h in hits for x in h])
    print(f"\n[gpu] plg_init {L} {flavour} {mode} {value}", flush=True)
    capi.init(L, 0)
    try:
        P = _props(torch, 4, f64)
        V = [_view(p, f64) for p in P]
        n = capi.baryons_udsc_size(*V, SRC, T, 0, capi.POSITION_SPACE)
        outs = []
        for v in (0.25, BAD[value] if not (f64 and value == "huge") else 1e308):
            P["udsc".index(flavour)].view(4, 4, 9, T, V3, 2)[SPINS[0], SPINS[1], COLOUR, SLICE, SITE, 0] = v
            out = torch.full((n, 2), float("nan"), dtype=torch.float64, device="cuda")
            capi.baryons_udsc(*V, SRC, T, [], capi.MODE_F64 if f64 else capi.MODE_MIXED, capi.POSITION_SPACE, capi.F64, out)
            torch.cuda.synchronize()
            outs.append(torch.view_as_complex(out.cpu()).numpy().reshape(-1, T, V3))
        assert outs[0].shape[0] == len(hit)
        _check(outs[0], outs[1], hit, value != "huge")
    finally:
        capi.finalize()
