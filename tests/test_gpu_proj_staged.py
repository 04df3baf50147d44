"""The separable projection's staged form (k_sep_xy) on lines that are not
whole groups of 4 sites, with few and with many momentum components: plane
heights of 8 and 16 lines a chunk, lines in one and two parts, partial column
groups.  Through plg_ft_apply against the exact-phase DFT in complex128 (the
sums run in FP64 and an FP32 field converts exactly: 1e-12 normwise), and a
batch on these lattices to show which form runs: the separable one where a chunk
of 8 lines (16 of an odd line) is within 256 FP32 or 128 FP64 sites, else the
phase-matrix GEMM."""
import math

import numpy as np
import pytest

from plegma_amd import capi

import gpu_util as G

pytestmark = pytest.mark.gpu

LATTICES = [[6, 8, 3], [10, 16, 2], [14, 8, 5], [3, 16, 4], [2, 8, 2], [18, 24, 1], [30, 8, 2]]


def _lists(L):
    few = capi.momlist(4)                       # at most five classes each way: the small tables
    many = [(x, y, z) for x in range(-min(3, L[0] // 2), min(6, (L[0] + 1) // 2)) for y in (-4, -1, 0, 2, 5)
            for z in (0, 1)]
    some = [(L[0] // 2, 0, 1), (1, L[1] // 2, 0), (-1, 1, 0), (1 + L[0], -1, 2), (0, 2, -L[2])]
    return {"few": few, "many": many, "some": some, "one": [(1, -2, 1)]}


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("lat", range(len(LATTICES)))
def test_staged_form(lat, prec):
    torch = G.torch_cuda()
    L = LATTICES[lat] + [2]
    assert L[0] % 4 and L[0] * L[1] % 16 == 0
    print(f"\n[gpu] plg_init {L} {prec}", flush=True)
    capi.init(L, 0)
    try:
        V3 = L[0] * L[1] * L[2]
        dt = torch.float32 if prec == "f32" else torch.float64
        g = torch.Generator(device="cuda")
        g.manual_seed(lat)
        x = np.arange(V3)
        r = np.stack([x % L[0], x // L[0] % L[1], x // (L[0] * L[1])])
        for name, moms in _lists(L).items():
            for dof, nt in ((1, 1), (3, 2), (17, 1)):
                f = torch.randn((dof * nt, V3, 2), dtype=dt, device="cuda", generator=g)
                out = torch.full((dof * nt * len(moms), 2), float("nan"), dtype=torch.float64, device="cuda")
                capi.ft_apply(f, capi.F32 if prec == "f32" else capi.F64, dof, nt, moms, -1, out)
                torch.cuda.synchronize()
                n = np.array(moms)
                ph = sum((n[:, i:i + 1] * r[i] % L[i]) / L[i] for i in range(3))
                want = torch.view_as_complex(f.cpu().double()).numpy() @ np.exp(-2j * math.pi * ph).T  # [dof * nt][m]
                got = torch.view_as_complex(out.cpu()).numpy()
                want = want.reshape(dof, nt, -1).transpose(1, 0, 2)
                got = got.reshape(nt, dof, -1)
                err = np.abs(got - want).max() / np.abs(want).max()
                assert err < 1e-12, (name, dof, nt, err)
            # the correlator of a batch on this list
            t, v = G.make_prop(L, 5, 7, 0, 0.5, prec=capi.F32 if prec == "f32" else capi.F64)
            m = capi.MODE_MIXED if prec == "f32" else capi.MODE_F64
            b = capi.Batch(capi.MESONS16, 0, [v], [([0, 0, 0, 0], 2, 0, 0)], moms, m)
            h = torch.zeros((b.info()[0], 2), dtype=torch.float64, device="cuda")
            names = [s for s, _ in b.profile(h)]
            b.close()
            staged = (16 if L[0] % 2 else 8) * L[0] <= (256 if prec == "f32" else 128)
            assert any(s.startswith("project_sep") for s in names) == staged, (name, names)
    finally:
        capi.finalize()
