"""The separable projection's matrix form (k_sep_xy_mm) through plg_ft_apply:
line lengths of one to eight 4-site groups (8-byte and 16-byte loads), plane
heights that leave waves without a line, column counts around its groups of
16, and momentum lists with aliased, L/2 and negative components, without
n = 0 and with one momentum, against the exact-phase DFT in complex128.  The
sums run in FP64 and an FP32 field converts exactly: 1e-12 normwise."""
import math

import numpy as np
import pytest

from plegma_amd import capi

import gpu_util as G

pytestmark = pytest.mark.gpu

LATTICES = [[4, 4, 3], [12, 4, 5], [20, 4, 2], [24, 6, 3], [28, 20, 2], [32, 1, 2], [8, 6, 2], [16, 3, 1], [64, 2, 2]]


def _lists(L):
    full = capi.momlist(4)
    one = [(1, -2, 1)]
    some = [(L[0] // 2, 0, 1), (1, L[1] // 2, 0), (-1, 1, 0), (1 + L[0], -1, 2), (0, 2, -L[2])]
    return {"list": full, "one": one, "some": some}


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("lat", range(len(LATTICES)))
def test_matrix_form(lat, prec):
    torch = G.torch_cuda()
    L = LATTICES[lat] + [2]
    print(f"\n[gpu] plg_init {L} {prec}", flush=True)
    capi.init(L, 0)
    try:
        V3 = L[0] * L[1] * L[2]
        dt = torch.float32 if prec == "f32" else torch.float64
        g = torch.Generator(device="cuda")
        g.manual_seed(lat)
        for name, moms in _lists(L).items():
            for dof, nt in ((1, 1), (3, 2), (17, 1)):
                f = torch.randn((dof * nt, V3, 2), dtype=dt, device="cuda", generator=g)
                out = torch.full((dof * nt * len(moms), 2), float("nan"), dtype=torch.float64, device="cuda")
                capi.ft_apply(f, capi.F32 if prec == "f32" else capi.F64, dof, nt, moms, -1, out)
                torch.cuda.synchronize()
                x = np.arange(V3)
                r = np.stack([x % L[0], x // L[0] % L[1], x // (L[0] * L[1])])
                n = np.array(moms)
                ph = sum((n[:, i:i + 1] * r[i] % L[i]) / L[i] for i in range(3))
                want = torch.view_as_complex(f.cpu().double()).numpy() @ np.exp(-2j * math.pi * ph).T  # [dof * nt][m]
                got = torch.view_as_complex(out.cpu()).numpy()
                want = want.reshape(dof, nt, -1).transpose(1, 0, 2)
                got = got.reshape(nt, dof, -1)
                err = np.abs(got - want).max() / np.abs(want).max()
                assert err < 1e-12, (name, dof, nt, err)
    finally:
        capi.finalize()
