"""Rounding of the FP32 baryon contraction (k_baryon): no larger than that of
the sums written out one after another in single precision.

The direct and the exchange term are sums of 36 and 16 x 36 products; a kernel
that folds one into the other sums larger terms and has to keep its chains
short for it.  The yardstick is such an evaluation in FMAs of single precision
(each product and sum exact in double precision, rounded once): W over (nu,
eps, eps'), the trace as a pairwise sum over the spins, the two terms apart,
each one chain.  Rms over 16 components of 4 slices of 6 x 6 x 4 sites (9 216
values with errors of mean-square fluctuation of order one: the rms is known to
about 1 %), bound 1.1 of the yardstick's."""
import numpy as np
import pytest

import closed_forms as C
from plegma_amd import capi

import gpu_util as G

L, SRC, TOTAL = [6, 6, 4, 4], [0, 0, 0, 0], 4
EPS = [(0, 1, 2, 1), (1, 2, 0, 1), (2, 0, 1, 1), (2, 1, 0, -1), (0, 2, 1, -1), (1, 0, 2, -1)]


def _fma(acc, a, b, sign, dt):
    """acc + sign a b, real and imaginary part as two FMAs each"""
    r = lambda x: x.astype(dt).astype(np.float64)  # noqa: E731
    re, im = acc
    re = r(r(re + sign * a.real * b.real) - sign * a.imag * b.imag)
    im = r(r(im + sign * a.real * b.imag) + sign * a.imag * b.real)
    return re, im


def _chain(pairs, shape, dt):
    acc = np.zeros(shape), np.zeros(shape)
    for a, b, s in pairs:
        acc = _fma(acc, a, b, s, dt)
    return acc[0] + 1j * acc[1]


def _round(x, dt):
    return x.real.astype(dt).astype(np.float64) + 1j * x.imag.astype(dt).astype(np.float64)


def _plain(P, Q, which, dt):
    """the 16 components of the proton (which = 0) or of Delta_which, sums in
    precision dt; P, Q: [mu][nu][a][b][site]"""
    A = C.Cc @ (C.g5 if which == 0 else (C.g1, C.g2, C.g3)[which - 1])
    St = np.einsum("nl,lpabv,pq->nqabv", A, Q, C.bar(A))  # one phase times one entry: exact
    n = P.shape[-1]
    q = [[None] * 3 for _ in range(3)]
    W = [[None] * 3 for _ in range(3)]
    for c in range(3):
        for k in range(3):
            e = [(a, b, ap, bp, s * t) for a, b, c1, s in EPS if c1 == c for bp, ap, k1, t in EPS if k1 == k]
            # the products of M(St, P) of the colours (c, k); P's second colour is a'
            W[c][k] = _chain([(St[m, :, None, b, bp], P[m, None, :, a, ap], s) for m in range(4)
                              for a, b, ap, bp, s in e], (4, 4, n), dt)
            tr = _chain([(St[:, :, b, bp], P[:, :, a, ap], s) for a, b, ap, bp, s in e], (4, 4, n), dt).reshape(16, n)
            while len(tr) > 1:
                tr = _round(tr[0::2] + tr[1::2], dt)
            q[c][k] = tr[0]
    # (the primed colours' order above is (b', a', c'): minus the sign of (a', b', c'))
    D = _chain([(P[:, :, c, k], q[c][k], -1) for c in range(3) for k in range(3)], (4, 4, n), dt)
    X = _chain([(P[:, m, None, c, k], W[c][k][m, None], 1) for m in range(4) for c in range(3) for k in range(3)],
               (4, 4, n), dt)
    return _round(D - X if which == 0 else 2 * D - 4 * X, dt)


def test_yardstick_is_the_contraction():
    """in double precision the yardstick is the spin-open proton (CPU)"""
    rng = np.random.default_rng(1)
    P, Q = (rng.normal(size=(4, 4, 3, 3, 5)) + 1j * rng.normal(size=(4, 4, 3, 3, 5)) for _ in range(2))
    want = C.proton(np.moveaxis(P, -1, 0), np.moveaxis(Q, -1, 0))
    got = np.moveaxis(_plain(P, Q, 0, np.float64), -1, 0)
    assert np.abs(got - want).max() < 1e-12 * np.abs(want).max()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["baryons", "twopt"])
def test_rounding_of_the_mixed_contraction(kind):
    torch = G.torch_cuda()
    V3 = L[0] * L[1] * L[2]
    print(f"\n[gpu] plg_init {L}", flush=True)
    capi.init(L, 0)
    try:
        g = torch.Generator(device="cuda")
        g.manual_seed(8)
        ts = [torch.randn((144, 4 * V3, 2), dtype=torch.float32, device="cuda", generator=g) for _ in range(2)]
        vs = [capi.plg_prop(t.data_ptr(), capi.F32, 0, 4, 0, 4 * V3) for t in ts]
        host = [torch.view_as_complex(t.cpu().double()).numpy().reshape(4, 4, 3, 3, -1) for t in ts]
        mask = capi.G_NUCL | capi.G_DELTAPP_ALL
        for two in ((False, True) if kind == "baryons" else (False,)):
            code = capi.BARYONS if kind == "baryons" else capi.TWOPT
            H = G.run_correlator(code, mask, vs[0], vs[1] if two else vs[0], SRC, TOTAL, 0, mode=capi.MODE_MIXED,
                                 space=capi.POSITION_SPACE)
            ng, nd, nch = capi.kind_shape(code, mask)
            H = H.reshape(ng, nd, 4 * V3, nch)[(1 if kind == "twopt" else 0):, 0]
            for which in range(4):
                P, Q = host[0], host[1] if two and which == 0 else host[0]
                want = _plain(P, Q, which, np.float64)
                plain = _plain(P, Q, which, np.float32)
                got = np.moveaxis(H[which].reshape(4 * V3, 4, 4), 0, -1)
                rms = lambda x: float(np.sqrt((np.abs(x) ** 2).mean()))  # noqa: E731
                e, ref = rms(got - want) / rms(want), rms(plain - want) / rms(want)
                print(f"[gpu] two={two} diquark {which}: {e:.2e}, written out {ref:.2e}", flush=True)
                assert e < 1.1 * ref, (kind, two, which)
    finally:
        capi.finalize()
