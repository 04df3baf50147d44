"""Performance cases of the two-point correlator library.

Every case is work that a measurement program of lattice QCD gives the
library through its public entry points (plegma_amd.capi): single correlator
calls as the drop-in classes make them, a batch of sources, the standalone
Fourier projection, the table-driven baryons and tetraquarks, the propagator
cast of the mixed path and the training of the learned estimator.

Inputs are point-to-all propagators with N(0,1) entries that decay as
exp(-lambda |t - t0|) from the source, held over the source's time window.
FP64 propagators feed the FP64 path.  FP32 propagators carry one power-of-two
exponent per time slice, as a cast propagator does, and feed the mixed path,
whose correlators are kept in single precision (the H_elem of a
PLEGMA_Correlator<float>).

exact() restates the correlators in complex128 with plain torch.
"""
import math

import numpy as np
import torch

from plegma_amd import capi

DEV = "cuda"
LIGHT, HEAVY, STRANGE, CHARM = 0.5, 1.2, 0.6, 0.9   # decay rates of the flavours
KINDS = {"mesons": capi.MESONS, "mesons16": capi.MESONS16, "mesons_new": capi.MESONS_NEW,
         "mesons_all": capi.MESONS_ALL, "baryons": capi.BARYONS, "mesmes": capi.MESON_MESON,
         "twopt": capi.TWOPT}
MASKS = {"nucl": capi.G_NUCL, "delta": capi.G_DELTAPP_ALL, "all": capi.G_NUCL | capi.G_DELTAPP_ALL}


# ------------------------------------------------------------------ the cases
def _lat(lx, ly, lz, lt):
    return {"lx": lx, "ly": ly, "lz": lz, "lt": lt}


def _src(sx, sy, sz, st, window):
    return {"sx": sx, "sy": sy, "sz": sz, "st": st, "window": window}


def _corr(kind, mode, lat, src, q2, mask="all", two=False, rot=0, bc=0, space="mom"):
    return {"what": "corr", "kind": kind, "mode": mode, **lat, **src, "q2": q2, "mask": mask, "two": two,
            "rot": rot, "bc": bc, "space": space}


def listed():
    cases = {
        # smallest call: a test ensemble's 16 mesons + proton in FP64; latency and launches
        "twopt_f64_8x16": _corr("twopt", "f64", _lat(8, 8, 8, 16), _src(0, 0, 0, 0, 16), 4, mask="nucl"),
        # contractMesons on two flavours in FP64, an ordinary lattice and its full time extent
        "mesons_f64_24x48": _corr("mesons", "f64", _lat(24, 24, 24, 48), _src(3, 17, 8, 5, 48), 9, two=True),
        # contractBaryons on two flavours in FP64, twisted-mass preparation fused, a window that wraps in time
        "baryons_f64_24x48": _corr("baryons", "f64", _lat(24, 24, 24, 48), _src(7, 0, 21, 40, 20), 9, two=True,
                                   rot=1, bc=40),
        # contractMesonsAll (34 channels) on a ragged lattice
        "mesons_all_f64_ragged": _corr("mesons_all", "f64", _lat(24, 20, 28, 40), _src(11, 3, 19, 30, 25), 9,
                                       two=True),
        # one source of a production lattice in the mixed path: mesons + proton + Delta, 257 momenta
        "twopt_mixed_32x64": _corr("twopt", "mixed", _lat(32, 32, 32, 64), _src(5, 30, 12, 50, 48), 16),
        # many sources of a configuration in one batched plan
        "batch_mixed_32x64": {"what": "batch", "mode": "mixed", **_lat(32, 32, 32, 64), "sources": 16, "wmin": 8,
                              "wmax": 32, "q2": 16, "mask": "all", "layout": 20261202},
        # the largest lattice: light-heavy mesons and meson-meson channels, 32 of the 128 slices
        "mesmes_mixed_64x128": _corr("mesmes", "mixed", _lat(64, 64, 64, 128), _src(0, 0, 0, 16, 32), 9, two=True),
        # contractBaryonsUDSC: all 20 flavour products (200 operators)
        "udsc_mixed_24x48": {"what": "udsc", "mode": "mixed", **_lat(24, 24, 24, 48), **_src(1, 2, 3, 10, 16),
                             "q2": 9},
        # contractTetraquarks: the heavy-light "udbb" product (16 operators)
        "tetra_mixed_16x32": {"what": "tetra", "family": "heavy-light", "mode": "mixed", **_lat(16, 16, 16, 32),
                              **_src(4, 9, 0, 20, 24), "q2": 4},
        # PLEGMA_FT::apply of a 16-component field
        "ft_f32_32x64": {"what": "ft", "mode": "f32", **_lat(32, 32, 32, 64), "dof": 16, "nt": 64, "q2": 16,
                         "sign": -1},
        # 100 Adam steps of the learned estimator (one chunk of a fit): forward, backward and update
        "mlp_train_2048": {"what": "mlp_train", "batch": 2048, "steps": 100, "hidden": 256},
        # the FP64 -> FP32 cast of a source's propagator that precedes the mixed path
        "cast_32x64": {"what": "cast", **_lat(32, 32, 32, 64), **_src(0, 0, 0, 24, 24)},
    }
    return [{"name": n, **c} for n, c in cases.items()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_lat(rng, tmax=64):
    if rng.random() < 0.65:   # cubic, any extent
        n = _log_int(rng, 4, 32)
        lx = ly = lz = n
    else:                     # unequal extents
        lx, ly, lz = (rng.choice([4, 6, 8, 10, 12, 16, 20, 24, 32]) for _ in range(3))
    return _lat(lx, ly, lz, _log_int(rng, 6, tmax))


def _draw_src(rng, lat, sites):
    v3 = lat["lx"] * lat["ly"] * lat["lz"]
    wmax = max(1, min(lat["lt"], sites // v3))
    return _src(rng.randrange(lat["lx"]), rng.randrange(lat["ly"]), rng.randrange(lat["lz"]),
                rng.randrange(lat["lt"]), _log_int(rng, min(4, wmax), wmax))


def draw(rng):
    what = rng.choices(["corr", "batch", "udsc", "tetra", "ft", "mlp_train", "mlp_forward", "cast"],
                       [10, 2, 2, 2, 2, 1, 1, 1])[0]
    lat = _draw_lat(rng)
    q2 = rng.choice([0, 1, 2, 4, 4, 9, 9, 16])
    mode = rng.choice(["f64", "mixed"])
    if what == "corr":
        kind = rng.choice(["mesons", "mesons16", "mesons_new", "mesons_all", "baryons", "baryons", "mesmes",
                           "twopt", "twopt", "twopt"])
        two = kind != "twopt" and rng.random() < 0.7
        src = _draw_src(rng, lat, 800_000)
        pos = lat["lx"] * lat["ly"] * lat["lz"] * src["window"] < 100_000 and rng.random() < 0.2
        prep = rng.random() < 0.25
        return _corr(kind, mode, lat, src, q2, mask=rng.choice(["nucl", "delta", "all", "all"]), two=two,
                     rot=rng.choice([1, -1]) if prep else 0, bc=src["st"] if prep else 0,
                     space="pos" if pos else "mom")
    if what == "batch":
        lat = _draw_lat(rng, 48)
        wmax = max(2, min(lat["lt"], 600_000 // (lat["lx"] * lat["ly"] * lat["lz"]), 24))
        return {"what": "batch", "mode": mode, **lat, "sources": rng.randrange(2, 9), "wmin": 1, "wmax": wmax,
                "q2": max(1, q2), "mask": rng.choice(["nucl", "all"]), "layout": rng.randrange(1 << 30)}
    if what == "udsc":
        return {"what": "udsc", "mode": mode, **lat, **_draw_src(rng, lat, 100_000), "q2": min(q2, 9)}
    if what == "tetra":
        return {"what": "tetra", "family": rng.choice(["heavy-light", "bcud"]), "mode": mode, **lat,
                **_draw_src(rng, lat, 30_000), "q2": min(q2, 9)}
    if what == "ft":
        return {"what": "ft", "mode": rng.choice(["f32", "f64"]), **lat, "dof": rng.choice([1, 3, 4, 12, 16]),
                "nt": rng.choice([1, lat["lt"]]), "q2": q2, "sign": rng.choice([1, -1])}
    if what == "mlp_train":
        return {"what": "mlp_train", "batch": _log_int(rng, 64, 4096), "steps": rng.randrange(4, 60),
                "hidden": rng.choice([64, 100, 128, 256])}
    if what == "mlp_forward":
        return {"what": "mlp_forward", "batch": _log_int(rng, 16, 4096), "hidden": rng.choice([64, 100, 256])}
    return {"what": "cast", **lat, **_draw_src(rng, lat, 800_000)}


# ------------------------------------------------------------------ inputs
def _gen(seed, k):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1009 + k)
    return g


def _dims(case):
    return [case["lx"], case["ly"], case["lz"], case["lt"]]


def _source(case):
    return [case["sx"], case["sy"], case["sz"], case["st"]]


_lattice = None


def _use_lattice(L):
    """plg_init of the case's lattice, once per lattice as a program does"""
    global _lattice
    if _lattice != L:
        capi.init(L, 0)
        _lattice = list(L)


def _propagator(seed, k, v3, t0, nt, lam, f64, T):
    """(tensor [144][nt v3][2], exponents or None): the propagator at the times
    t0 .. t0 + nt - 1 (mod T).  FP32 entries are stored times 2^-e(t)."""
    t = torch.empty((144, nt, v3, 2), dtype=torch.float64 if f64 else torch.float32, device=DEV)
    t.normal_(generator=_gen(seed, k))
    dist = torch.tensor([abs((t0 + i) % T - t0) for i in range(nt)], dtype=torch.float64, device=DEV)
    e = None
    if f64:
        t.mul_(torch.exp(-lam * dist).view(1, nt, 1, 1))
    else:
        e = torch.round(-lam * dist / math.log(2.0)).to(torch.int32)
        t.mul_(torch.exp(-lam * dist - e.double() * math.log(2.0)).float().view(1, nt, 1, 1))
    return t.view(144, nt * v3, 2), e


def _view(prop, f64, t0, nt, v3, rot=0, bc=0):
    t, e = prop
    v = capi.plg_prop(t.data_ptr(), capi.F64 if f64 else capi.F32, t0, nt, 0, nt * v3,
                      None if e is None else e.data_ptr())
    v.rotate_sign, v.bc_t0 = rot, bc
    return v


def _flavours(case):
    """decay rates of the propagators a case reads"""
    if case["what"] == "udsc":
        return [LIGHT, LIGHT, STRANGE, CHARM]
    if case["what"] == "tetra":
        return [LIGHT, HEAVY] if case["family"] == "heavy-light" else [LIGHT, CHARM, HEAVY]
    if case["what"] == "cast":
        return [LIGHT]
    return [LIGHT, HEAVY if case["kind"] == "mesmes" else STRANGE] if case["two"] else [LIGHT]


def _props(case, seed):
    """the case's propagators over its window"""
    L = _dims(case)
    v3 = L[0] * L[1] * L[2]
    f64 = case["what"] == "cast" or case["mode"] == "f64"
    return [_propagator(seed, k, v3, case["st"], case["window"], lam, f64, L[3])
            for k, lam in enumerate(_flavours(case))]


def _batch_jobs(case):
    """[(source, window)] of a batch, fixed by the case"""
    rng = np.random.default_rng(case["layout"])
    L = _dims(case)
    return [([int(rng.integers(0, n)) for n in L], int(rng.integers(case["wmin"], case["wmax"] + 1)))
            for _ in range(case["sources"])]


def _net(case):
    return [17, case["hidden"], case["hidden"], 11]


def _params(case, seed):
    """He-normal weights and zero biases, FP32, in the library's layout"""
    rng = np.random.default_rng(seed)
    parts = []
    for i, o in zip(_net(case)[:-1], _net(case)[1:]):
        parts += [rng.normal(0.0, np.sqrt(2.0 / i), size=o * i), np.zeros(o)]
    return np.concatenate(parts).astype(np.float32)


def _samples(case, seed):
    """standardised inputs, and targets that depend on them smoothly"""
    x = torch.empty((case["batch"], 17), device=DEV).normal_(generator=_gen(seed, 0))
    m = torch.empty((17, 11), device=DEV).normal_(generator=_gen(seed, 1))
    n = torch.empty((case["batch"], 11), device=DEV).normal_(generator=_gen(seed, 2))
    return x, (torch.tanh(x.double() @ m.double() / 4) + 0.05 * n.double()).float()


def prepare(case, seed):
    what = case["what"]
    s = {"case": case}
    if what in ("mlp_train", "mlp_forward"):
        s["net"] = capi.Mlp(_net(case), case["batch"])
        s["net"].set_params(_params(case, seed))
        s["x"], s["t"] = _samples(case, seed)
        s["y"] = torch.empty((case["batch"], 11), device=DEV)
        return s
    L = _dims(case)
    v3 = L[0] * L[1] * L[2]
    _use_lattice(L)
    if what == "cast":
        (src, _), = _props(case, seed)
        nt = case["window"]
        s["keep"] = src
        s["dst"] = torch.empty(src.shape, dtype=torch.float32, device=DEV)
        s["exp"] = torch.empty(nt, dtype=torch.int32, device=DEV)
        s["from"] = _view((src, None), True, case["st"], nt, v3)
        s["to"] = _view((s["dst"], s["exp"]), False, case["st"], nt, v3)
        return s
    s["moms"] = capi.momlist(case["q2"])
    if what == "ft":
        f64 = case["mode"] == "f64"
        s["field"] = torch.empty((case["dof"], case["nt"] * v3, 2), dtype=torch.float64 if f64 else torch.float32,
                                 device=DEV).normal_(generator=_gen(seed, 0))
        s["moms"] = np.array(s["moms"], dtype=np.int32).reshape(-1, 3)
        s["out"] = torch.empty((case["nt"] * case["dof"] * len(s["moms"]), 2), dtype=torch.float64, device=DEV)
        return s
    f64 = case["mode"] == "f64"
    if what == "batch":
        kind, mask = capi.TWOPT, MASKS[case["mask"]]
        s["keep"], views, jobs, off = [], [], [], 0
        for k, (src, w) in enumerate(_batch_jobs(case)):
            p = _propagator(seed, k, v3, src[3], w, LIGHT, f64, L[3])
            s["keep"].append(p)
            views.append(_view(p, f64, src[3], w, v3))
            jobs.append((src, w, k, off))
            off += capi.correlator_size(kind, mask, src, w, len(s["moms"]))
        s["batch"] = capi.Batch(kind, mask, views, jobs, s["moms"], capi.MODE_F64 if f64 else capi.MODE_MIXED,
                                flags=capi.BATCH_GRAPH | capi.BATCH_TUNE)
        s["out"] = torch.empty((off, 2), dtype=torch.float64, device=DEV)
        return s
    s["keep"] = _props(case, seed)
    s["views"] = [_view(p, f64, case["st"], case["window"], v3, case.get("rot", 0), case.get("bc", 0))
                  for p in s["keep"]]
    v, src, w, nm = s["views"], _source(case), case["window"], len(s["moms"])
    if what == "corr":
        space = capi.POSITION_SPACE if case["space"] == "pos" else capi.MOMENTUM_SPACE
        n = capi.correlator_size(KINDS[case["kind"]], MASKS[case["mask"]], src, w, nm, space)
    elif what == "udsc":
        n = capi.baryons_udsc_size(v[0], v[1], v[2], v[3], src, w, nm)
    else:
        n = capi.tetraquarks_size(*_tetra_views(s), src, w, nm, family=case["family"])
    s["out"] = torch.empty((n, 2), dtype=torch.float64 if f64 else torch.float32, device=DEV)
    return s


def _tetra_views(s):
    """(lt, st, ch, bt)"""
    v = s["views"]
    return (v[0], None, None, v[1]) if s["case"]["family"] == "heavy-light" else (v[0], None, v[1], v[2])


# ------------------------------------------------------------------ one pass
def run(s):
    case = s["case"]
    what = case["what"]
    if what == "mlp_train":
        loss = s["net"].train(s["x"], s["t"], case["steps"], 1e-3)
        return {"loss": np.float32(loss), "params": s["net"].get_params()}
    if what == "mlp_forward":
        s["net"].forward(s["x"], s["y"])
        return s["y"]
    if what == "cast":
        capi.cast_prop(s["to"], s["from"])
        return {"prop": s["dst"], "exp": s["exp"]}
    if what == "ft":
        f64 = case["mode"] == "f64"
        capi.ft_apply(s["field"], capi.F64 if f64 else capi.F32, case["dof"], case["nt"], s["moms"], case["sign"],
                      s["out"])
        return s["out"]
    f64 = case["mode"] == "f64"
    if what == "batch":
        s["batch"].run(s["out"])
        return s["out"] if f64 else s["out"].float()
    mode, prec = (capi.MODE_F64, capi.F64) if f64 else (capi.MODE_MIXED, capi.F32)
    v, src, w = s["views"], _source(case), case["window"]
    if what == "corr":
        space = capi.POSITION_SPACE if case["space"] == "pos" else capi.MOMENTUM_SPACE
        capi.correlator(KINDS[case["kind"]], MASKS[case["mask"]], v[0], v[-1], src, w, s["moms"], mode, space, prec,
                        s["out"])
    elif what == "udsc":
        capi.baryons_udsc(v[0], v[1], v[2], v[3], src, w, s["moms"], mode, capi.MOMENTUM_SPACE, prec, s["out"])
    else:
        capi.tetraquarks(*_tetra_views(s), src, w, s["moms"], mode, capi.MOMENTUM_SPACE, prec, s["out"],
                         family=case["family"])
    return s["out"]


# ------------------------------------------------------------------ necessary work
def _nmom(q2):
    r = math.isqrt(q2)
    return sum(1 for x in range(-r, r + 1) for y in range(-r, r + 1) for z in range(-r, r + 1)
               if x * x + y * y + z * z <= q2)


def _channels(case):
    """(channels written per site and momentum, complex multiply-adds per site)"""
    kind = case.get("kind", "twopt")
    ng = {"nucl": 1, "delta": 3, "all": 4}[case["mask"]]
    block = 16 * (4 * 36 + 36)   # a diquark block: exchange and closing products
    if kind in ("mesons", "mesons16"):
        nch = 10 if kind == "mesons" else 16
        return 2 * nch, (2 if case["two"] else 1) * 9 * 40
    if kind == "mesons_new":
        return 10, 9 * 64
    if kind == "mesons_all":
        return 34, 9 * 144
    if kind == "mesmes":
        return 20, 9 * 64 + 2 * 16 * (4 * 27 + 18)
    if kind == "baryons":
        return 32 * ng, (2 if case["two"] else 1) * ng * block
    return 16 + 16 * ng, 9 * 64 + ng * block


def work(case):
    what = case["what"]
    if what in ("mlp_train", "mlp_forward"):
        d = _net(case)
        w = sum(i * o for i, o in zip(d[:-1], d[1:]))
        rows = case["batch"]
        if what == "mlp_forward":
            return {"bytes": 4 * rows * (17 + 11) + 4 * w, "flops": 2 * rows * w}
        # a step: forward, both products of the backward, parameters and Adam moments read and written
        return {"bytes": case["steps"] * (4 * rows * (17 + 11) + 28 * w), "flops": case["steps"] * 6 * rows * w}
    v3 = case["lx"] * case["ly"] * case["lz"]
    if what == "cast":
        n = 144 * v3 * case["window"]
        return {"bytes": n * (16 + 8), "flops": 2 * n}
    nm = _nmom(case["q2"])
    # separable sums over x: both phases of about sqrt(q2) + 1 classes per site and column
    dft = 4 * 2 * (math.isqrt(case["q2"]) + 1)
    if what == "ft":
        cols = case["dof"] * case["nt"]
        return {"bytes": cols * (v3 * (16 if case["mode"] == "f64" else 8) + nm * 16), "flops": cols * v3 * dft}
    elem = 16 if case["mode"] == "f64" else 8
    if what == "batch":
        rows = sum(w for _, w in _batch_jobs(case))
        nch, cmac = _channels(case)
        return {"bytes": rows * (144 * v3 * elem + nch * nm * elem), "flops": rows * v3 * (8 * cmac + nch * dft)}
    rows = case["window"]
    nprop = len(_flavours(case))
    if what == "udsc":      # per product: the colour diquarks, distinct terms and entries of its table
        nch, cmac = 200, 293_000
    elif what == "tetra":
        nch, cmac = (16, 82_000) if case["family"] == "heavy-light" else (57, 380_000)
    else:
        nch, cmac = _channels(case)
    out = nch * (v3 if case.get("space") == "pos" else nm)
    flops = v3 * (8 * cmac + (0 if case.get("space") == "pos" else nch * dft))
    return {"bytes": rows * (nprop * 144 * v3 * elem + out * elem), "flops": rows * flops}


# ------------------------------------------------------------------ exact values
_C = torch.complex128


def _gammas():
    g1 = np.array([[0, 0, 0, 1j], [0, 0, 1j, 0], [0, -1j, 0, 0], [-1j, 0, 0, 0]])
    g2 = np.array([[0, 0, 0, 1], [0, 0, -1, 0], [0, -1, 0, 0], [1, 0, 0, 0]], dtype=complex)
    g3 = np.array([[0, 0, 1j, 0], [0, 0, 0, -1j], [-1j, 0, 0, 0], [0, 1j, 0, 0]])
    g4 = np.diag([1, 1, -1, -1]).astype(complex)
    g5 = g1 @ g2 @ g3 @ g4
    sig = lambda a, b: -0.5j * (a @ b - b @ a)  # noqa: E731
    return [np.eye(4, dtype=complex), g1, g2, g3, g4, g5, g5 @ g1, g5 @ g2, g5 @ g3, g5 @ g4, sig(g1, g2),
            sig(g1, g3), sig(g2, g3), sig(g4, g1), sig(g4, g2), sig(g4, g3)]


GAM = _gammas()
MESON10 = [5, 0, 6, 7, 8, 9, 1, 2, 3, 4]
EPS = [(0, 1, 2, 1), (1, 2, 0, 1), (2, 0, 1, 1), (2, 1, 0, -1), (0, 2, 1, -1), (1, 0, 2, -1)]


def _trace_pair(S1, S2, A, B, dots):
    """sum over colours of Tr_spin[A S1 B S2^dag] for signed permutations A, B"""
    out = 0
    for d in range(4):
        for a in range(4):
            for b in range(4):
                for z in range(4):
                    w = A[d, a] * B[b, z]
                    if w == 0:
                        continue
                    key = (a, b, d, z)
                    if key not in dots:
                        dots[key] = (S1[a, b] * S2[d, z].conj()).sum((0, 1))
                    out = out + complex(w) * dots[key]
    return out


def _meson_channels(S1, S2, ops):
    """Tr[G S1 g5 G S2^dag g5] per operator"""
    dots, g5 = {}, GAM[5]
    return [_trace_pair(S1, S2, g5 @ GAM[op], g5 @ GAM[op], dots) for op in ops]


def _baryon_channels(P, Q, which):
    """the 16 spin components of the proton (which = 0) or of the Delta with
    diquark C gamma_which"""
    A = 1j * GAM[2] @ GAM[4] @ (GAM[5] if which == 0 else GAM[which])
    Ab = GAM[4] @ A.conj().T @ GAM[4]
    t = lambda m: torch.tensor(m, dtype=_C, device=DEV)  # noqa: E731
    st = torch.einsum("nl,lpabv,pq->nqabv", t(A), Q, t(Ab))
    D = torch.zeros((4, 4, P.shape[-1]), dtype=_C, device=DEV)
    X = torch.zeros_like(D)
    q = [[0] * 3 for _ in range(3)]
    W = [[0] * 3 for _ in range(3)]
    for a, b, c, s in EPS:
        for ap, bp, cp, sp in EPS:
            q[c][cp] = q[c][cp] + (s * sp) * (P[:, :, a, ap] * st[:, :, b, bp]).sum((0, 1))
            for n in range(4):   # W[c][a'][nu'][mu'] = sum_nu st[nu][nu'] P[nu][mu']
                W[c][ap] = W[c][ap] + (s * sp) * st[n, :, None, b, bp] * P[n, None, :, a, cp]
    for c in range(3):
        for k in range(3):
            D += q[c][k] * P[:, :, c, k]
            for n in range(4):
                X += P[:, n, None, c, k] * W[c][k][n, None]
    r = D - X if which == 0 else 2 * D - 4 * X
    return [r[m, n] for m in range(4) for n in range(4)]


def _mesmes_channels(S1, S2):
    m12 = lambda S: S.permute(4, 0, 2, 1, 3).reshape(-1, 12, 12)  # noqa: E731
    L12, H12 = m12(S1), m12(S2).conj().transpose(1, 2)
    out = _meson_channels(S1, S2, range(16))
    for op in (5, 1, 2, 3):
        X = torch.tensor(np.kron(GAM[5] @ GAM[op], np.eye(3)), dtype=_C, device=DEV)
        # Tr[A A] of A = G S_L X S_H^dag g5, by the cyclic trace of M = S_L X S_H^dag X
        M = torch.matmul(L12 @ X, (H12 @ X).contiguous())
        tr = M.diagonal(dim1=1, dim2=2).sum(-1)
        out.append(tr * tr - (M * M.transpose(1, 2)).sum((1, 2)))
    return out


def _groups(case, S):
    """computed channels of a time slice as [group][dataset][channel][site]"""
    kind = case.get("kind", "twopt")
    which = {"nucl": [0], "delta": [1, 2, 3], "all": [0, 1, 2, 3]}[case["mask"]]
    S1, S2 = S[0], S[-1]
    if kind in ("mesons", "mesons16"):
        ops = MESON10 if kind == "mesons" else range(16)
        return [[_meson_channels(S1, S1, ops), _meson_channels(S2, S2, ops)]]
    if kind == "mesons_new":
        return [[_meson_channels(S1, S2, MESON10)]]
    if kind == "mesons_all":
        dots, g5 = {}, GAM[5]
        ch = _meson_channels(S1, S2, (5, 0))
        for p in (0, 5):
            ch += [_trace_pair(S1, S2, GAM[1 + i + p], GAM[1 + j + p], dots) for i in range(4) for j in range(4)]
        return [[ch]]
    if kind == "mesmes":
        return [[_mesmes_channels(S1, S2)]]
    if kind == "baryons":
        return [[_baryon_channels(S1, S2 if w == 0 else S1, w), _baryon_channels(S2, S1 if w == 0 else S2, w)]
                for w in which]
    return [[_meson_channels(S1, S1, range(16))]] + [[_baryon_channels(S1, S1, w)] for w in which]


def _momenta(q2):
    """momentum triples in the library's order"""
    return [(x, y, z) for q in range(q2 + 1) for x in range(q, -q - 1, -1) for y in range(q, -q - 1, -1)
            for z in range(q, -q - 1, -1) if x * x + y * y + z * z == q]


def _dft(c, L, moms, sign, src=(0, 0, 0)):
    """sum_x c[n][x] exp(sign i 2 pi k.(x - src) / L): [n][momentum]"""
    c = c.reshape(-1, L[2], L[1], L[0])
    n = np.array(moms).reshape(-1, 3)
    idx, mats = [], []
    for d in range(3):
        u, inv = np.unique(n[:, d], return_inverse=True)
        ph = (u[:, None] * (np.arange(L[d])[None, :] - src[d])) % L[d]
        mats.append(torch.tensor(np.exp(sign * 2j * np.pi * ph / L[d]), dtype=_C, device=DEV))
        idx.append(torch.tensor(inv.reshape(-1), device=DEV))
    g = c @ mats[0].t()                       # [n][z][y][kx]
    g = torch.matmul(mats[1], g)              # [n][z][ky][kx]
    g = torch.matmul(mats[2], g.flatten(2)).view(c.shape[0], mats[2].shape[0], mats[1].shape[0], -1)
    return g[:, idx[2], idx[1], idx[0]]


def _slice(case, prop, plane, t, v3):
    """one time slice of a propagator in complex128, prepared, as S[mu][nu][a][b][site]"""
    data, e = prop
    S = torch.view_as_complex(data.view(144, -1, v3, 2)[:, plane].double().contiguous())
    if e is not None:
        S = S * 2.0 ** float(e[plane])
    S = S.view(4, 4, 3, 3, v3)
    if case.get("rot"):   # S -> U S U with U = (1 + i s g5) / sqrt 2
        U = torch.tensor((np.eye(4) + 1j * case["rot"] * GAM[5]) / np.sqrt(2), dtype=_C, device=DEV)
        S = torch.einsum("mk,klabv,ln->mnabv", U, S, U)
    return -S if t < case.get("bc", 0) else S


def _times(L, src, window):
    """lattice times of a correlator's rows: the wrapped slices first"""
    T, t0 = L[3], src[3]
    start = (T - t0) % T
    start = 0 if start >= window else start
    wrapped = min(window, T + start) - start if start > 0 else 0
    return [j if j < wrapped else t0 + j - wrapped for j in range(wrapped + min(window, T - t0))]


def _correlator(case, props, src, window):
    """complex128 correlator in the H_elem order [g][d][row][momentum or site][channel]"""
    L = _dims(case)
    v3 = L[0] * L[1] * L[2]
    moms = _momenta(case["q2"])
    rows = []
    for t in _times(L, src, window):
        S = [_slice(case, p, (t - src[3]) % L[3], t, v3) for p in props]
        per = []
        for g in _groups(case, S):
            for ch in g:
                c = torch.stack(ch)
                per.append((c if case.get("space") == "pos" else _dft(c, L, moms, -1, src)).t())
        rows.append(torch.stack(per))                   # [g d][momentum][channel]
    return torch.stack(rows, 1).reshape(-1)


def exact(case, seed):
    what = case["what"]
    if what == "mlp_forward":
        p, off = torch.tensor(_params(case, seed), device=DEV).double(), 0
        y, d = _samples(case, seed)[0].double(), _net(case)
        for k, (i, o) in enumerate(zip(d[:-1], d[1:])):
            y = y @ p[off:off + i * o].view(o, i).t() + p[off + i * o:off + i * o + o]
            off += i * o + o
            y = torch.nn.functional.silu(y) if k < len(d) - 2 else y
        return y
    if what == "cast":
        (src, _), = _props(case, seed)
        m = src.view(144, case["window"], -1).abs().amax((0, 2))
        e = torch.frexp(m)[1] - 1
        return {"prop": (src.view(144, case["window"], -1) * torch.exp2(-e.double()).view(1, -1, 1)).view(src.shape),
                "exp": e.to(torch.int32)}
    if what == "ft":
        L = _dims(case)
        field = prepare(case, seed)["field"].double().view(case["dof"], case["nt"], -1, 2)
        rows = [_dft(torch.view_as_complex(field[:, t].contiguous()), L, _momenta(case["q2"]), case["sign"])
                for t in range(case["nt"])]
        return torch.view_as_real(torch.stack(rows).reshape(-1))
    if what == "batch":
        L = _dims(case)
        v3 = L[0] * L[1] * L[2]
        out = [_correlator(case, [_propagator(seed, k, v3, src[3], w, LIGHT, case["mode"] == "f64", L[3])], src, w)
               for k, (src, w) in enumerate(_batch_jobs(case))]
        return torch.view_as_real(torch.cat(out))
    if what == "corr":
        return torch.view_as_real(_correlator(case, _props(case, seed), _source(case), case["window"]))
    # a training run is a chain of bf16 roundings, and the udsc and tetraquark
    # operators are thousands of table terms per site: no short 64-bit form
    return None
