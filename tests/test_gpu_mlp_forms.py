"""The forms of a training step leave the same bits: the captured step graph
and the same launches one by one (networks with a layer of 512 columns or
more), and the two launches of narrower networks against a launch per product.

A narrow network set into a wider one by zero weights -- hidden columns that
are zero and stay zero -- takes the other form: its products run over the same
terms in the same order, followed by zeros."""
import numpy as np
import pytest

from plegma_amd import capi, learned

import gpu_util as G

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.tensor(np.ascontiguousarray(a, dtype=np.float32), device="cuda")


def test_wide_training_graph_matches_eager(monkeypatch):
    """as test_training_graph_matches_eager, on a network whose step is
    captured: over several calls, with forward passes, a gradient and
    synchronisations between the replays, and after new inputs"""
    torch = G.torch_cuda()
    rng = np.random.default_rng(31)
    dims = [17, 512, 64, 11]
    x = [_dev(rng.normal(size=(48, 17))) for _ in range(2)]
    t = [_dev(rng.normal(size=(48, 11))) for _ in range(2)]
    params = []
    for eager in ("1", "0"):
        monkeypatch.setenv("PLG_MLP_EAGER", eager)
        net = capi.Mlp(dims, 64)
        net.set_params(learned.init_params(dims, 32))
        y = torch.empty((48, 11), dtype=torch.float32, device="cuda")
        losses = []
        for xi, ti, n in ((x[0], t[0], 40), (x[0], t[0], 25), (x[1], t[1], 30), (x[0], t[0], 5)):
            losses.append(net.train(xi, ti, n, 2e-3))
            net.forward(xi, y)
            torch.cuda.synchronize()
            net.gradient(xi, ti)
        params.append(net.get_params())
        print(f"[gpu] training eager={eager}: losses {losses}", flush=True)
        net.close()
    assert np.array_equal(params[0], params[1])


def _embed(p, dims, wide):
    """parameters of `wide` whose extra hidden columns have zero weights, and
    where those of `dims` lie in them"""
    out, where, off, woff = [], [], 0, 0
    for i, o, wi, wo in zip(dims[:-1], dims[1:], wide[:-1], wide[1:]):
        W, b = np.zeros((wo, wi), np.float32), np.zeros(wo, np.float32)
        W[:o, :i] = p[off:off + o * i].reshape(o, i)
        b[:o] = p[off + o * i:off + o * i + o]
        off += o * i + o
        out += [W.reshape(-1), b]
        k = woff + np.arange(wo * wi).reshape(wo, wi)
        where += [k[:o, :i].reshape(-1), woff + wo * wi + np.arange(o)]
        woff += wo * wi + wo
    return np.concatenate(out), np.concatenate(where)


@pytest.mark.parametrize("dims,wide,B,steps", [([17, 64, 11], [17, 512, 11], 48, 30),
                                               ([17, 100, 100, 11], [17, 512, 100, 11], 361, 20),
                                               ([5, 128, 3], [5, 600, 3], 700, 12)])
def test_two_launch_step_has_the_bits_of_the_products(dims, wide, B, steps):
    torch = G.torch_cuda()
    rng = np.random.default_rng(9)
    x, t = _dev(rng.normal(size=(B, dims[0]))), _dev(rng.normal(size=(B, dims[-1])))
    p = learned.init_params(dims, 5) + rng.normal(scale=0.05, size=learned.init_params(dims, 5).shape).astype(np.float32)
    pw, where = _embed(p, dims, wide)
    assert np.array_equal(pw[where], p)
    got = []
    for d, q in ((dims, p), (wide, pw)):
        net = capi.Mlp(d, B)
        net.set_params(q)
        y = torch.empty((B, dims[-1]), device="cuda")
        net.forward(x, y)
        _, g = net.gradient(x, t)
        loss = net.train(x, t, steps, 1e-3)
        r = net.get_params()
        if d is wide:
            rest = np.ones(len(r), bool)
            rest[where] = False
            assert not r[rest].any() and not g[rest].any()
            g, r = g[where], r[where]
        got.append((y.cpu().numpy(), g, loss, r))
        net.close()
    for a, b, what in zip(got[0], got[1], ("outputs", "gradient", "loss", "parameters")):
        assert np.array_equal(a, b), what
