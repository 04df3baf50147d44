"""The two-launch form of the learned network (widths below 512) at the edges
of its tiles: widths of one column, not a multiple of 16, of more than 16 column
tiles and of the most it takes; batches of less than a row block, with split K
ranges (600, 2 100) and of more blocks than CUs (4 100); and a network just
beyond it.  Forward, loss and gradient against the oracle with the device's
bf16 rounding points (FP64 sums): tolerances as in the gradient test of the
network (rounding ties move single elements by 2^-8), and training steps that
leave finite parameters which lower the loss."""
import numpy as np
import pytest

from oracle import mlp as M
from plegma_amd import capi, learned

import gpu_util as G

pytestmark = pytest.mark.gpu

CASES = [([5, 1], 7), ([3, 17, 2], 33), ([40, 511, 33, 256], 600), ([17, 256, 256, 11], 2100),
         ([17, 48, 48, 48, 11], 4100), ([24, 512, 40], 96)]


@pytest.mark.parametrize("dims,B", CASES)
def test_rows_form_matches_oracle(dims, B):
    torch = G.torch_cuda()
    print(f"\n[gpu] mlp dims={dims} B={B}", flush=True)
    rng = np.random.default_rng(3)
    dev = lambda a: torch.tensor(np.ascontiguousarray(a, dtype=np.float32), device="cuda")  # noqa: E731
    net = capi.Mlp(dims, B + 5)
    p = learned.init_params(dims, 17)
    p += rng.normal(scale=0.05, size=p.shape).astype(np.float32)   # biases too
    net.set_params(p)
    for n in (B, max(1, B // 3)):   # a smaller call after a larger one: no stale rows
        x = rng.normal(size=(n, dims[0])).astype(np.float32)
        t = rng.normal(size=(n, dims[-1])).astype(np.float32)
        xd, td = dev(x), dev(t)
        y = torch.full((n, dims[-1]), float("nan"), dtype=torch.float32, device="cuda")
        net.forward(xd, y)
        ref, _ = M.forward(p.astype(np.float64), dims, x.astype(np.float64), emulate=True)
        err = np.abs(y.cpu().numpy() - ref).max(axis=1) / np.abs(ref).max()
        assert np.sum(err > 1e-5) <= max(1, n // 32) and err.max() < 1e-2
        loss, g = net.gradient(xd, td)
        lref, gref = M.loss_grad(p.astype(np.float64), dims, x.astype(np.float64), t.astype(np.float64), emulate=True)
        e = np.linalg.norm(g - gref) / np.linalg.norm(gref)
        print(f"[gpu] n={n} forward {err.max():.1e} grad {e:.1e}", flush=True)
        assert loss == pytest.approx(lref, rel=1e-4) and e < 1e-3
    l1 = net.train(xd, td, 30, 1e-3)
    assert np.isfinite(net.get_params()).all() and l1 < loss
    net.close()


def test_forward_in_place_of_its_input():
    """outputs over the inputs' own memory: every input is read first"""
    torch = G.torch_cuda()
    net = capi.Mlp([12, 64, 12], 512)
    net.set_params(learned.init_params([12, 64, 12], 2))
    x = torch.randn((512, 12), device="cuda")
    y = torch.empty_like(x)
    net.forward(x, y)
    net.forward(x, x)
    torch.cuda.synchronize()
    assert torch.equal(x, y)
    net.close()
