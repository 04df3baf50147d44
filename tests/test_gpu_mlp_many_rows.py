"""The learned network on more rows than blocks of eight rows serve (above
2 048): blocks of 16 rows whose waves follow the widest layer (1, 4, 8 or 16).

A row's outputs do not depend on the others, so a pass over many rows has the
bits of passes over slices of at most 2 048 (which take the blocks of eight
rows); the gradient is held to the oracle with the device's bf16 rounding points
as in the other tests of the network.  The forward pass of many rows and few
columns keeps to the bandwidth it had as separate products."""
import numpy as np
import pytest

from oracle import mlp as M
from plegma_amd import capi, learned

import gpu_util as G

pytestmark = pytest.mark.gpu

# widths at the edges of 1, 4, 8 and 16 waves, wide inputs of narrow layers, a layer of one column
DIMS = [[17, 11], [32, 16, 1], [33, 16, 3], [5, 17, 64], [65, 33, 2], [17, 65, 11], [40, 192, 7], [193, 20, 4],
        [17, 193, 5]]


@pytest.mark.parametrize("dims", DIMS, ids=lambda d: "-".join(map(str, d)))
def test_many_rows(dims):
    torch = G.torch_cuda()
    B = 4103
    print(f"\n[gpu] mlp dims={dims} B={B}", flush=True)
    rng = np.random.default_rng(6)
    p = learned.init_params(dims, 8) + rng.normal(scale=0.05, size=learned.init_params(dims, 8).shape).astype(np.float32)
    net = capi.Mlp(dims, B)
    net.set_params(p)
    x = rng.normal(size=(B, dims[0])).astype(np.float32)
    t = rng.normal(size=(B, dims[-1])).astype(np.float32)
    xd, td = torch.tensor(x, device="cuda"), torch.tensor(t, device="cuda")
    y = torch.full((B, dims[-1]), float("nan"), device="cuda")
    z = torch.full((B, dims[-1]), float("nan"), device="cuda")
    net.forward(xd, y)
    for r in range(0, B, 1500):
        net.forward(xd[r:r + 1500], z[r:r + 1500])
    torch.cuda.synchronize()
    assert torch.equal(y, z)
    loss, g = net.gradient(xd, td)
    lref, gref = M.loss_grad(p.astype(np.float64), dims, x.astype(np.float64), t.astype(np.float64), emulate=True)
    e = np.linalg.norm(g - gref) / np.linalg.norm(gref)
    print(f"[gpu] grad {e:.1e}", flush=True)
    assert loss == pytest.approx(lref, rel=1e-4) and e < 1e-3
    net.close()


def test_many_rows_of_few_columns_keep_their_rate():
    """1 M rows of 17-11: 112 MB of inputs and outputs, 86 us as separate
    products; within twice that"""
    torch = G.torch_cuda()
    B = 1_000_000
    net = capi.Mlp([17, 11], B)
    net.set_params(learned.init_params([17, 11], 1))
    x = torch.randn((B, 17), device="cuda")
    y = torch.empty((B, 11), device="cuda")
    best = 1e9
    for _ in range(5):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        net.forward(x, y)
        torch.cuda.synchronize()
        a.record()
        for _ in range(10):
            net.forward(x, y, torch.cuda.current_stream().cuda_stream)
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 100)
    print(f"\n[gpu] {best:.1f} us", flush=True)
    assert best < 172
    net.close()
