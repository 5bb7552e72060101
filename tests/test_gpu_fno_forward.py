"""The inference pass on the matrix cores (k_fno_*): both grids, every role of
a plane kernel (first and last layer at once at L = 2, first then last at
L = 3, a layer between at L = 4), and batches around the 16-DOF tiles and
64-DOF workgroups of the mode product, against the float64 oracle.  Tolerance
1e-5 rel-L2 per DOF, as for the other FP32 forwards (sums of at most 512 terms
per stage).  A DOF's output has the same bits in any batch."""
import numpy as np
import pytest

from oracle import surrogate as osur
from tests.cases import rel_l2

pytestmark = pytest.mark.gpu

W, M = 32, 8
FWD_TOL = 1e-5


def _dev_net(backend, N, L, seed=11):
    from frfs_amd.surrogate import FourierSurrogate, init_params
    th = init_params(L, seed)
    off = osur.layout(W, M, L)
    for l in range(L):
        th[off[f'R{l}']:off[f'R{l}'] + 2 * W * W * M ** 3] *= 8.0
    th = th.astype(np.float32).astype(np.float64)
    return FourierSurrogate(backend, layers=L, theta=th, nv=N), th


def _g(B, N, seed):
    """Smooth positive inputs of order one plus 10 % noise."""
    rng = np.random.default_rng(seed)
    x = np.linspace(-4, 4, N)
    base = np.exp(-0.5 * (x[:, None, None] ** 2 + x[None, :, None] ** 2 + x[None, None, :] ** 2)).ravel()
    g = base * rng.uniform(0.5, 1.5, (B, 1)) + 0.1 * rng.standard_normal((B, N ** 3))
    return g.astype(np.float32)


@pytest.mark.parametrize('N,L,B', [(16, 2, 1), (16, 3, 15), (16, 4, 17), (32, 2, 3), (32, 3, 1), (32, 4, 2)])
def test_layers(backend, N, L, B):
    import torch
    net, th = _dev_net(backend, N, L)
    g = _g(B, N, 5)
    print(f'[fno forward N={N} L={L} B={B}]', flush=True)
    out = net.predict(torch.tensor(g, device='cuda')).cpu().numpy()
    want = osur.forward(th, g.astype(np.float64), N, W, M, L)
    assert max(rel_l2(out[b], want[b]) for b in range(B)) <= FWD_TOL


@pytest.mark.parametrize('B', [63, 64, 65, 130])
def test_batch_tiles(backend, B):
    """First, last and tile-edge DOFs against the oracle; the bits of each DOF
    alone and in the batch."""
    import torch
    net, th = _dev_net(backend, 16, 3)
    g = _g(B, 16, 6)
    print(f'[fno batch B={B}]', flush=True)
    out = net.predict(torch.tensor(g, device='cuda')).cpu().numpy()
    pick = sorted({0, 15, 16, 62, B - 1})
    want = osur.forward(th, g[pick].astype(np.float64), 16, W, M, 3)
    for j, b in enumerate(pick):
        assert rel_l2(out[b], want[j]) <= FWD_TOL, b
        one = net.predict(torch.tensor(g[b:b + 1], device='cuda')).cpu().numpy()
        assert np.array_equal(one[0], out[b]), b


def test_special_values(backend):
    """A DOF with a NaN or an infinity does not reach its neighbours."""
    import torch
    net, _ = _dev_net(backend, 16, 4)
    g = _g(18, 16, 7)
    clean = net.predict(torch.tensor(g, device='cuda')).cpu().numpy()
    bad = g.copy()
    bad[3, 100] = np.nan
    bad[16, 7] = np.inf
    out = net.predict(torch.tensor(bad, device='cuda')).cpu().numpy()
    keep = [b for b in range(18) if b not in (3, 16)]
    assert np.array_equal(out[keep], clean[keep])
    assert np.isnan(out[3]).all() and not np.isfinite(out[16]).any()


def test_unaligned_rows(backend):
    """g and out one float past an aligned address: the same bits as aligned."""
    import torch
    net, _ = _dev_net(backend, 16, 3)
    g = torch.tensor(_g(5, 16, 8), device='cuda')
    want = net.predict(g).cpu().numpy()
    n = g.numel()
    gu, ou = (torch.zeros(n + 1, device='cuda')[1:].view(5, -1) for _ in range(2))
    gu.copy_(g)
    print('[fno unaligned]', flush=True)
    net.forward(gu, ou)
    assert np.array_equal(ou.cpu().numpy(), want)
