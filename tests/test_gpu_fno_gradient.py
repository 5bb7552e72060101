"""The backward kernels on the matrix cores (k_fnt_*, k_fno_mix<true>): every
role of k_fnt_back (first and last layer at once at L = 1, L = 2, a layer
between at L = 3), batches around the tiles of 4, 16 and 64 DOFs, and batches
with and without room for the packed weights, against the float64 oracle.
Tolerance 1e-4 of the largest gradient per block, as for the other gradients."""
import numpy as np
import pytest

from oracle import surrogate as osur
from tests.test_gpu_fno_forward import M, W, _dev_net, _g

pytestmark = pytest.mark.gpu

GRAD_TOL = 1e-4


def _backward(net, th, L, g, gout):
    import torch
    gd, od = torch.tensor(g, device='cuda'), torch.tensor(gout, device='cuda')
    out = torch.empty_like(gd)
    acts = net.forward(gd, out, training=True)
    grads = []
    for _ in range(2):                      # a second pass over the same activations
        grad = torch.zeros(len(th), dtype=torch.float32, device='cuda')
        net.backward(gd, acts, od, grad)
        grads.append(grad.cpu().numpy())
    return out.cpu().numpy(), grads


@pytest.mark.parametrize('N,L,B', [(16, 1, 3), (16, 2, 1), (16, 3, 8), (16, 3, 9), (16, 2, 13), (16, 2, 70),
                                   (32, 1, 1), (32, 3, 2), (32, 2, 5)])
def test_gradient(backend, N, L, B):
    net, th = _dev_net(backend, N, L)
    g = _g(B, N, 8)
    gout = np.random.default_rng(9).standard_normal((B, N ** 3)).astype(np.float32) / N ** 3
    print(f'[fno gradient N={N} L={L} B={B}]', flush=True)
    _, (got, again) = _backward(net, th, L, g, gout)
    want = osur.backward(th, g.astype(np.float64), gout.astype(np.float64), N, W, M, L)
    want = want[-1] if isinstance(want, tuple) else want
    off = osur.layout(W, M, L)
    edges = sorted(off.values()) + [len(th)]
    for grad in (got, again):
        for a, b in zip(edges[:-1], edges[1:]):
            if b > a:
                assert np.abs(grad[a:b] - want[a:b]).max() <= GRAD_TOL * np.abs(want[a:b]).max() + 1e-30, (a, b)
