"""fq_sur_backward only reads the activations of the forward pass: they hold the
same bits afterwards, and two calls with work arrays of their own can share
them on two streams.  Gradients against the float64 oracle on either side of
the batch from which a layer's packed weights find room (16^3: 12 DOFs) and of a
round of 16 DOFs of k_fnt_mix_grad, with one to eight layers, and on 32^3.
Tolerance 1e-4 of the largest gradient per block, as for the other gradients."""
import ctypes as C

import numpy as np
import pytest

from oracle import surrogate as osur
from tests.test_gpu_fno_forward import M, W, _dev_net, _g
from tests.test_gpu_fno_gradient import GRAD_TOL

pytestmark = pytest.mark.gpu


def _check(grad, th, L, N, g, gout):
    want = osur.backward(th, g.astype(np.float64), gout.astype(np.float64), N, W, M, L)
    want = want[-1] if isinstance(want, tuple) else want
    edges = sorted(osur.layout(W, M, L).values()) + [len(th)]
    for a, b in zip(edges[:-1], edges[1:]):
        if b > a:
            assert np.abs(grad[a:b] - want[a:b]).max() <= GRAD_TOL * np.abs(want[a:b]).max() + 1e-30, (a, b)


def _gout(B, N, seed):
    return np.random.default_rng(seed).standard_normal((B, N ** 3)).astype(np.float32) / N ** 3


@pytest.mark.parametrize('kind', ['fp32', 'bf16'])
@pytest.mark.parametrize('N,L,B', [(16, 1, 3), (16, 2, 12), (16, 6, 9), (32, 2, 2)])
def test_activations_are_only_read(backend, N, L, B, kind):
    import torch
    net, th = _dev_net(backend, N, L)
    net.train_acts = kind
    g = torch.tensor(_g(B, N, 21), device='cuda')
    gout = torch.tensor(_gout(B, N, 22), device='cuda')
    print(f'[backward acts N={N} L={L} B={B} {kind}]', flush=True)
    acts = net.forward(g, torch.empty_like(g), training=True)
    before = acts.view(torch.int32).clone()
    net.backward(g, acts, gout, torch.zeros(len(th), dtype=torch.float32, device='cuda'))
    assert torch.equal(acts.view(torch.int32), before)


@pytest.mark.parametrize('N,L,B', [(16, 4, 11), (16, 4, 12), (16, 4, 16), (16, 4, 17), (16, 1, 12), (16, 1, 33),
                                   (16, 8, 12), (32, 6, 2), (32, 2, 1)])
def test_gradient_workspace_edges(backend, N, L, B):
    import torch
    net, th = _dev_net(backend, N, L)
    g, gout = _g(B, N, 23), _gout(B, N, 24)
    gd = torch.tensor(g, device='cuda')
    print(f'[backward workspace N={N} L={L} B={B}]', flush=True)
    acts = net.forward(gd, torch.empty_like(gd), training=True)
    grad = torch.zeros(len(th), dtype=torch.float32, device='cuda')
    net.backward(gd, acts, torch.tensor(gout, device='cuda'), grad)
    _check(grad.cpu().numpy(), th, L, N, g, gout)


def test_two_streams_share_the_activations(backend):
    import torch
    from frfs_amd import _lib
    N, L, B = 16, 3, 12
    net, th = _dev_net(backend, N, L)
    g = _g(B, N, 25)
    gd = torch.tensor(g, device='cuda')
    acts = net.forward(gd, torch.empty_like(gd), training=True)
    work = net._sizes(B, True)[2]
    jobs = []
    for seed in (26, 27):
        gout = _gout(B, N, seed)
        jobs.append((gout, torch.tensor(gout, device='cuda'), torch.zeros(len(th), dtype=torch.float32, device='cuda'),
                     torch.empty(work, dtype=torch.float32, device='cuda'), torch.cuda.Stream()))
    torch.cuda.synchronize()
    print('[backward on two streams]', flush=True)
    for _, god, grad, w, st in jobs:
        _lib.check(_lib.load().fq_sur_backward(C.byref(net.shape), net.theta.data_ptr(), gd.data_ptr(), B, 0,
                                               acts.data_ptr(), god.data_ptr(), grad.data_ptr(), w.data_ptr(),
                                               st.cuda_stream))
    torch.cuda.synchronize()
    for gout, _, grad, _, _ in jobs:
        _check(grad.cpu().numpy(), th, L, N, g, gout)
