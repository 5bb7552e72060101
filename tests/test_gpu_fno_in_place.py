"""The stand-in's inference written over its input gives the bits of the output
beside it, with the first and the last layer in one kernel (two layers) and
apart, on both grids."""
import pytest

from tests.test_gpu_fno_forward import _dev_net, _g

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N,L,B', [(16, 1, 3), (16, 2, 70), (16, 3, 5), (32, 2, 3), (32, 3, 2)])
def test_out_over_g(backend, N, L, B):
    import torch
    net, _ = _dev_net(backend, N, L)
    g = torch.tensor(_g(B, N, 41), device='cuda')
    print(f'[fno in place N={N} L={L} B={B}]', flush=True)
    want = net.predict(g).cpu()
    net.predict(g, out=g)
    assert torch.equal(g.cpu(), want)
