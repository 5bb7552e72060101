"""The stand-in's inference reads g at any float's address on both grids: g and
out one to three floats past an aligned address give the same bits as aligned."""
import pytest

from tests.test_gpu_fno_forward import _dev_net, _g

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('off', [1, 2, 3])
@pytest.mark.parametrize('N,L,B', [(16, 2, 3), (32, 1, 2), (32, 2, 2), (32, 3, 2)])
def test_any_float_address(backend, N, L, B, off):
    import torch
    net, _ = _dev_net(backend, N, L)
    g = torch.tensor(_g(B, N, 31), device='cuda')
    want = net.predict(g).cpu().numpy()
    gu, ou = (torch.zeros(g.numel() + off, device='cuda')[off:].view(B, -1) for _ in range(2))
    gu.copy_(g)
    print(f'[unaligned g N={N} L={L} off={off}]', flush=True)
    net.forward(gu, ou)
    assert (ou.cpu().numpy() == want).all()
