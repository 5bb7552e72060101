"""k_out (8^3 and 16^3) loads f ahead of the loss transform for small batches and
where it is used for large ones (more than eight workgroups per CU: 512 DOFs on
16^3, 2048 on 8^3, at 256 CUs): a DOF has the same bits either way, also written
over f, and the first one agrees with the oracle at 1e-5."""
import numpy as np
import pytest

from tests.cases import oracle_vhs, rel_l2, vhs_cfg
from tests.test_gpu_parity import MIXED_TOL
from tests.test_zz_no_alloc import _call, _model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N,most', [(16, 512), (8, 2048)])
def test_same_bits_on_both_sides(backend, N, most):
    from frfs_amd import _lib
    from frfs_amd.inputs import mixture_device, mixture_params, to_aosoa
    from oracle import fastspectral as fsp
    cfg = vhs_cfg(N, 2, 6, 5.0, precision='mixed')
    orc, prm, tab = oracle_vhs(cfg)
    vm, sm = _model(backend, cfg, False)
    f = mixture_device(vm.cv(), mixture_params(most + 8, 17))
    ref = None
    for n in (most + 8, most + 1, most, 5):
        print(f'[k_out N={N}] {n} DOFs', flush=True)
        fin = backend.matrix((1, N ** 3, n))
        to_aosoa(f[:n], fin)
        q = backend.matrix(fin.ioshape)
        _lib.check(_call(sm._h._h, _lib.load().fq_eval, fin, q, n))
        got = q.get()
        _lib.check(_call(sm._h._h, _lib.load().fq_eval, fin, fin, n))
        assert np.array_equal(fin.get(), got)
        if ref is None:
            ref = got
            assert rel_l2(ref[0, :, 0], fsp.vhs_fs(f[0].cpu().numpy(), orc, tab, prm['prefac'])) <= MIXED_TOL
        assert np.array_equal(got, ref[..., :n])
