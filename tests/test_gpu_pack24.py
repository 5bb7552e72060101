"""The FP64 product kernel of the 24^3 grid (k_pack) in each of its forms: the
real part of a group sum (VHS), single-product groups (VSS) and the twin sums of
the bilinear model, against the oracle, and the same bits in any batch.
Tolerance 1e-12 rel-L2 per DOF, as for the other FP64 paths."""
import numpy as np
import pytest

from tests.cases import oracle_vhs, oracle_vss, rel_l2, vhs_cfg, vss_cfg
from tests.test_gpu_parity import FP64_TOL, _from_io, _io, _run_vhs, _run_vss

pytestmark = pytest.mark.gpu

N = 24


def _run_nodal(backend, cfg, f, g, nupts, neles):
    import torch
    from frfs_amd.scattering import DGFSVHSGLLNodalScatteringModel
    from frfs_amd.velocitymesh import DGFSVelocityMesh
    sm = DGFSVHSGLLNodalScatteringModel(backend, cfg, DGFSVelocityMesh(backend, cfg))
    fi, gi = (backend.matrix((nupts, N ** 3, neles), _io(a, nupts, neles)) for a in (f, g))
    qo = backend.matrix((nupts, N ** 3, neles))
    sm.fs_batch(fi, gi, qo)
    torch.cuda.synchronize()
    return _from_io(qo.get())


@pytest.mark.parametrize('Nrho,M', [(2, 6), (3, 6), (2, 16)])
def test_twin_sums(backend, Nrho, M):
    """Bilinear: f and g of unlike size (g a thousandth of f)."""
    from oracle import fastspectral as fsp
    cfg = vhs_cfg(N, Nrho, M, 5.0, model='vhs-gll-nodal')
    vm, prm, tab = oracle_vhs(cfg)
    f = fsp.two_maxwellian_batch(vm['cv'], 2, seed=41)
    g = 1e-3 * fsp.two_maxwellian_batch(vm['cv'], 2, seed=42)
    print(f'[pack24 nodal Nrho={Nrho} M={M}]', flush=True)
    Q = _run_nodal(backend, cfg, f, g, 1, 2)
    assert max(rel_l2(Q[d], fsp.vhs_nodal_fs(f[d], g[d], vm, tab, prm['prefac'])) for d in range(2)) <= FP64_TOL


@pytest.mark.parametrize('Nrho,M', [(2, 6), (3, 6), (2, 16)])
def test_group_sums(backend, Nrho, M):
    from oracle import fastspectral as fsp
    cfg = vhs_cfg(N, Nrho, M, 5.0)
    vm, prm, tab = oracle_vhs(cfg)
    f = fsp.two_maxwellian_batch(vm['cv'], 2, seed=43)
    print(f'[pack24 vhs Nrho={Nrho} M={M}]', flush=True)
    Q, _ = _run_vhs(backend, cfg, f, 1, 2)
    assert max(rel_l2(Q[d], fsp.vhs_fs(f[d], vm, tab, prm['prefac'])) for d in range(2)) <= FP64_TOL


def test_single_product_groups(backend):
    from oracle import fastspectral as fsp
    cfg = vss_cfg(N, 3, 12, 5.0)
    vm, prm, tab = oracle_vss(cfg, 1)
    f = fsp.two_maxwellian_batch(vm['cv'], 2, seed=44)
    print('[pack24 vss]', flush=True)
    (Q,), _ = _run_vss(backend, cfg, [f], 1, 2)
    assert max(rel_l2(Q[d], fsp.vss_fs([f[d]], vm, tab, prm)[0]) for d in range(2)) <= FP64_TOL


def test_same_bits_in_any_batch(backend):
    from oracle import fastspectral as fsp
    cv = oracle_vhs(vhs_cfg(N, 2, 6, 5.0))[0]['cv']
    f, g = fsp.two_maxwellian_batch(cv, 20, seed=45), fsp.two_maxwellian_batch(cv, 20, seed=46)
    print('[pack24 batches]', flush=True)
    Q = _run_nodal(backend, vhs_cfg(N, 2, 6, 5.0, model='vhs-gll-nodal'), f, g, 2, 10)
    for chunk in (1, 7):
        assert np.array_equal(_run_nodal(backend, vhs_cfg(N, 2, 6, 5.0, model='vhs-gll-nodal', max_chunk=chunk), f, g,
                                         2, 10), Q)


@pytest.mark.parametrize('prec', ['double', 'mixed'])
def test_row_groups_with_projection(backend, prec):
    """Five DOFs (one past a group of four slots) in batches of 1, 3 and 5: the
    same bits, and collision invariants at rounding level of sum |Q phi|."""
    from oracle import fastspectral as fsp
    cfg = vhs_cfg(N, 2, 6, 5.0, precision=prec, project=1)
    cv = oracle_vhs(cfg)[0]['cv']
    f = fsp.two_maxwellian_batch(cv, 5, seed=47)
    print(f'[rows24 {prec}]', flush=True)
    Q, _ = _run_vhs(backend, cfg, f, 1, 5)
    phi = np.stack([np.ones(N ** 3), *cv, (cv ** 2).sum(0)])
    assert (np.abs(Q @ phi.T) <= 1e-12 * (np.abs(Q) @ np.abs(phi).T)).all()
    for chunk in (1, 3):
        q, _ = _run_vhs(backend, vhs_cfg(N, 2, 6, 5.0, precision=prec, project=1, max_chunk=chunk), f, 1, 5)
        assert np.array_equal(q, Q)
