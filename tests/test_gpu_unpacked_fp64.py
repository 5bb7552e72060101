"""FP64 on 8^3 and 16^3 with pair-pack = 0: the product kernels with one volume
per group (k_prod), which plans of one target take only by this key, against
the oracle for VHS, VSS and the bilinear model.  Tolerance rel-L2 <= 1e-12 per DOF."""
import pytest

from tests.cases import oracle_vhs, oracle_vss, rel_l2, vhs_cfg, vss_cfg
from tests.test_gpu_parity import FP64_TOL, _from_io, _io, _run_vhs, _run_vss

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N', [8, 16])
@pytest.mark.parametrize('project', [0, 1])
def test_vhs(backend, N, project):
    from oracle import fastspectral as fsp
    cfg = vhs_cfg(N, 3, 6, 5.0, pack=0)
    vm, prm, tab = oracle_vhs(cfg)
    f = fsp.two_maxwellian_batch(vm['cv'], 5, seed=60 + N)
    print(f'[unpacked vhs N={N} project={project}]', flush=True)
    Q, sm = _run_vhs(backend, vhs_cfg(N, 3, 6, 5.0, pack=0, project=project), f, 1, 5)
    assert sm._h.paths() == ['fused'] and not sm._h.lds_volume()
    if project:
        P, _ = _run_vhs(backend, vhs_cfg(N, 3, 6, 5.0, project=1), f, 1, 5)
    for d in range(5):
        assert rel_l2(Q[d], P[d] if project else fsp.vhs_fs(f[d], vm, tab, prm['prefac'])) <= FP64_TOL


@pytest.mark.parametrize('N', [8, 16])
def test_vss(backend, N):
    from oracle import fastspectral as fsp
    cfg = vss_cfg(N, 3, 12, 5.0, pack=0)
    vm, prm, tab = oracle_vss(cfg, 1)
    f = fsp.two_maxwellian_batch(vm['cv'], 3, seed=70 + N)
    print(f'[unpacked vss N={N}]', flush=True)
    (Q,), sm = _run_vss(backend, cfg, [f], 1, 3)
    assert sm._h.paths() == ['fused'] and not sm._h.lds_volume()
    assert max(rel_l2(Q[d], fsp.vss_fs([f[d]], vm, tab, prm)[0]) for d in range(3)) <= FP64_TOL


@pytest.mark.parametrize('N', [8, 16])
def test_bilinear(backend, N):
    import torch
    from oracle import fastspectral as fsp
    from frfs_amd.scattering import DGFSVHSGLLNodalScatteringModel
    from frfs_amd.velocitymesh import DGFSVelocityMesh
    cfg = vhs_cfg(N, 2, 6, 5.0, model='vhs-gll-nodal', pack=0)
    vm, prm, tab = oracle_vhs(cfg)
    f = fsp.two_maxwellian_batch(vm['cv'], 3, seed=81)
    g = fsp.two_maxwellian_batch(vm['cv'], 3, seed=82)
    sm = DGFSVHSGLLNodalScatteringModel(backend, cfg, DGFSVelocityMesh(backend, cfg))
    assert sm._h.paths() == ['fused'] and not sm._h.lds_volume()
    fi, gi = (backend.matrix((1, N ** 3, 3), _io(a, 1, 3)) for a in (f, g))
    qo = backend.matrix((1, N ** 3, 3))
    print(f'[unpacked nodal N={N}]', flush=True)
    sm.fs_batch(fi, gi, qo)
    torch.cuda.synchronize()
    Q = _from_io(qo.get())
    assert max(rel_l2(Q[d], fsp.vhs_nodal_fs(f[d], g[d], vm, tab, prm['prefac'])) for d in range(3)) <= FP64_TOL
