"""The library-transform path in FP64 where FP64 plans take the LDS-resident
kernels by default (even grids up to 20^3, one target): with library-fft = 1,
and on 22^3, the smallest grid that takes it by itself.  Against the oracle for
VHS, VSS and the bilinear model, in batches shorter than the library plans'
slots, and captured in a HIP graph.  Tolerance rel-L2 <= 1e-12 per DOF."""
import numpy as np
import pytest

from tests.cases import oracle_vhs, oracle_vss, rel_l2, vhs_cfg, vss_cfg
from tests.test_gpu_parity import FP64_TOL, _from_io, _io, _run_vhs, _run_vss

pytestmark = pytest.mark.gpu


def _library(cfg):
    cfg.set('scattering-model', 'library-fft', 1)
    return cfg


def _is_library(sm):
    return sm._h.paths() == ['library_fft'] and not sm._h.lds_volume()


@pytest.mark.parametrize('N', [4, 6, 12, 20, 22])
def test_vhs(backend, N):
    from oracle import fastspectral as fsp
    cfg = _library(vhs_cfg(N, 4, 6, 5.0))
    vm, prm, tab = oracle_vhs(cfg)
    f = fsp.two_maxwellian_batch(vm['cv'], 6, seed=20 + N)
    print(f'[library vhs N={N}]', flush=True)
    Q, sm = _run_vhs(backend, cfg, f, 2, 3)
    assert _is_library(sm)
    assert max(rel_l2(Q[d], fsp.vhs_fs(f[d], vm, tab, prm['prefac'])) for d in range(6)) <= FP64_TOL


@pytest.mark.parametrize('N', [12, 22])
def test_bilinear(backend, N):
    import torch
    from oracle import fastspectral as fsp
    from frfs_amd.scattering import DGFSVHSGLLNodalScatteringModel
    from frfs_amd.velocitymesh import DGFSVelocityMesh
    cfg = _library(vhs_cfg(N, 3, 6, 5.0, model='vhs-gll-nodal'))
    vm, prm, tab = oracle_vhs(cfg)
    f = fsp.two_maxwellian_batch(vm['cv'], 2, seed=91)
    g = fsp.two_maxwellian_batch(vm['cv'], 2, seed=92)
    sm = DGFSVHSGLLNodalScatteringModel(backend, cfg, DGFSVelocityMesh(backend, cfg))
    assert _is_library(sm)
    fi, gi = (backend.matrix((1, N ** 3, 2), _io(a, 1, 2)) for a in (f, g))
    qo = backend.matrix((1, N ** 3, 2))
    print(f'[library nodal N={N}]', flush=True)
    sm.fs_batch(fi, gi, qo)
    torch.cuda.synchronize()
    Q = _from_io(qo.get())
    assert max(rel_l2(Q[d], fsp.vhs_nodal_fs(f[d], g[d], vm, tab, prm['prefac'])) for d in range(2)) <= FP64_TOL


def test_vss(backend):
    from oracle import fastspectral as fsp
    cfg = _library(vss_cfg(20, 3, 12, 5.0))
    vm, prm, tab = oracle_vss(cfg, 1)
    f = fsp.two_maxwellian_batch(vm['cv'], 3, seed=33)
    print('[library vss N=20]', flush=True)
    (Q,), sm = _run_vss(backend, cfg, [f], 1, 3)
    assert _is_library(sm)
    assert max(rel_l2(Q[d], fsp.vss_fs([f[d]], vm, tab, prm)[0]) for d in range(3)) <= FP64_TOL


def test_ragged_batches(backend):
    """7 DOFs as 3 + 3 + 1 in a 3-slot scratch, and in one batch of a larger one."""
    from oracle import fastspectral as fsp
    vm, prm, tab = oracle_vhs(vhs_cfg(12, 3, 6, 5.0))
    f = fsp.two_maxwellian_batch(vm['cv'], 7, seed=61)
    print('[library ragged N=12]', flush=True)
    Q1, sm1 = _run_vhs(backend, _library(vhs_cfg(12, 3, 6, 5.0)), f, 1, 7)
    Q3, sm3 = _run_vhs(backend, _library(vhs_cfg(12, 3, 6, 5.0, max_chunk=3)), f, 1, 7)
    assert _is_library(sm1) and _is_library(sm3) and sm3._h.chunk_dofs() == 3
    for d in range(7):
        ref = fsp.vhs_fs(f[d], vm, tab, prm['prefac'])
        assert max(rel_l2(Q3[d], ref), rel_l2(Q1[d], ref)) <= FP64_TOL


def test_graph_replay_matches_eager(backend):
    """A captured SSP-RK2 step, replayed three times with eager work between the
    replays, equals eager steps bit for bit."""
    import torch
    from frfs_amd.system import DGFSCollisionSystem, STEPPERS
    from oracle import fastspectral as fsp

    def system(graph):
        sysm = DGFSCollisionSystem(backend, _library(vhs_cfg(12, 3, 6, 5.0, omega=1.0)), 1, 2)
        assert _is_library(sysm.sm)
        return sysm, STEPPERS['dgfs-tvd-rk2'](sysm, graph=graph)
    (sysm_g, stp_g), (sysm_e, stp_e) = system(True), system(False)
    f0 = fsp.bkw(sysm_g.vm.cv(), 5.5)
    init = _io(np.stack([f0, 0.5 * f0]), 1, 2)
    sysm_g.banks[0].set(init)
    sysm_e.banks[0].set(init)
    dt = 0.05 / (4 * np.pi * sysm_g.sm._prefactor)
    print('[library graph N=12]', flush=True)
    for k in range(3):
        stp_g.step(k * dt, dt)
        torch.cuda.synchronize()
        stp_e.step(k * dt, dt)
        torch.cuda.synchronize()
        assert np.isfinite(torch.randn(1 << 20, device='cuda', dtype=torch.float64).sum().item())
        assert np.array_equal(sysm_g.banks[0].get(), sysm_e.banks[0].get()), k
