"""The LDS-resident FP64 kernels (k_cube_fwd, k_cube, k_cube_out): every grid
they are built for, in each of their forms (products of a group summed, general
pairs, single-product groups), groups longer than one segment, and the same
bits in any batch.  Tolerance 1e-12 rel-L2 per DOF against the oracle, as for
the other FP64 paths."""
import numpy as np
import pytest

from tests.cases import oracle_vhs, oracle_vss, rel_l2, vhs_cfg, vss_cfg
from tests.test_gpu_parity import FP64_TOL, _from_io, _io, _run_vhs, _run_vss

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N', [4, 8, 10, 14, 16, 18, 20])
@pytest.mark.parametrize('M', [6, 16])
def test_group_sums(backend, N, M):
    """VHS: M = 6 is one segment per group, M = 16 two; 5 DOFs, projection off."""
    from oracle import fastspectral as fsp
    cfg = vhs_cfg(N, 2, M, 5.0)
    vm, prm, tab = oracle_vhs(cfg)
    f = fsp.two_maxwellian_batch(vm['cv'], 5, seed=60 + N)
    print(f'[cube vhs N={N} M={M}]', flush=True)
    Q, sm = _run_vhs(backend, cfg, f, 1, 5)
    assert max(rel_l2(Q[d], fsp.vhs_fs(f[d], vm, tab, prm['prefac'])) for d in range(5)) <= FP64_TOL


@pytest.mark.parametrize('N', [6, 8, 16, 18, 20])
def test_single_product_groups(backend, N):
    """VSS: 18 groups, segments of 6 groups."""
    from oracle import fastspectral as fsp
    cfg = vss_cfg(N, 3, 12, 5.0)
    vm, prm, tab = oracle_vss(cfg, 1)
    f = fsp.two_maxwellian_batch(vm['cv'], 3, seed=70 + N)
    print(f'[cube vss N={N}]', flush=True)
    (Q,), sm = _run_vss(backend, cfg, [f], 1, 3)
    assert max(rel_l2(Q[d], fsp.vss_fs([f[d]], vm, tab, prm)[0]) for d in range(3)) <= FP64_TOL


@pytest.mark.parametrize('N', [8, 10, 16, 20])
def test_general_pairs(backend, N):
    """Bilinear vhs-gll-nodal: the two items of a product read different sources."""
    import torch
    from oracle import fastspectral as fsp
    from frfs_amd.scattering import DGFSVHSGLLNodalScatteringModel
    from frfs_amd.velocitymesh import DGFSVelocityMesh
    cfg = vhs_cfg(N, 2, 6, 5.0, model='vhs-gll-nodal')
    vm, prm, tab = oracle_vhs(cfg)
    f = fsp.two_maxwellian_batch(vm['cv'], 3, seed=81)
    g = fsp.two_maxwellian_batch(vm['cv'], 3, seed=82)
    sm = DGFSVHSGLLNodalScatteringModel(backend, cfg, DGFSVelocityMesh(backend, cfg))
    fi, gi = (backend.matrix((1, N ** 3, 3), _io(a, 1, 3)) for a in (f, g))
    qo = backend.matrix((1, N ** 3, 3))
    print(f'[cube nodal N={N}]', flush=True)
    sm.fs_batch(fi, gi, qo)
    torch.cuda.synchronize()
    Q = _from_io(qo.get())
    assert max(rel_l2(Q[d], fsp.vhs_nodal_fs(f[d], g[d], vm, tab, prm['prefac'])) for d in range(3)) <= FP64_TOL


@pytest.mark.parametrize('N', [10, 16])
def test_same_bits_in_any_batch(backend, N):
    from oracle import fastspectral as fsp
    f = fsp.two_maxwellian_batch(oracle_vhs(vhs_cfg(N, 2, 6, 5.0))[0]['cv'], 70, seed=90)
    print(f'[cube batches N={N}]', flush=True)
    Q, _ = _run_vhs(backend, vhs_cfg(N, 2, 6, 5.0), f, 2, 35)
    for chunk in (1, 3, 33):
        q, sm = _run_vhs(backend, vhs_cfg(N, 2, 6, 5.0, max_chunk=chunk), f, 2, 35)
        assert sm._h.chunk_dofs() == chunk and np.array_equal(q, Q)
