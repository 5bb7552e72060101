"""Batches of few DOFs on the 32^3 group-pair path take kernels of their own
(k_nyqt + k_nyqc, k_hz + k_hsum, fewer points per k_project_b workgroup): a DOF
gets the same bits in any batch, on either side of each rule's line."""
import numpy as np
import pytest

from cases import vss_cfg

pytestmark = pytest.mark.gpu

MASSES = (39.96e-3, 2 * 39.96e-3)


def _model(be, ns, project):
    from frfs_amd.scattering import DGFSBiVSSGLLScatteringModel
    from frfs_amd.velocitymesh import DGFSBiVelocityMesh
    cfg = vss_cfg(32, 2, 12, 6.0, masses=MASSES[:ns], precision='mixed', project=project)
    return DGFSBiVSSGLLScatteringModel(be, cfg, DGFSBiVelocityMesh(be, cfg, ns))


@pytest.mark.parametrize('ns,sizes', [(1, (1, 16, 17, 60, 61, 256, 257)), (2, (1, 8, 9, 30, 31, 128, 129))])
def test_same_bits_in_any_batch(ns, sizes):
    from frfs_amd.backend import HIPBackend
    from frfs_amd.inputs import mixture_device, mixture_params, to_aosoa
    be = HIPBackend()
    m = _model(be, ns, 1)
    assert 'group_pairs' in m._h.paths()
    nd = max(sizes) + 3
    f, q, one = [], [], []
    for s in range(ns):
        a = be.matrix((1, 32 ** 3, nd))
        to_aosoa(mixture_device(m.vm.cv(), mixture_params(nd, 31 + s)), a)
        f.append(a)
        q.append(be.matrix(a.ioshape))
        one.append(be.matrix(a.ioshape))
    m.fs_batch(*f, *one)                                   # the largest batch: the one-kernel forms
    ref = [a.get() for a in one]
    for d in sizes:
        print(f'[small batches] {ns} species, {d} DOFs', flush=True)
        for a in q:
            a.data.fill_(7.0)
        m.fs_batch(*f, *q, first_dof=3, ndof=d)
        for a, r in zip(q, ref):
            got = a.get()
            assert np.array_equal(got[..., 3:3 + d], r[..., 3:3 + d])
            assert (got[..., :3] == 7.0).all() and (got[..., 3 + d:] == 7.0).all()
