"""Scratch of the FP64 plans whose kernels take more per DOF than the product
volumes (or the library path's arrays) would: for the same max_chunk they hold
no more bytes, or no more than the default budget; plans that fq_eval_noalloc
serves with the product volumes are served; the projection's plane sums take no
scratch of their own."""
import numpy as np
import pytest

from tests.cases import vhs_cfg
from tests.test_zz_no_alloc import _call, _inputs, _model

pytestmark = pytest.mark.gpu

VOL = 16                                   # bytes of a grid point in a complex volume


def _vhs_model(backend, **kw):
    return _model(backend, vhs_cfg(**kw), False)[1]


BUDGET = 8 << 30                           # the default scratch


@pytest.mark.parametrize('Nrho,max_chunk', [(32, 8192), (60, 12000)])
def test_cube_within_the_library_paths_bytes(backend, Nrho, max_chunk):
    """20^3: the spectrum, gain and loss, and three work volumes per slot, or the
    default budget where that is more."""
    slot = 6 * VOL * 20 ** 3
    sm = _vhs_model(backend, Nv=20, Nrho=Nrho, M=6, max_chunk=max_chunk)
    print('[scratch cube]', sm._h.scratch_bytes(), sm._h.chunk_dofs(), flush=True)
    assert sm._h.lds_volume() and sm._h.chunk_dofs() < max_chunk
    assert 0.99 * max(BUDGET, max_chunk * slot) <= sm._h.scratch_bytes() <= max(BUDGET, max_chunk * slot)


def test_cube_takes_max_chunk_within_the_budget(backend):
    for kw in (dict(Nrho=32, max_chunk=100), dict(Nrho=2, max_chunk=8192)):
        sm = _vhs_model(backend, Nv=20, M=6, **kw)
        assert sm._h.chunk_dofs() == kw['max_chunk']
    assert _vhs_model(backend, Nv=20, Nrho=32, M=6)._h.scratch_bytes() <= BUDGET


def test_twin_packing_within_the_unpacked_bytes(backend):
    from frfs_amd.scattering import DGFSVHSGLLNodalScatteringModel
    from frfs_amd.velocitymesh import DGFSVelocityMesh
    got = {}
    for pack in (1, 0):
        cfg = vhs_cfg(24, 4, 16, 5.0, model='vhs-gll-nodal', max_chunk=6000, pack=pack)
        got[pack] = DGFSVHSGLLNodalScatteringModel(backend, cfg, DGFSVelocityMesh(backend, cfg))._h.scratch_bytes()
    print('[scratch twin]', got, flush=True)
    assert BUDGET < got[1] <= got[0]


@pytest.mark.parametrize('N,prec', [(24, 'double'), (24, 'mixed'), (32, 'double'), (32, 'mixed')])
def test_projection_takes_no_scratch(backend, N, prec):
    a, b = (_vhs_model(backend, Nv=N, Nrho=2, M=6, precision=prec, project=p, max_chunk=4)._h.scratch_bytes()
            for p in (0, 1))
    assert a == b


def test_noalloc_serves_many_segments(backend):
    """16^3, Nrho = 700, M = 96: 46 MB per DOF with a product volume per group,
    and 275 MB with a volume per eight products."""
    from frfs_amd import _lib
    lib = _lib.load()
    vm, sm = _model(backend, vhs_cfg(16, 700, 96, 5.0, max_chunk=1), False)
    fin = _inputs(backend, vm, 1, seed=61)
    q, w = backend.matrix(fin.ioshape), backend.matrix(fin.ioshape)
    print('[noalloc many segments]', flush=True)
    _lib.check(_call(sm._h._h, lib.fq_eval_noalloc, fin, q, 1))
    _lib.check(_call(sm._h._h, lib.fq_eval, fin, w, 1))
    assert np.isfinite(w.get()).all() and np.array_equal(q.get(), w.get())
