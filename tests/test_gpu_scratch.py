"""Scratch that a handle holds: the projection's plane sums take none of their own,
and plans that fq_eval_noalloc serves with a volume per group are served."""
import numpy as np
import pytest

from tests.cases import vhs_cfg
from tests.test_zz_no_alloc import _call, _inputs, _model

pytestmark = pytest.mark.gpu


def _vhs_model(backend, **kw):
    return _model(backend, vhs_cfg(**kw), False)[1]


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
