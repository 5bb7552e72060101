"""Scratch that a handle holds: the projection's plane sums take none of their own."""
import pytest

from tests.cases import vhs_cfg
from tests.test_zz_no_alloc import _model

pytestmark = pytest.mark.gpu


def _vhs_model(backend, **kw):
    return _model(backend, vhs_cfg(**kw), False)[1]


@pytest.mark.parametrize('N,prec', [(24, 'double'), (24, 'mixed'), (32, 'double'), (32, 'mixed')])
def test_projection_takes_no_scratch(backend, N, prec):
    a, b = (_vhs_model(backend, Nv=N, Nrho=2, M=6, precision=prec, project=p, max_chunk=4)._h.scratch_bytes()
            for p in (0, 1))
    assert a == b
