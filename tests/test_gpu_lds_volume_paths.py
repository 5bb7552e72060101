"""Which kernels a handle runs: the LDS-resident FP64 kernels report
FQ_PATH_LDS_VOLUME, no other plan does, and the stages that the profile counts
are theirs (three launches per batch, no z stage and no accumulation of their
own) or the other path's."""
import pytest

from tests.cases import vhs_cfg, vss_cfg
from tests.test_zz_no_alloc import _call, _inputs, _model

pytestmark = pytest.mark.gpu


def _stages(backend, cfg, vss):
    """lds_volume and the names of the stages of one call on two DOFs."""
    from frfs_amd import _lib
    vm, sm = _model(backend, cfg, vss)
    fin = _inputs(backend, vm, 2, seed=71)
    q = backend.matrix(fin.ioshape)
    sm._h.profile(True)
    _lib.check(_call(sm._h._h, _lib.load().fq_eval, fin, q, 2))
    ran = {k: n for k, (_, n) in sm._h.profile_read().items() if n}
    sm._h.profile(False)
    return sm._h.lds_volume(), ran


@pytest.mark.parametrize('N', [4, 6, 8, 10, 12, 14, 16, 18, 20])
@pytest.mark.parametrize('vss', [False, True])
def test_lds_volume(backend, N, vss):
    cfg = vss_cfg(N, 2, 12, 5.0) if vss else vhs_cfg(N, 2, 6, 5.0)
    print(f'[lds volume N={N} vss={vss}]', flush=True)
    lds, ran = _stages(backend, cfg, vss)
    assert lds and ran == {'k_fwd_xy': 1, 'k_prod': 1, 'k_out': 1}


def _library(cfg):
    cfg.set('scattering-model', 'library-fft', 1)
    return cfg


@pytest.mark.parametrize('label,make', [
    ('library flag', lambda: _library(vhs_cfg(12, 2, 6, 5.0))), ('library flag 16', lambda: _library(vhs_cfg(16, 2, 6, 5.0))),
    ('mixed', lambda: vhs_cfg(12, 2, 6, 5.0, precision='mixed')), ('22', lambda: vhs_cfg(22, 2, 6, 5.0)),
    ('mixed 16', lambda: vhs_cfg(16, 2, 6, 5.0, precision='mixed')), ('unfused', lambda: vhs_cfg(16, 2, 6, 5.0, fused=0)),
    ('unpacked', lambda: vhs_cfg(8, 2, 6, 5.0, pack=0)), ('24', lambda: vhs_cfg(24, 2, 6, 5.0))])
def test_other_paths(backend, label, make):
    print(f'[not lds volume: {label}]', flush=True)
    lds, ran = _stages(backend, make(), False)
    assert not lds and 'k_accum' in ran and 'k_fwd_z' in ran


@pytest.mark.parametrize('N,project', [(8, 0), (16, 1), (18, 0)])
def test_in_place(backend, N, project):
    """Q written over f, in several batches, has the bits of Q beside f."""
    import numpy as np
    from frfs_amd import _lib
    vm, sm = _model(backend, vhs_cfg(N, 2, 6, 5.0, project=project, max_chunk=5), False)
    assert sm._h.lds_volume()
    fin = _inputs(backend, vm, 37, seed=72)
    q = backend.matrix(fin.ioshape)
    print(f'[lds volume in place N={N}]', flush=True)
    _lib.check(_call(sm._h._h, _lib.load().fq_eval, fin, q, 37))
    want = q.get()
    _lib.check(_call(sm._h._h, _lib.load().fq_eval, fin, fin, 37))
    assert np.array_equal(fin.get(), want)
