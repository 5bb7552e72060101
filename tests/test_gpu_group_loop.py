"""FP64 32^3 with single-product groups: k_prod takes several groups per
workgroup once four workgroups per CU remain (at 256 CUs, 18 groups: 16 and 2
per workgroup from 128 DOFs, 8, 8 and 2 from 86, 4, 4, 4, 4 and 2 from 52, two
from 29).  Each batch gives a DOF the bits of one DOF alone, which takes one
group per workgroup and is checked against the oracle at 1e-12.  With 12 groups
the loop takes all of a slot's in one workgroup."""
import numpy as np
import pytest

from tests.cases import oracle_vss, rel_l2, vss_cfg
from tests.test_gpu_parity import FP64_TOL, _run_vss

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('Nrho,sizes', [(3, (150, 130, 90, 55, 30)), (2, (256,))])
def test_groups_per_workgroup(backend, Nrho, sizes):
    from oracle import fastspectral as fsp
    cfg = vss_cfg(32, Nrho, 12, 6.0)
    vm, prm, tab = oracle_vss(cfg, 1)
    nd = max(sizes)
    f = np.repeat(fsp.two_maxwellian_batch(vm['cv'], 10, seed=90), -(-nd // 10), axis=0)[:nd]
    f *= (1 + np.arange(nd) / nd)[:, None]
    print(f'[group loop Nrho={Nrho}] one DOF at a time', flush=True)
    (one,), sm = _run_vss(backend, vss_cfg(32, Nrho, 12, 6.0, max_chunk=1), [f], 1, nd)
    assert sm._h.paths() == ['fused', 'pair_pack'] and sm.plan_info()['n_groups'] == 6 * Nrho
    for d in (0, nd - 1):
        assert rel_l2(one[d], fsp.vss_fs([f[d]], vm, tab, prm)[0]) <= FP64_TOL
    for n in sizes:
        print(f'[group loop Nrho={Nrho}] {n} DOFs', flush=True)
        (Q,), sm = _run_vss(backend, vss_cfg(32, Nrho, 12, 6.0, max_chunk=max(n, 96)), [f[:n]], 1, n)
        assert np.array_equal(Q, one[:n])
