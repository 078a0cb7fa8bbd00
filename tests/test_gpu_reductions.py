"""Sums of the per-block partials: block counts around the 16 ranges of a sum and the 8 loads in flight (1, 2, 15 .. 17, 127 ..
129 blocks of 256 points), output counts around 64.  RESULTS and V^i_ab of the FP64 evaluation against the oracle.

Tolerance: every number is a sum of about 1e5 products of order one at 1e-16 each, in another order, with up to 1e3 in
cancellation -> 1e-10 of the largest.
"""
import dataclasses

import numpy as np
import pytest

from publicrelease_2020_amd import system as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,up,dn,M", [(1, 1, 0, 100), (1, 1, 0, 256), (1, 2, 1, 257), (1, 4, 4, 3840), (2, 4, 3, 4096), (2, 5, 4, 4097),
                                       (1, 3, 2, 32512), (1, 3, 2, 32768), (1, 3, 2, 33000)])
def test_partial_sums(K, up, dn, M):
    from oracle import oracle as O
    from publicrelease_2020_amd import flosic as F
    full = S.make_synthetic(K, up, 90 + K, S.XC_LSDA, nrad=180, nang=194, box=5.0)
    full.nocc[1], full.fod[1] = dn, full.fod[1][:dn]
    idx = np.arange(M) * (full.mesh.npts // M)
    sysm = dataclasses.replace(full, mesh=S.Mesh(xyz=np.ascontiguousarray(full.mesh.xyz[idx]),
                                                 w=np.ascontiguousarray(full.mesh.w[idx])))
    r = O.evaluate(sysm, nthreads=16)
    assert r["status"] == 0
    e = F.Flosic(0)
    e.load_system(sysm, F.PREC_FP64)
    e.evaluate()
    got = e.results()
    e.close()
    for s in range(2):
        if sysm.nocc[s] == 0:
            continue
        for k in ("results", "vab"):
            g, o = np.asarray(got["spins"][s][k]), np.asarray(r["spins"][s][k])
            assert np.abs(g - o).max() <= 1e-10 * np.abs(o).max(), k
