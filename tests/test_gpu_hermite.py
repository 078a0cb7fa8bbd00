"""Hermite coefficients at the edges of the column tiles (16 | 17, 32 | 33, 64 | 65 FLOs, one FLO): the FP64 evaluation on a
small mesh against the oracle, which builds the pair expansion by another route.

Tolerance: every number is a sum of about 1e5 products of order one at 1e-16 each, in another order, with up to 1e3 in
cancellation between Hermite rows: 1e-16 * 1e3 * sqrt(1e5) -> 1e-10 relative.
"""
import numpy as np
import pytest

from publicrelease_2020_amd import system as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,up,dn", [(1, 1, 0), (2, 8, 8), (3, 9, 8), (4, 16, 16), (5, 17, 16), (8, 32, 32), (8, 33, 32)])
def test_column_edges(K, up, dn):
    from oracle import oracle as O
    from publicrelease_2020_amd import flosic as F
    sysm = S.make_synthetic(K, up, 70 + K, S.XC_LSDA, nrad=4, nang=14, box=5.0)
    sysm.nocc[1], sysm.fod[1] = dn, sysm.fod[1][:dn]
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
        g, o = np.asarray(got["spins"][s]["results"]), np.asarray(r["spins"][s]["results"])
        print(f"{up + dn} FLOs, spin {s + 1}: {np.abs(g - o).max() / np.abs(o).max():.1e}", flush=True)
        assert np.abs(g - o).max() <= 1e-10 * np.abs(o).max()
