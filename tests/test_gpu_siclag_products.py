"""flosic_siclag_der on both sides of 80 FLOs, where the three gradient products go from one product of 3 N rows to three of N
rows: resident and mesh-block mode, LSDA and PBE, against the oracle.

Tolerance: sums of about 1e4 products of order one at 1e-16 each, up to 1e3 in cancellation -> 1e-10 of the largest.
"""
import numpy as np
import pytest

from publicrelease_2020_amd import system as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("xc,block", [(S.XC_LSDA, 0), (S.XC_LSDA, 256), (S.XC_PBE, 0)])
@pytest.mark.parametrize("up,dn", [(40, 40), (41, 40)])
def test_products(xc, block, up, dn):
    from oracle import oracle as O
    from publicrelease_2020_amd import flosic as F
    sysm = S.make_synthetic(8, up, 77, xc, nrad=4, nang=14, box=6.0)
    sysm.nocc[1], sysm.fod[1] = dn, sysm.fod[1][:dn]
    ctx = F.Flosic(0)
    ctx.load_system(sysm)
    if block:
        ctx.set_mesh_block(block)
    ctx.evaluate()
    d = ctx.siclag_der()
    ctx.close()
    ref = O.evaluate(sysm, nthreads=16, want_potentials=True, want_vab=False)
    assert ref["status"] == 0
    d_ref = O.siclag_der(sysm, np.vstack([ref["spins"][0]["vpot"], ref["spins"][1]["vpot"]]))
    assert d.shape == d_ref.shape
    assert np.abs(d - d_ref).max() <= 1e-10 * np.abs(d_ref).max()
