"""Batched Coulomb launches at narrow column blocks whose tiles do not share out evenly: 64-column blocks of three and four
tiles (7, 10 and 13 tiles in all), where a column wave of the smaller block holds a single tile.  The batched launch has to
give the bits of the launch for one system.  The context of the batch evaluated the FODs in another order before, so a column
that the launch leaves unwritten shows another orbital's potential.
"""
import numpy as np
import pytest

from publicrelease_2020_amd import system as S

pytestmark = pytest.mark.gpu


def _vh(e, sysm):
    return np.array([e.potential(s + 1, i + 1)[1] for s in range(2) for i in range(sysm.nocc[s])])


@pytest.mark.parametrize("prec", [0, 1, 2, 3])
@pytest.mark.parametrize("K,up,dn", [(16, 49, 48), (16, 56, 56), (24, 80, 80), (24, 97, 96)])
def test_uneven_blocks(K, up, dn, prec):
    from publicrelease_2020_amd import flosic as F
    sysm = S.make_synthetic(K, up, 40 + K, S.XC_LSDA, nrad=4, nang=26, box=8.0)
    sysm.nocc[1], sysm.fod[1] = dn, sysm.fod[1][:dn]
    e = F.Flosic(0)
    e.load_system(sysm, prec)
    e.set_coulomb_cols(64)
    e.evaluate()
    ref = _vh(e, sysm)
    e.close()
    e = F.Flosic(0)
    e.load_system(sysm, prec)
    e.set_coulomb_cols(64)
    for s in (1, 2):
        e.set_fods(s, np.roll(sysm.fod[s - 1], 1, axis=0))
    e.evaluate()
    assert not np.isclose(_vh(e, sysm), ref, rtol=1e-6, atol=0.0).all(1).any()
    for s in (1, 2):
        e.set_fods(s, sysm.fod[s - 1])
    b = F.FlosicBatch([e])
    b.evaluate()
    assert np.array_equal(_vh(e, sysm), ref)
    b.close()
    e.close()


def test_autotuned_width():
    """200 FLOs: blocks of 256 and of 128 columns are the same launch, which counts as the wider one."""
    from publicrelease_2020_amd import flosic as F
    sysm = S.make_synthetic(24, 100, 64, S.XC_LSDA, nrad=4, nang=26, box=8.0)
    e = F.Flosic(0)
    e.load_system(sysm)
    e.evaluate()
    ref = _vh(e, sysm)
    e.set_coulomb_cols(-1)
    e.evaluate()
    assert e.coulomb_cols() in (256, 64)
    assert np.abs(_vh(e, sysm) - ref).max() <= 1e-12 * np.abs(ref).max()  # FP64 sums of other runs of rows
    e.close()
