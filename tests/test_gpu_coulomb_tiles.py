"""FP64 and FP32 Coulomb kernels at the edges of their tiles: FLO counts around the 16-column tiles, the column-wave and
column-block limits (16 | 17, 64 | 65, 96 | 97, 192 | 193), meshes that end inside a 64-point tile, group counts that end
inside a unit.  Reference: the per-thread VALU form (another kernel, FP64, summing group by group).

Tolerances.  FP64: both forms sum the same ~1e4 products in another order; with at most 1e3 in cancellation between
Hermite rows that is 1e-16 * 1e3 * sqrt(1e4) = 1e-11 of the largest potential.  FP32: operands rounded to 2^-24 and
chunk sums of 64 rows in FP32, 6e-8 * 1e2 in cancellation -> 1e-5.
"""
import numpy as np
import pytest

from publicrelease_2020_amd import system as S

pytestmark = pytest.mark.gpu


def _vh(sysm, prec):
    from publicrelease_2020_amd import flosic as F
    e = F.Flosic(0)
    e.load_system(sysm, prec)
    e.evaluate()
    out = np.array([e.potential(s + 1, i + 1)[1] for s in range(2) for i in range(sysm.nocc[s])])
    e.close()
    return out


@pytest.mark.parametrize("K,up,dn,nrad,nang,box", [
    (1, 1, 0, 5, 7, 4.0), (2, 8, 8, 9, 14, 4.5), (3, 9, 8, 8, 24, 4.5), (8, 32, 32, 6, 26, 6.0),
    (8, 33, 32, 6, 26, 6.0), (16, 48, 48, 5, 26, 7.0), (16, 49, 48, 5, 26, 7.0), (24, 96, 96, 4, 26, 8.0),
    (24, 97, 96, 4, 27, 8.0)])
def test_tile_edges(K, up, dn, nrad, nang, box, monkeypatch):
    sysm = S.make_synthetic(K, up, 40 + K, S.XC_LSDA, nrad=nrad, nang=nang, box=box)
    sysm.nocc[1], sysm.fod[1] = dn, sysm.fod[1][:dn]
    v64, v32 = _vh(sysm, 0), _vh(sysm, 1)
    monkeypatch.setenv("FLOSIC_COULOMB", "valu")
    ref = _vh(sysm, 0)
    top = np.abs(ref).max()
    print(f"{up + dn} FLOs, {sysm.mesh.npts} points: FP64 {np.abs(v64 - ref).max() / top:.1e}, "
          f"FP32 {np.abs(v32 - ref).max() / top:.1e}", flush=True)
    assert np.abs(v64 - ref).max() <= 1e-11 * top
    assert np.abs(v32 - ref).max() <= 1e-5 * top
