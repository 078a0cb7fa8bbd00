"""Split-BF16 Coulomb kernels at the edges of their tiles: FLO counts around the 16-column tiles and the limits between one,
two and four column waves and further column blocks (16 | 17, 48 | 49, 96 | 97, 192 | 193), meshes that end inside the first or
second 64-point tile of a block, group counts that end inside a chunk.  Reference: the per-thread VALU form (another kernel,
FP64, summing group by group).  The batched launch has to give the bits of the single one.

Tolerances.  Three pieces carry an operand to 2^-24 and R is made in FP32: 6e-8 * 1e2 in cancellation between Hermite rows
-> 1e-5 of the largest potential.  Two pieces carry 2^-16 per operand: 3e-5 * 1e2 -> 3e-3.
"""
import numpy as np
import pytest

from publicrelease_2020_amd import system as S

pytestmark = pytest.mark.gpu


def _vh(e, sysm):
    return np.array([e.potential(s + 1, i + 1)[1] for s in range(2) for i in range(sysm.nocc[s])])


@pytest.mark.parametrize("K,up,dn,nrad,nang,box", [
    (1, 1, 0, 5, 7, 4.0), (2, 8, 8, 9, 14, 4.5), (3, 9, 8, 8, 24, 4.5), (6, 24, 24, 5, 26, 6.0), (6, 25, 24, 5, 26, 6.0),
    (8, 33, 32, 6, 26, 6.0), (16, 48, 48, 5, 26, 7.0), (16, 49, 48, 5, 27, 7.0), (24, 96, 96, 4, 26, 8.0),
    (24, 97, 96, 4, 27, 8.0)])
def test_tile_edges(K, up, dn, nrad, nang, box, monkeypatch):
    from publicrelease_2020_amd import flosic as F
    sysm = S.make_synthetic(K, up, 40 + K, S.XC_LSDA, nrad=nrad, nang=nang, box=box)
    sysm.nocc[1], sysm.fod[1] = dn, sysm.fod[1][:dn]
    got = {}
    for prec in (2, 3):
        e = F.Flosic(0)
        e.load_system(sysm, prec)
        e.evaluate()
        got[prec] = _vh(e, sysm)
        b = F.FlosicBatch([e])
        b.evaluate()
        assert np.array_equal(_vh(e, sysm), got[prec])
        b.close()
        e.close()
    monkeypatch.setenv("FLOSIC_COULOMB", "valu")
    e = F.Flosic(0)
    e.load_system(sysm, 0)
    e.evaluate()
    ref = _vh(e, sysm)
    e.close()
    top = np.abs(ref).max()
    d3, d2 = (np.abs(got[p] - ref).max() / top for p in (2, 3))
    print(f"{up + dn} FLOs, {sysm.mesh.npts} points: three pieces {d3:.1e}, two {d2:.1e}", flush=True)
    assert d3 <= 1e-5
    assert d2 <= 3e-3


@pytest.mark.parametrize("M", [256 * 64, 256 * 64 + 1, 512 * 64, 512 * 64 + 1, 768 * 64 + 1])
def test_waves_per_tile(M, monkeypatch):
    """Mesh sizes on both sides of the limits between eight waves on one tile and four on each of two (up to 48 FLOs): 256 and
    512 tiles; the tolerance as above, and the batched launch gives the same bits."""
    import dataclasses
    from publicrelease_2020_amd import flosic as F
    full = S.make_synthetic(2, 9, 61, S.XC_LSDA, nrad=150, nang=194, box=5.0)
    idx = np.arange(M) % full.mesh.npts
    sysm = dataclasses.replace(full, mesh=S.Mesh(xyz=np.ascontiguousarray(full.mesh.xyz[idx]),
                                                 w=np.ascontiguousarray(full.mesh.w[idx])))
    e = F.Flosic(0)
    e.load_system(sysm, 2)
    e.evaluate()
    got = _vh(e, sysm)
    b = F.FlosicBatch([e])
    b.evaluate()
    assert np.array_equal(_vh(e, sysm), got)
    b.close()
    e.close()
    monkeypatch.setenv("FLOSIC_COULOMB", "valu")
    e = F.Flosic(0)
    e.load_system(sysm, 0)
    e.evaluate()
    ref = _vh(e, sysm)
    e.close()
    assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()
