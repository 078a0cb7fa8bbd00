"""Basis planes on buffers that hold another mesh's planes: a function screened at a point has to be stored as zero there, in
resident and in mesh-block mode, for any share of the shells per block (1, 255 .. 257 points and thousands).  A context
that has evaluated a first mesh gives on a second one, bit for bit, what a fresh context gives (same kernels, same order),
and the atoms are so far apart that each screens the other's functions.
"""
import dataclasses

import numpy as np
import pytest

from publicrelease_2020_amd import system as S

pytestmark = pytest.mark.gpu


def _run(e, sysm, block):
    e.set_mesh_block(block)
    e.set_mesh(sysm.mesh.xyz, sysm.mesh.w)
    e.evaluate()
    return [np.asarray(e.results()["spins"][s][k]) for s in range(2) for k in ("results", "sic", "vab", "debdax")]


@pytest.mark.parametrize("xc", [S.XC_LSDA, S.XC_PBE])
@pytest.mark.parametrize("M,block", [(100, 0), (255, 0), (257, 0), (3000, 0), (3000, 512)])
def test_reused_planes(xc, M, block):
    from publicrelease_2020_amd import flosic as F
    sysm = S.make_synthetic(3, 3, 31, xc, nrad=24, nang=50, box=60.0)
    n = sysm.mesh.npts
    near = np.arange(M) * (n // M)
    second = dataclasses.replace(sysm, mesh=S.Mesh(xyz=np.ascontiguousarray(sysm.mesh.xyz[near]),
                                                   w=np.ascontiguousarray(sysm.mesh.w[near])))
    first = dataclasses.replace(sysm, mesh=S.Mesh(xyz=np.ascontiguousarray(second.mesh.xyz[::-1]),
                                                  w=np.ascontiguousarray(second.mesh.w[::-1])))
    e = F.Flosic(0)
    e.load_system(first, F.PREC_FP64)
    _run(e, first, block)
    used = _run(e, second, block)
    e.close()
    e = F.Flosic(0)
    e.load_system(second, F.PREC_FP64)
    fresh = _run(e, second, block)
    e.close()
    for a, b in zip(used, fresh):
        assert np.all(np.isfinite(b)) and np.array_equal(a, b)
