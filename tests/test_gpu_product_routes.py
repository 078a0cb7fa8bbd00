"""The sums over the mesh on both sides of the limits at which the library's product takes over from the kernel: 5e9 (49 to 64,
97 to 128, .. columns) and 3e9 (above 192) rows x columns x points, 48 | 49 columns, with points that no slice count divides;
and DERSIC with its gradient planes stacked, one by one in the kernel, and one by one in the library.  SIC(j,i), the AO SIC
Hamiltonian and DERSIC are formed again by torch in float64 from the library's potentials and TMAT.

Tolerance: sums of 2e5 rounded products, 1e-16 * sqrt(2e5) with up to 1e3 in cancellation: 5e-11 of the largest.
"""
import numpy as np
import pytest

from publicrelease_2020_amd import system as S

pytestmark = pytest.mark.gpu


# side: points up to the limit (-1) and beyond it (1)
@pytest.mark.parametrize("up,dn,side,block", [(24, 24, 0, 0), (25, 24, 0, 0), (32, 31, -1, 0), (32, 31, 1, 0), (56, 54, -1, 0), (56, 54, 1, 0),
                                              (56, 54, 1, 16384), (100, 97, -1, 0), (100, 97, 1, 0)])
def test_sums_over_points(up, dn, side, block):
    import torch
    from publicrelease_2020_amd import flosic as F
    K, nF, box = 22, up + dn, 13.0
    N = S.make_synthetic(K, 2, 232, S.XC_LSDA, nrad=2, nang=14, box=box).basis.nbas
    npts = 20011 if side == 0 else int((3e9 if nF > 192 else 5e9) / (N * nF)) + 77 * side
    sysm = S.make_synthetic(K, up, 232, S.XC_LSDA, nrad=-(-npts // (K * 100)), nang=110, box=box)
    assert sysm.basis.nbas == N and sysm.mesh.npts >= npts
    sysm.mesh = S.Mesh(xyz=sysm.mesh.xyz[-npts:].copy(), w=sysm.mesh.w[-npts:].copy())
    sysm.nocc[1], sysm.fod[1] = dn, sysm.fod[1][:dn]
    e = F.Flosic(0)
    e.load_system(sysm, F.PREC_MIXED)
    e.evaluate()
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")
    chi = t(S.eval_basis(sysm.basis, sysm.mesh.xyz, 1))
    w, cflo, V = t(sysm.mesh.w)[:, None], [], []
    for s, n in ((1, up), (2, dn)):
        cflo.append(t(sysm.coef[s - 1][:, :n]) @ t(e.fermi_orbitals(s)["tmat"]).T)
        V.append(torch.stack([t(e.potential(s, i + 1)[0]) for i in range(n)], 1))
    if block:
        e.set_mesh_block(block)
        e.evaluate()

    def near(got, ref):
        return np.abs(got - ref.cpu().numpy()).max() <= 5e-11 * float(ref.abs().max())
    der, at = [], t(np.array([a for a, *_ in sysm.basis.functions()]))
    for s, n in ((1, up), (2, dn)):
        c, C = cflo[s - 1], t(sysm.coef[s - 1])
        phi = chi[0] @ c
        U = w * V[s - 1] * phi
        G = chi[0].T @ U
        assert near(e.siclagm(s), -torch.cat([c, C[:, n:]], 1).T @ G)
        B = chi[0].T @ (w * phi)
        assert near(e.sic_hamiltonian(s), 0.5 * (G @ B.T + B @ G.T))
        D = torch.stack([-c * (chi[1 + x].T @ U) for x in range(3)], 2)
        der.append(torch.zeros(sysm.basis.natom, n, 3, dtype=torch.float64, device="cuda").index_add_(0, at, D))
    assert near(e.siclag_der(), torch.cat(der, 1))
    e.close()
