"""Projector products at the edges of their tile choice (32, 64 and 128 wide tiles, one to many
K slices, outputs that are not multiples of the tile, one band, one projector): the non-local
part of Hψ and Enl against the same sums in 64-bit torch, Γ and complex bases.

Errors are measured against the same sums over absolute values (a single projector's sum can
cancel): each of the two products rounds its inputs and its partial sums, 1.1e-16 (FP64) or 6e-8
(FP32) of that size a few times over, so the bars are 1e-15 and 5e-7.
"""
import numpy as np
import pytest

from helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu

# atoms, l of the projectors, bands, cell replication
SHAPES = [(1, [0], 1, 1), (3, [0, 1], 16, 1), (8, [0, 1, 1, 1], 16, 1), (11, [0, 1, 2], 31, 1),
          (8, [0, 1, 1, 1], 33, 1), (17, [0, 1, 1, 1], 65, 1), (64, [0, 1, 1, 1], 128, 1),
          (33, [0, 1, 1, 1], 129, 2), (100, [0, 1, 1, 1, 2, 2, 2, 2, 2], 257, 1),
          (300, [0, 1, 1, 1], 320, 1)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("real", [True, False])
def test_tiles(gpu_ctx, shape, real):
    import torch
    from helpers import make_gpu_basis
    from qball_amd import Hamiltonian
    from qball_amd.workload import make_system
    natoms, lproj, nst, ncell = shape
    sysm = make_system(ncell=ncell, ecut_ry=25.0 if ncell == 1 else 18.0, nbands=nst, seed=31,
                       complex_basis=not real)
    rng = np.random.default_rng(32)
    tau = rng.uniform(0.0, 10.0, (natoms, 3))
    twnl = rng.standard_normal((len(lproj), sysm.ngw)) / (1.0 + sysm.g2)
    wt = rng.uniform(-1.0, 1.0, len(lproj))
    occ = rng.uniform(0.0, 2.0, nst)
    kpg = torch.from_numpy(sysm.kpg).cuda()
    ph = -(kpg @ torch.from_numpy(tau).cuda().T)
    ph = torch.complex(torch.cos(ph), torch.sin(ph)).T
    t = torch.from_numpy(twnl).cuda()
    beta = torch.cat([(-1j) ** l * t[i] * ph for i, l in enumerate(lproj)])
    D = torch.from_numpy(np.repeat(wt, natoms) / sysm.omega).cuda()
    psi = torch.from_numpy(np.ascontiguousarray(sysm.psi.T)).cuda()

    def view(c):
        return torch.view_as_real(c).reshape(len(c), -1)
    if real:
        F = 2.0 * view(beta) @ view(psi).T - beta[:, :1].real @ psi[:, :1].real.T
        ref = torch.view_as_complex(((D[:, None] * F).T @ view(beta)).reshape(psi.shape + (2,)))
    else:
        F = beta.conj() @ psi.T
        ref = (D[:, None] * F).T @ beta
    Fa = 2.0 * view(beta).abs() @ view(psi).abs().T
    size = float(((D.abs()[:, None] * Fa).T @ view(beta).abs()).norm())
    enl_ref = float((D[:, None] * torch.from_numpy(occ).cuda() * F.abs().square()).sum())
    enl_size = float((D.abs()[:, None] * torch.from_numpy(occ).cuda() * Fa.square()).sum())
    ref = ref.cpu().numpy().T

    basis = make_gpu_basis(gpu_ctx, sysm)
    ham = Hamiltonian(gpu_ctx, basis)
    ham.set_projectors([natoms], [len(lproj)], lproj, wt, twnl.ravel(), tau.ravel(), sysm.omega)
    ham.set_tuning("fnl_algo", 17)
    ham.set_tuning("enl_algo", 17)
    cd = to_dev(sysm.psi)
    for flags, tol in ((0x1, 1e-15), (0x11, 5e-7)):
        hd = torch.full_like(cd, np.nan)
        torch.cuda.synchronize()
        enl = ham.hpsi(cd.data_ptr(), basis.ngw, nst, occ, hd.data_ptr(), basis.ngw, flags=flags,
                       want_enl=True)
        gpu_ctx.sync()
        assert np.linalg.norm(from_dev(hd, basis.ngw, nst) - ref) <= tol * size, flags
        assert abs(enl - enl_ref) <= tol * enl_size, flags
        ham.hpsi(cd.data_ptr(), basis.ngw, nst, occ, hd.data_ptr(), basis.ngw, flags=flags | 0x8)
        gpu_ctx.sync()
        assert np.linalg.norm(from_dev(hd, basis.ngw, nst) - 2 * ref) <= 2 * tol * size, flags
    ham.close()
    basis.close()


# atoms, bands, cutoff; widths of the tiles of F and Hψ += βF in FP64, then in FP32
WIDE = [(150, 200, 80.0, (128, 128), (128, 32)), (250, 390, 60.0, (128, 64), (128, 64)),
        (200, 390, 60.0, (64, 64), (64, 64)), (100, 100, 60.0, (32, 64), (32, 32))]


@pytest.mark.parametrize("natoms,nst,ecut,tiles64,tiles32", WIDE)
def test_wide_tiles(gpu_ctx, natoms, nst, ecut, tiles64, tiles32):
    """The 64 and 128 wide tiles of both products over several tiles and slices (Γ), with the
    tiles that ran."""
    import torch
    from helpers import make_gpu_basis, product_tile
    from qball_amd import Hamiltonian
    from qball_amd.workload import make_system
    lproj = [0, 1, 1, 1]
    sysm = make_system(ncell=1, ecut_ry=ecut, nbands=nst, seed=33)
    P, Q = 4 * natoms, 2 * sysm.ngw
    for fp32, tiles in ((0, tiles64), (1, tiles32)):
        assert (product_tile(fp32, P, nst, Q)[0], product_tile(2 + fp32, nst, Q, P)[0]) == tiles
    rng = np.random.default_rng(34)
    tau = rng.uniform(0.0, 10.0, (natoms, 3))
    twnl = rng.standard_normal((4, sysm.ngw)) / (1.0 + sysm.g2)
    wt = rng.uniform(-1.0, 1.0, 4)
    ph = -(torch.from_numpy(sysm.kpg).cuda() @ torch.from_numpy(tau).cuda().T)
    ph = torch.complex(torch.cos(ph), torch.sin(ph)).T
    t = torch.from_numpy(twnl).cuda()
    beta = torch.view_as_real(torch.cat([(-1j) ** l * t[i] * ph for i, l in enumerate(lproj)]))
    psi = torch.view_as_real(torch.from_numpy(np.ascontiguousarray(sysm.psi.T)).cuda())
    beta, psi = beta.reshape(P, Q), psi.reshape(nst, Q)
    D = torch.from_numpy(np.repeat(wt, natoms) / sysm.omega).cuda()
    F = 2.0 * beta @ psi.T - beta[:, :1] @ psi[:, :1].T
    ref = ((D[:, None] * F).T @ beta).cpu().numpy().view(np.complex128).T
    size = float(((D.abs()[:, None] * (2.0 * beta.abs() @ psi.abs().T)).T @ beta.abs()).norm())
    basis = make_gpu_basis(gpu_ctx, sysm)
    ham = Hamiltonian(gpu_ctx, basis)
    ham.set_projectors([natoms], [4], lproj, wt, twnl.ravel(), tau.ravel(), sysm.omega)
    ham.set_tuning("fnl_algo", 17)
    ham.set_tuning("enl_algo", 17)
    cd = to_dev(sysm.psi)
    for flags, tol in ((0x1, 1e-15), (0x11, 5e-7)):
        hd = torch.full_like(cd, np.nan)
        torch.cuda.synchronize()
        ham.hpsi(cd.data_ptr(), basis.ngw, nst, sysm.occ, hd.data_ptr(), basis.ngw, flags=flags)
        gpu_ctx.sync()
        assert np.linalg.norm(from_dev(hd, basis.ngw, nst) - ref) <= tol * size, flags
    ham.close()
    basis.close()
