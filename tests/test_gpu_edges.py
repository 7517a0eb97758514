"""Transforms at every kind of grid edge with a register transform, each edge along each axis,
with the sphere at about half the edge and filling it: backward, forward, local Hψ and density
against the oracle.  FP64 relative 2-norm <= 1e-12; FP32 2e-6 (float rounding of log2(n)
butterfly stages both ways)."""
import numpy as np
import pytest

from helpers import from_dev, real_to_dev, rel_err, to_dev

pytestmark = pytest.mark.gpu

EDGES = (18, 20, 24, 30, 42, 44, 56, 66, 70, 84, 88, 110, 112, 126, 132, 150, 154, 176)
GRIDS = [(EDGES[i], EDGES[(i + 6) % 18], EDGES[(i + 12) % 18]) for i in range(18)]


@pytest.mark.parametrize("grid,nb,real", [(g, 2 * (i % 3) + 1, i % 4 != 3)
                                          for i, g in enumerate(GRIDS)])
def test_register_edges(gpu_ctx, grid, nb, real):
    import torch
    from oracle import fft as offt
    from oracle import hpsi as oh
    from oracle.basis import Basis as OB, FFTMaps, UnitCell
    from qball_amd import Basis, Hamiltonian
    from qball_amd.workload import make_system
    sysm = make_system(ncell=1, ecut_ry=25.0, nbands=nb, seed=21, complex_basis=not real)
    maps = FFTMaps(OB(UnitCell(sysm.a), sysm.ecut, force_complex=not real), *grid)
    r = sysm.rods
    basis = Basis(gpu_ctx, real, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"], grid, sysm.b)
    N, c = basis.N, sysm.psi
    cd = to_dev(c)
    nslots = (nb + 1) // 2 if real else nb
    f = torch.zeros(2 * nslots * N, dtype=torch.float64, device="cuda")
    basis.backward(cd.data_ptr(), basis.ngw, nb, real, f.data_ptr())
    back = torch.zeros_like(cd)
    rng = np.random.default_rng(22)
    g = rng.standard_normal((nslots, N)) + 1j * rng.standard_normal((nslots, N))
    gd = torch.from_numpy(g.view(np.float64).ravel().copy()).cuda()
    torch.cuda.synchronize()
    basis.forward(gd.data_ptr(), nb, real, back.data_ptr(), basis.ngw)
    gpu_ctx.sync()
    fg = f.cpu().numpy().view(np.complex128).reshape(nslots, N)
    bg = from_dev(back, basis.ngw, nb)
    for s in range(nslots):
        gs = g[s].reshape(maps.np2, maps.np1, maps.np0)
        if real:
            two = 2 * s + 1 < nb
            ref = offt.backward(maps, c[:, 2 * s], c[:, 2 * s + 1] if two else None)
            c1, c2 = offt.forward(maps, gs, pair=True)
            assert rel_err(bg[:, 2 * s], c1) <= 1e-12
            if two:
                assert rel_err(bg[:, 2 * s + 1], c2) <= 1e-12
        else:
            ref = offt.backward(maps, c[:, s])
            assert rel_err(bg[:, s], offt.forward(maps, gs)) <= 1e-12
        assert rel_err(fg[s], ref.ravel()) <= 1e-12
    v = rng.standard_normal(N)
    vd = real_to_dev(v)
    ham = Hamiltonian(gpu_ctx, basis)
    ham.set_vloc(vd.data_ptr())
    hd = torch.zeros_like(cd)
    ref = oh.rs_mul_add(maps, c, v, np.zeros_like(c))
    for flags, tol in ((0x4, 1e-12), (0x14, 2e-6)):
        ham.hpsi(cd.data_ptr(), basis.ngw, nb, sysm.occ, hd.data_ptr(), basis.ngw, flags=flags)
        gpu_ctx.sync()
        assert rel_err(from_dev(hd, basis.ngw, nb), ref) <= tol
    rho = torch.zeros(N, dtype=torch.float64, device="cuda")
    basis.density(cd.data_ptr(), basis.ngw, nb, sysm.occ, 1.0, sysm.omega, rho.data_ptr())
    gpu_ctx.sync()
    assert rel_err(rho.cpu().numpy(),
                   oh.compute_density(maps, c, sysm.occ, 1.0, sysm.omega)) <= 1e-12
    ham.close()
    basis.close()


@pytest.mark.parametrize("grid", [(18, 20, 30), (40, 64, 36), (60, 72, 42), (88, 90, 50),
                                  (110, 24, 144), (140, 66, 28), (256, 20, 18), (162, 30, 22)])
@pytest.mark.parametrize("flags,tol", [(0, 1e-12), (0x10, 2e-6)])
def test_forward_from_grid(gpu_ctx, grid, flags, tol):
    """forward (Γ pairs with a lone last band, and single bands) and forward_real at short,
    long and Stockham x edges, row counts that leave the last workgroup part empty."""
    import torch
    from oracle import fft as offt
    from oracle.basis import Basis as OB, FFTMaps, UnitCell
    from qball_amd import Basis
    from qball_amd.workload import make_system
    sysm = make_system(ncell=1, ecut_ry=25.0, nbands=5, seed=23, generate_psi=False)
    maps = FFTMaps(OB(UnitCell(sysm.a), sysm.ecut), *grid)
    r = sysm.rods
    basis = Basis(gpu_ctx, True, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"], grid, sysm.b)
    rng = np.random.default_rng(24)
    g = rng.standard_normal((3, basis.N)) + 1j * rng.standard_normal((3, basis.N))
    gd = torch.from_numpy(g.view(np.float64).ravel().copy()).cuda()
    out = torch.zeros(2 * basis.ngw * 5, dtype=torch.float64, device="cuda")
    shape = (maps.np2, maps.np1, maps.np0)
    for nb, pair in ((5, True), (3, False)):
        basis.forward(gd.data_ptr(), nb, pair, out.data_ptr(), basis.ngw, flags)
        gpu_ctx.sync()
        got = from_dev(out[:2 * basis.ngw * nb], basis.ngw, nb)
        for s in range(3):
            ref = offt.forward(maps, g[s].reshape(shape), pair=pair)
            ref = ref if pair else (ref,)
            for j, c in enumerate(ref):
                if (2 if pair else 1) * s + j < nb:
                    assert rel_err(got[:, (2 if pair else 1) * s + j], c) <= tol
    rho = rng.standard_normal(basis.N)
    rd = real_to_dev(rho)
    basis.forward_real(rd.data_ptr(), 2.5, out.data_ptr(), flags)
    gpu_ctx.sync()
    ref = offt.forward(maps, (2.5 * rho).astype(np.complex128).reshape(shape))
    assert rel_err(from_dev(out[:2 * basis.ngw], basis.ngw, 1)[:, 0], ref) <= tol
    basis.close()


@pytest.mark.parametrize("real,nb", [(True, 15), (True, 16), (True, 45), (False, 9), (False, 23)])
@pytest.mark.parametrize("grid", [(36, 40, 42), (22, 24, 18)])
def test_density_slot_ranges(real, nb, grid):
    """Density summed over slot ranges (counts that do not divide into them, lone last band,
    empty bands), in one chunk and in chunks too small for ranges, added to what rho holds."""
    import torch
    from oracle import hpsi as oh
    from oracle.basis import Basis as OB, FFTMaps, UnitCell
    from qball_amd import Basis, Context
    from qball_amd.workload import make_system
    sysm = make_system(ncell=1, ecut_ry=25.0, nbands=nb, seed=25, complex_basis=not real)
    maps = FFTMaps(OB(UnitCell(sysm.a), sysm.ecut, force_complex=not real), *grid)
    occ = np.where(np.arange(nb) % 5 == 3, 0.0, 1.0 + 0.1 * np.arange(nb))
    ref = oh.compute_density(maps, sysm.psi, occ, 1.0, sysm.omega)
    rng = np.random.default_rng(26)
    r = sysm.rods
    cd = to_dev(sysm.psi)
    for cap in (8 << 30, 1 << 20):
        ctx = Context(0, None)
        ctx.set_workspace_cap(cap)
        basis = Basis(ctx, real, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"], grid, sysm.b)
        start = rng.standard_normal(basis.N)
        for flags, tol in ((0, 1e-12), (0x10, 2e-6)):
            rho = real_to_dev(start)
            torch.cuda.synchronize()
            basis.density(cd.data_ptr(), basis.ngw, nb, occ, 1.0, sysm.omega, rho.data_ptr(), flags)
            ctx.sync()
            assert rel_err(rho.cpu().numpy() - start, ref) <= tol * 10  # start is ~10x ref
        basis.close()
        ctx.close()


@pytest.mark.parametrize("real,nb", [(False, 1), (False, 7), (False, 26), (True, 5)])
@pytest.mark.parametrize("grid", [(24, 36, 30), (44, 18, 40), (64, 42, 20), (72, 20, 36),
                                  (140, 24, 18), (22, 24, 18)])
def test_current_edges(real, nb, grid):
    """The current density (band sums of products of transforms), bands with no weight among
    them, in one chunk and in chunks of a few bands, against the oracle's transforms."""
    import torch
    from oracle import fft as offt
    from oracle.basis import Basis as OB, FFTMaps, UnitCell
    from qball_amd import Basis, Context
    from qball_amd.workload import make_system
    sysm = make_system(ncell=1, ecut_ry=25.0, nbands=nb, seed=27, complex_basis=not real)
    maps = FFTMaps(OB(UnitCell(sysm.a), sysm.ecut, force_complex=not real), *grid)
    occ = np.where(np.arange(nb) % 4 == 2, 0.0, 1.0 + 0.05 * np.arange(nb))
    ref = np.zeros((3, int(np.prod(grid))))
    size = np.zeros(3)
    for n in range(nb):
        f0 = offt.backward(maps, sysm.psi[:, n]).ravel()
        for d in range(3):
            fd = offt.backward(maps, 1j * sysm.kpg[:, d] * sysm.psi[:, n]).ravel()
            ref[d] -= occ[n] / sysm.omega * (np.conj(f0) * fd).imag
            size[d] += occ[n] / sysm.omega * np.linalg.norm(np.abs(f0) * np.abs(fd))
    r = sysm.rods
    cd = to_dev(sysm.psi)
    for cap in (8 << 30, 4 << 20):
        ctx = Context(0, None)
        ctx.set_workspace_cap(cap)
        basis = Basis(ctx, real, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"], grid, sysm.b)
        j = torch.full((3, basis.N), np.nan, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        total = basis.current(cd.data_ptr(), basis.ngw, nb, occ, 1.0, sysm.omega,
                              j_ptr=j.data_ptr())
        ctx.sync()
        got = j.cpu().numpy()
        for d in range(3):
            assert np.linalg.norm(got[d] - ref[d]) <= 1e-13 * size[d]
            assert abs(total[d] - sysm.omega / basis.N * ref[d].sum()) <= \
                1e-13 * sysm.omega / basis.N * size[d] * np.sqrt(basis.N)
        basis.close()
        ctx.close()


@pytest.mark.parametrize("n", (18, 20, 24, 30, 42, 44, 56, 66, 70, 84, 88, 110, 112, 132, 154,
                               176))
@pytest.mark.parametrize("real", (True, False))
def test_fp32_stockham_order(gpu_ctx, n, real):
    """FP32 register transforms that keep the Stockham passes' radix order round like them:
    backward, forward and local Hψ bit for bit, the edge along each axis."""
    import torch
    from qball_amd import Basis, Hamiltonian
    from qball_amd.workload import make_system
    nb = 3
    sysm = make_system(ncell=1, ecut_ry=12.0, nbands=nb, seed=31, complex_basis=not real)
    r, cd = sysm.rods, to_dev(sysm.psi)
    nslots = (nb + 1) // 2 if real else nb
    rng = np.random.default_rng(n)
    for axis in range(3):
        grid = [22, 22, 22]  # (no register form)
        grid[axis] = n
        basis = Basis(gpu_ctx, real, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"], grid,
                      sysm.b)
        vd = real_to_dev(rng.standard_normal(basis.N))
        gd = real_to_dev(rng.standard_normal(2 * nslots * basis.N))
        ham = Hamiltonian(gpu_ctx, basis)
        ham.set_vloc(vd.data_ptr())
        out = []
        for reg in (1, 0):
            ham.set_tuning("zy_reg", reg)
            ham.set_tuning("x_reg", reg)
            f = torch.zeros(2 * nslots * basis.N, dtype=torch.float64, device="cuda")
            hd, back = torch.zeros_like(cd), torch.zeros_like(cd)
            torch.cuda.synchronize()
            basis.backward(cd.data_ptr(), basis.ngw, nb, real, f.data_ptr(), 0x10)
            basis.forward(gd.data_ptr(), nb, real, back.data_ptr(), basis.ngw, 0x10)
            ham.hpsi(cd.data_ptr(), basis.ngw, nb, sysm.occ, hd.data_ptr(), basis.ngw, flags=0x14)
            gpu_ctx.sync()
            out.append((f, back, hd))
        for a, b in zip(*out):
            assert torch.equal(a, b)
        ham.close()
        basis.close()


@pytest.mark.parametrize("n,np2,ecut,nb,real", [
    (18, 20, 12.0, 1, True), (20, 18, 25.0, 3, False), (36, 30, 25.0, 6, True),
    (44, 24, 25.0, 2, False), (48, 50, 170.0, 2, True), (60, 22, 25.0, 5, True),
    (64, 30, 60.0, 3, False), (72, 36, 60.0, 67, True), (80, 20, 25.0, 4, False),
    (84, 20, 25.0, 3, True), (88, 28, 60.0, 2, False), (108, 20, 25.0, 4, True)])
def test_plane_vmul(gpu_ctx, n, np2, ecut, nb, real):
    """Local Hψ on square cross-sections, whose y, x and y passes are one kernel: with one and
    several slots per workgroup, the two workgroup sizes, spheres filling the plane (more
    columns than are loaded ahead) and partly filled last row groups."""
    import torch
    from oracle import hpsi as oh
    from oracle.basis import Basis as OB, FFTMaps, UnitCell
    from qball_amd import Basis, Hamiltonian
    from qball_amd.workload import make_system
    sysm = make_system(ncell=1, ecut_ry=ecut, nbands=nb, seed=41, complex_basis=not real)
    maps = FFTMaps(OB(UnitCell(sysm.a), sysm.ecut, force_complex=not real), n, n, np2)
    r, c = sysm.rods, sysm.psi
    basis = Basis(gpu_ctx, real, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"],
                  (n, n, np2), sysm.b)
    v = np.random.default_rng(n).standard_normal(basis.N)
    vd, cd = real_to_dev(v), to_dev(c)
    hd = torch.zeros_like(cd)
    ham = Hamiltonian(gpu_ctx, basis)
    ham.set_vloc(vd.data_ptr())
    gpu_ctx.timing_report()
    gpu_ctx.set_timing(True)
    ham.hpsi(cd.data_ptr(), basis.ngw, nb, sysm.occ, hd.data_ptr(), basis.ngw, flags=0x4)
    gpu_ctx.sync()
    ran = gpu_ctx.timing_report()
    gpu_ctx.set_timing(False)
    assert "plane_vmul" in ran
    ref = oh.rs_mul_add(maps, c, v, np.zeros_like(c))
    assert rel_err(from_dev(hd, basis.ngw, nb), ref) <= 1e-12
    ham.close()
    basis.close()


@pytest.mark.parametrize("n,np2,ecut,nb,real", [
    (18, 20, 12.0, 1, True), (28, 18, 25.0, 3, False), (40, 30, 25.0, 7, True),
    (48, 50, 170.0, 3, True), (64, 30, 60.0, 66, False), (72, 36, 60.0, 37, True),
    (80, 20, 25.0, 4, False), (90, 20, 25.0, 3, True), (100, 28, 60.0, 2, False)])
def test_plane_grids(gpu_ctx, n, np2, ecut, nb, real):
    """Grid transforms and density on square cross-sections (y and x pass in one kernel): one
    and several slots per workgroup and slot ranges, added to what the density grid holds."""
    import torch
    from oracle import fft as offt
    from oracle import hpsi as oh
    from oracle.basis import Basis as OB, FFTMaps, UnitCell
    from qball_amd import Basis
    from qball_amd.workload import make_system
    sysm = make_system(ncell=1, ecut_ry=ecut, nbands=nb, seed=43, complex_basis=not real)
    maps = FFTMaps(OB(UnitCell(sysm.a), sysm.ecut, force_complex=not real), n, n, np2)
    r, c = sysm.rods, sysm.psi
    basis = Basis(gpu_ctx, real, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"],
                  (n, n, np2), sysm.b)
    N, cd = basis.N, to_dev(c)
    rng = np.random.default_rng(n)
    nslots = (nb + 1) // 2 if real else nb
    f = torch.zeros(2 * nslots * N, dtype=torch.float64, device="cuda")
    g = rng.standard_normal((nslots, N)) + 1j * rng.standard_normal((nslots, N))
    gd = torch.from_numpy(g.view(np.float64).ravel().copy()).cuda()
    h = rng.standard_normal(N)
    hd, rho0 = real_to_dev(h), rng.standard_normal(N)
    rho = real_to_dev(rho0)
    back, one = torch.zeros_like(cd), torch.zeros(2 * basis.ngw, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    gpu_ctx.timing_report()
    gpu_ctx.set_timing(True)
    basis.backward(cd.data_ptr(), basis.ngw, nb, real, f.data_ptr())
    basis.forward(gd.data_ptr(), nb, real, back.data_ptr(), basis.ngw)
    basis.forward_real(hd.data_ptr(), 0.7, one.data_ptr())
    basis.density(cd.data_ptr(), basis.ngw, nb, sysm.occ, 1.0, sysm.omega, rho.data_ptr())
    gpu_ctx.sync()
    ran = gpu_ctx.timing_report()
    gpu_ctx.set_timing(False)
    assert "plane_density" in ran
    assert ({"plane_store", "plane_load"} <= set(ran)) == (n <= 64)
    fg = f.cpu().numpy().view(np.complex128).reshape(nslots, N)
    bg = from_dev(back, basis.ngw, nb)
    shape = (np2, n, n)
    for s in range(nslots):
        if real:
            two = 2 * s + 1 < nb
            ref = offt.backward(maps, c[:, 2 * s], c[:, 2 * s + 1] if two else None)
            c1, c2 = offt.forward(maps, g[s].reshape(shape), pair=True)
            assert rel_err(bg[:, 2 * s], c1) <= 1e-12
            if two:
                assert rel_err(bg[:, 2 * s + 1], c2) <= 1e-12
        else:
            ref = offt.backward(maps, c[:, s])
            assert rel_err(bg[:, s], offt.forward(maps, g[s].reshape(shape))) <= 1e-12
        assert rel_err(fg[s], ref.ravel()) <= 1e-12
    assert rel_err(from_dev(one, basis.ngw, 1)[:, 0],
                   offt.forward(maps, 0.7 * h.reshape(shape))) <= 1e-12
    ref = rho0 + oh.compute_density(maps, c, sysm.occ, 1.0, sysm.omega)
    assert rel_err(rho.cpu().numpy(), ref) <= 1e-12
    basis.close()


@pytest.mark.parametrize("real", (True, False))
@pytest.mark.parametrize("grid", [(24, 36, 30), (72, 20, 36), (140, 24, 18), (22, 24, 18)])
@pytest.mark.parametrize("occ", [(0, 2, 2, 0, 0, 1, 2, 0), (2, 0, 0, 0, 0, 0, 0, 0),
                                 (0, 0, 0, 0, 0, 0, 0, 1), (0, 0, 0, 0, 0, 0, 0, 0)])
def test_current_leaves_out_empty_bands(gpu_ctx, real, grid, occ):
    """Bands without a positive weight do not enter the current, whatever they hold: NaN and
    infinities in them leave its bits as they are with zeros there.  Grids with and without a
    register x transform."""
    import torch
    from qball_amd import Basis
    from qball_amd.workload import make_system
    nb, occ = len(occ), np.array(occ, dtype=np.float64)
    sysm = make_system(ncell=1, ecut_ry=25.0, nbands=nb, seed=28, complex_basis=not real)
    r = sysm.rods
    basis = Basis(gpu_ctx, real, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"], grid, sysm.b)
    out = []
    for fill in (0.0, np.nan, np.inf):
        c = sysm.psi.copy()
        c[:, occ == 0.0] = fill
        cd = to_dev(c)
        j = torch.full((3, basis.N), np.nan, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        total = basis.current(cd.data_ptr(), basis.ngw, nb, occ, 1.0, sysm.omega,
                              j_ptr=j.data_ptr())
        gpu_ctx.sync()
        out.append((j.cpu().numpy(), np.array(total)))
    assert np.isfinite(out[0][0]).all() and (real or occ.any() == out[0][0].any())
    for j, total in out[1:]:
        assert np.array_equal(j, out[0][0]) and np.array_equal(total, out[0][1])
    basis.close()


@pytest.mark.parametrize("n", (28, 32, 36, 40, 48, 50, 54, 60, 64, 72, 80, 90, 96, 100, 108, 120,
                               128, 140, 144, 160, 168, 180, 192, 210, 224, 240, 256))
def test_fp32_forward_error(gpu_ctx, n):
    """FP32 forward transforms from complex and real grids are as close to the 64-bit ones with
    the register x pass as with the Stockham one.  Both read tabled twiddles, so their errors
    have the same size, found here from at least 8 x 1151 coefficients to about 0.7 %; the bar
    is 2 %."""
    import torch
    from oracle import fft as offt
    from oracle.basis import Basis as OB, FFTMaps, UnitCell
    from qball_amd import Basis, Hamiltonian
    from qball_amd.workload import make_system
    sysm = make_system(ncell=1, ecut_ry=25.0, nbands=1, seed=23, generate_psi=False)
    grid, shape, m = (n, 22, 22), (22, 22, n), 8
    maps = FFTMaps(OB(UnitCell(sysm.a), sysm.ecut), *grid)
    r = sysm.rods
    basis = Basis(gpu_ctx, True, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"], grid, sysm.b)
    ham = Hamiltonian(gpu_ctx, basis)  # (holds the basis' tuning)
    rng = np.random.default_rng(n)
    g = rng.standard_normal((m, basis.N)) + 1j * rng.standard_normal((m, basis.N))
    rho = rng.standard_normal((2 * m, basis.N))
    ref = [offt.forward(maps, x.reshape(shape)).ravel() for x in g]
    ref_real = [offt.forward(maps, x.astype(np.complex128).reshape(shape)).ravel() for x in rho]
    gd, rd = real_to_dev(g.view(np.float64).ravel()), real_to_dev(rho.ravel())
    err = {}
    for reg in (1, 0):
        ham.set_tuning("x_reg", reg)
        out = torch.zeros((m, 2 * basis.ngw), dtype=torch.float64, device="cuda")
        real = torch.zeros((2 * m, 2 * basis.ngw), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        basis.forward(gd.data_ptr(), m, False, out.data_ptr(), basis.ngw, 0x10)
        for k in range(2 * m):
            basis.forward_real(rd[k * basis.N:].data_ptr(), 1.0, real[k].data_ptr(), 0x10)
        gpu_ctx.sync()
        err[reg] = (rel_err(out.cpu().numpy().view(np.complex128), ref),
                    rel_err(real.cpu().numpy().view(np.complex128), ref_real))
    for k in range(2):
        assert err[1][k] <= 1.02 * err[0][k], err
    ham.close()
    basis.close()


@pytest.mark.parametrize("nb,vmul,store,load,density", [
    (1, False, False, False, False), (3, False, False, False, False), (8, True, True, True, True)])
@pytest.mark.parametrize("n", (54, 56))
def test_plane_needs_enough_planes(gpu_ctx, n, nb, vmul, store, load, density):
    """A sphere that fills most of the plane (nlx = 43): few slots take the passes, which spread
    one slot over the chip, more take the plane kernel; the oracle's results either way."""
    import torch
    from oracle import fft as offt
    from oracle import hpsi as oh
    from oracle.basis import Basis as OB, FFTMaps, UnitCell
    from qball_amd import Basis, Hamiltonian
    from qball_amd.workload import make_system
    sysm = make_system(ncell=1, ecut_ry=170.0, nbands=nb, seed=47)
    maps = FFTMaps(OB(UnitCell(sysm.a), sysm.ecut), n, n, 50)
    r, c = sysm.rods, sysm.psi
    basis = Basis(gpu_ctx, True, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"], (n, n, 50),
                  sysm.b)
    N, cd, nslots = basis.N, to_dev(c), (nb + 1) // 2
    rng = np.random.default_rng(n)
    v = rng.standard_normal(N)
    vd, hd, back = real_to_dev(v), torch.zeros_like(cd), torch.zeros_like(cd)
    f = torch.zeros(2 * nslots * N, dtype=torch.float64, device="cuda")
    rho = torch.zeros(N, dtype=torch.float64, device="cuda")
    ham = Hamiltonian(gpu_ctx, basis)
    ham.set_vloc(vd.data_ptr())
    torch.cuda.synchronize()
    gpu_ctx.timing_report()
    gpu_ctx.set_timing(True)
    ham.hpsi(cd.data_ptr(), basis.ngw, nb, sysm.occ, hd.data_ptr(), basis.ngw, flags=0x4)
    basis.backward(cd.data_ptr(), basis.ngw, nb, True, f.data_ptr())
    basis.forward(f.data_ptr(), nb, True, back.data_ptr(), basis.ngw)
    basis.density(cd.data_ptr(), basis.ngw, nb, sysm.occ, 1.0, sysm.omega, rho.data_ptr())
    gpu_ctx.sync()
    ran = gpu_ctx.timing_report()
    gpu_ctx.set_timing(False)
    assert ["plane_" + k in ran for k in ("vmul", "store", "load", "density")] == \
        [vmul, store, load, density]
    ref = oh.rs_mul_add(maps, c, v, np.zeros_like(c))
    assert rel_err(from_dev(hd, basis.ngw, nb), ref) <= 1e-12
    fg = f.cpu().numpy().view(np.complex128).reshape(nslots, N)
    for s in range(nslots):
        two = 2 * s + 1 < nb
        ref = offt.backward(maps, c[:, 2 * s], c[:, 2 * s + 1] if two else None)
        assert rel_err(fg[s], ref.ravel()) <= 1e-12
    assert rel_err(from_dev(back, basis.ngw, nb), c) <= 1e-12
    assert rel_err(rho.cpu().numpy(),
                   oh.compute_density(maps, c, sysm.occ, 1.0, sysm.omega)) <= 1e-12
    ham.close()
    basis.close()


@pytest.mark.parametrize("grid,ecut,nlx,real,nb", [
    ((32, 18, 24), 25.0, 17, True, 3), ((36, 30, 28), 60.0, 25, False, 2),
    ((72, 50, 44), 170.0, 43, True, 2), ((128, 66, 70), 395.0, 65, True, 3)])
def test_spheres_just_past_half_the_edge(gpu_ctx, grid, ecut, nlx, real, nb):
    """Local Hψ and density of spheres of a few lines more than half the edge (the x pass'
    middle count of line elements), long and short edges."""
    import torch
    from oracle import hpsi as oh
    from oracle.basis import Basis as OB, FFTMaps, UnitCell
    from qball_amd import Basis, Hamiltonian
    from qball_amd.workload import make_system
    sysm = make_system(ncell=1, ecut_ry=ecut, nbands=nb, seed=48, complex_basis=not real)
    maps = FFTMaps(OB(UnitCell(sysm.a), sysm.ecut, force_complex=not real), *grid)
    assert 2 * int(np.abs(sysm.idx[:, 0]).max()) + 1 == nlx and grid[0] < 2 * nlx < grid[0] + 18
    r, c = sysm.rods, sysm.psi
    basis = Basis(gpu_ctx, real, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"], grid, sysm.b)
    v = np.random.default_rng(nlx).standard_normal(basis.N)
    vd, cd = real_to_dev(v), to_dev(c)
    hd = torch.zeros_like(cd)
    ham = Hamiltonian(gpu_ctx, basis)
    ham.set_vloc(vd.data_ptr())
    ref = oh.rs_mul_add(maps, c, v, np.zeros_like(c))
    rho_ref = oh.compute_density(maps, c, sysm.occ, 1.0, sysm.omega)
    for flags, tol in ((0, 1e-12), (0x10, 2e-6)):
        rho = torch.zeros(basis.N, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        ham.hpsi(cd.data_ptr(), basis.ngw, nb, sysm.occ, hd.data_ptr(), basis.ngw,
                 flags=0x4 | flags)
        basis.density(cd.data_ptr(), basis.ngw, nb, sysm.occ, 1.0, sysm.omega, rho.data_ptr(),
                      flags)
        gpu_ctx.sync()
        assert rel_err(from_dev(hd, basis.ngw, nb), ref) <= tol
        assert rel_err(rho.cpu().numpy(), rho_ref) <= tol
    ham.close()
    basis.close()


@pytest.mark.parametrize("n,np2,ecut,nb,real", [
    (24, 18, 12.0, 3, True), (28, 20, 25.0, 2, False), (30, 24, 25.0, 5, True),
    (32, 18, 25.0, 4, False), (42, 20, 25.0, 7, True), (50, 28, 60.0, 3, False),
    (54, 20, 25.0, 5, True), (56, 30, 60.0, 2, False), (66, 24, 25.0, 3, True),
    (70, 20, 25.0, 4, False), (90, 18, 25.0, 5, True), (96, 30, 60.0, 2, False),
    (100, 24, 25.0, 3, True)])
def test_plane_every_edge(gpu_ctx, n, np2, ecut, nb, real):
    """Local Hψ and density in the plane kernel at the edges the tests above leave out (each is
    an instantiation with its own rows, padding and wavefronts)."""
    import torch
    from oracle import hpsi as oh
    from oracle.basis import Basis as OB, FFTMaps, UnitCell
    from qball_amd import Basis, Hamiltonian
    from qball_amd.workload import make_system
    sysm = make_system(ncell=1, ecut_ry=ecut, nbands=nb, seed=49, complex_basis=not real)
    maps = FFTMaps(OB(UnitCell(sysm.a), sysm.ecut, force_complex=not real), n, n, np2)
    r, c = sysm.rods, sysm.psi
    basis = Basis(gpu_ctx, real, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"],
                  (n, n, np2), sysm.b)
    v = np.random.default_rng(n).standard_normal(basis.N)
    vd, cd = real_to_dev(v), to_dev(c)
    hd = torch.zeros_like(cd)
    rho = torch.zeros(basis.N, dtype=torch.float64, device="cuda")
    ham = Hamiltonian(gpu_ctx, basis)
    ham.set_vloc(vd.data_ptr())
    torch.cuda.synchronize()
    gpu_ctx.timing_report()
    gpu_ctx.set_timing(True)
    ham.hpsi(cd.data_ptr(), basis.ngw, nb, sysm.occ, hd.data_ptr(), basis.ngw, flags=0x4)
    basis.density(cd.data_ptr(), basis.ngw, nb, sysm.occ, 1.0, sysm.omega, rho.data_ptr())
    gpu_ctx.sync()
    ran = gpu_ctx.timing_report()
    gpu_ctx.set_timing(False)
    assert {"plane_vmul", "plane_density"} <= set(ran)
    ref = oh.rs_mul_add(maps, c, v, np.zeros_like(c))
    assert rel_err(from_dev(hd, basis.ngw, nb), ref) <= 1e-12
    assert rel_err(rho.cpu().numpy(),
                   oh.compute_density(maps, c, sysm.occ, 1.0, sysm.omega)) <= 1e-12
    ham.close()
    basis.close()
