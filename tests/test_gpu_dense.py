"""Γ orthonormalisation at the edges of its blocks (64-wide factorisation blocks, 32 to 128 wide
product tiles, doubling of odd block counts) against the oracle, with padding rows, a small
workspace, and a singular overlap.

Bar: the factor L of these overlaps has a condition number of at most 1e3, each rotated band
sums at most 320 others: 1e3 sqrt(320) 1.1e-16 = 2e-12, taken as 1e-11 like the existing tests.
"""
import numpy as np
import pytest

from helpers import from_dev, rel_err, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cell():
    from qball_amd.workload import make_system
    return make_system(ncell=1, ecut_ry=25.0, nbands=320, seed=41)


@pytest.mark.parametrize("nst", [1, 2, 31, 63, 64, 65, 127, 129, 192, 257, 320])
def test_gram_blocks(gpu_ctx, cell, nst):
    from helpers import make_gpu_basis
    from oracle import hpsi as oh
    c = cell.psi[:, :nst]
    basis = make_gpu_basis(gpu_ctx, cell)
    cd = to_dev(c)
    basis.gram(cd.data_ptr(), basis.ngw, nst)
    gpu_ctx.sync()
    got = from_dev(cd, basis.ngw, nst)
    assert rel_err(got, oh.gram(c, True)) <= 1e-11
    v = got.view(np.float64).reshape(basis.ngw, nst, 2)
    s = 2 * np.einsum("gmc,gnc->mn", v, v) - np.outer(got[0].real, got[0].real)
    assert np.abs(s - np.eye(nst)).max() <= 1e-12
    basis.close()


def test_gram_padding_small_workspace_and_singular(cell):
    import torch
    from oracle import hpsi as oh
    from qball_amd import Basis, Context, QbhError
    ctx = Context(0, None)
    ctx.set_workspace_cap(1.0)
    r = cell.rods
    basis = Basis(ctx, True, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"], cell.np, cell.b)
    nst, ld = 70, cell.ngw + 3
    c = np.zeros((ld, nst), dtype=np.complex128, order="F")
    c[:cell.ngw] = cell.psi[:, :nst]
    c[cell.ngw:] = 7.0
    cd = to_dev(c)
    basis.gram(cd.data_ptr(), ld, nst)
    ctx.sync()
    got = from_dev(cd, ld, nst)
    assert rel_err(got[:cell.ngw], oh.gram(cell.psi[:, :nst], True)) <= 1e-11
    assert (got[cell.ngw:] == 7.0).all()
    c[:, 66] = 0.0  # an empty band: zero pivot
    cd = to_dev(c)
    before = cd.clone()
    torch.cuda.synchronize()
    with pytest.raises(QbhError, match="positive definite"):
        basis.gram(cd.data_ptr(), ld, nst)
    assert torch.equal(cd, before)
    basis.close()
    ctx.close()


@pytest.mark.parametrize("nst,sym,tri", [(385, 32, 64), (640, 128, 128), (768, 64, 128),
                                         (900, 128, 128)])
def test_gram_wide_tiles(gpu_ctx, nst, sym, tri):
    """The 64 and 128 wide tiles of the symmetric and the triangular product over several tile
    rows and slices, with the tiles that ran (same bar: 900 bands, condition of L 11)."""
    from helpers import make_gpu_basis, product_tile
    from oracle import hpsi as oh
    from qball_amd.workload import make_system
    big = make_system(ncell=1, ecut_ry=60.0, nbands=nst, seed=41)
    K = 2 * big.ngw
    assert product_tile(4, nst, nst, K)[0] == sym and product_tile(2, nst, K, nst)[0] == tri
    basis = make_gpu_basis(gpu_ctx, big)
    cd = to_dev(big.psi)
    basis.gram(cd.data_ptr(), basis.ngw, nst)
    gpu_ctx.sync()
    got = from_dev(cd, basis.ngw, nst)
    assert rel_err(got, oh.gram(big.psi, True)) <= 1e-11
    basis.close()


@pytest.mark.parametrize("nst", [1, 16, 70, 129])
def test_gram_of_bands_at_an_odd_double(gpu_ctx, cell, nst):
    """A psi aligned to 8 bytes only, which the matrix-core products do not read (rocBLAS and
    rocSOLVER): the same bands."""
    import torch
    from helpers import make_gpu_basis
    from oracle import hpsi as oh
    c = cell.psi[:, :nst]
    basis = make_gpu_basis(gpu_ctx, cell)
    buf = torch.zeros(2 * cell.ngw * nst + 1, dtype=torch.float64, device="cuda")
    buf[1:] = to_dev(c)
    assert buf[1:].data_ptr() % 16 == 8
    torch.cuda.synchronize()
    basis.gram(buf[1:].data_ptr(), basis.ngw, nst)
    gpu_ctx.sync()
    assert rel_err(from_dev(buf[1:].contiguous(), basis.ngw, nst), oh.gram(c, True)) <= 1e-11
    basis.close()
