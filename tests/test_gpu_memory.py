"""Device memory that a context keeps after a call: the transform workspace up to its cap (one
transform at least) and two blocks of temporaries, each no larger than the cap and 256 MiB."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIB = 1 << 20
SLACK = 32 * MIB  # granularity of the allocations, small blocks the runtime holds on to


@pytest.fixture(scope="module")
def cell(gpu_ctx):
    from qball_amd.workload import make_system
    return make_system(ncell=1, ecut_ry=60.0, nbands=1, seed=51, generate_psi=False)


def kept(cell, call, cap):
    """Bytes a new context holds after the call, which has run on another one on the same stream
    before (code objects, the queue's scratch)."""
    import torch
    from qball_amd import Basis, Context
    r = cell.rods
    for _ in range(2):
        ctx = Context(0, torch.cuda.current_stream().cuda_stream)
        ctx.set_workspace_cap(cap)
        basis = Basis(ctx, True, r["rod_h"], r["rod_k"], r["rod_lmin"], r["rod_size"], cell.np,
                      cell.b)
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        call(basis)
        ctx.sync()
        torch.cuda.synchronize()
        used = before - torch.cuda.mem_get_info()[0]
        basis.close()
        ctx.close()
    return used


@pytest.mark.parametrize("what", ("gram", "current", "density"))
def test_small_cap_bounds_what_is_kept(gpu_ctx, cell, what):
    import torch
    cap, nst = 4 * MIB, 700 if what == "gram" else 1000
    g = torch.Generator(device="cuda")
    g.manual_seed(52)
    psi = torch.randn(2 * cell.ngw * nst, dtype=torch.float64, device="cuda", generator=g)
    occ = np.full(nst, 2.0)
    N = int(np.prod(cell.np))
    out = torch.zeros(3 * N, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()

    def call(basis):
        if what == "gram":
            basis.gram(psi.data_ptr(), basis.ngw, nst)
        elif what == "current":
            basis.current(psi.data_ptr(), basis.ngw, nst, occ, 1.0, cell.omega,
                          j_ptr=out.data_ptr())
        else:
            basis.density(psi.data_ptr(), basis.ngw, nst, occ, 1.0, cell.omega, out.data_ptr())
    # four fields of one band at a time at most: T1 and T2 of each on this grid
    slot = 16 * (int(np.prod(cell.np[1:])) + N)
    assert kept(cell, call, cap) <= 2 * cap + max(cap, 4 * slot) + SLACK


def test_current_of_many_bands_keeps_a_bounded_workspace(gpu_ctx, cell):
    """Four transforms per band, but at most 2 GiB of them at a time, whatever the cap allows."""
    import torch
    nst, g = 700, torch.Generator(device="cuda")
    g.manual_seed(53)
    psi = torch.randn(2 * cell.ngw * nst, dtype=torch.float64, device="cuda", generator=g)
    out = torch.zeros(3 * int(np.prod(cell.np)), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()

    def call(basis):
        basis.current(psi.data_ptr(), basis.ngw, nst, np.full(nst, 2.0), 1.0, cell.omega,
                      j_ptr=out.data_ptr())
    assert kept(cell, call, 64 << 30) <= (2 << 30) + 2 * 256 * MIB + SLACK
