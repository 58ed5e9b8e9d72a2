"""Calls of the C ABI made from inside an enrolled boundary: every stage of a cycle calls it,
between the kernels that reduce the cycle's time step and hand it to the host."""
import pytest

from idefix_amd import problems

pytestmark = pytest.mark.gpu


def _block(dim, n, mhd, nstages, calls):
    from idefix_amd.datablock import DataBlock
    g = DataBlock(dim, n, mhd=mhd, recon="plm", solver="hlld" if mhd else "hllc", cfl=0.3, cfl_max_var=1e6,
                  bc=[("userdef", "outflow")] + ["periodic"] * (dim - 1), nstages=nstages, first_dt=1e-5)
    g.upload(*(problems.random_mhd if mhd else problems.random_hd)(g))
    b = g.beg[0]

    def fill(d, side, t, Vc, Vs):
        Vc[..., :b] = Vc[..., b:b + 1]
        if Vs is not None:
            Vs[1:, ..., :b] = Vs[1:, ..., b:b + 1]
        for name in calls:
            getattr(g, name)()
    g.set_userdef_boundary(fill)
    return g


@pytest.mark.parametrize("nstages", [1, 2, 3])
@pytest.mark.parametrize("dim,n,mhd", [(1, (70,), False), (2, (20, 12), False), (2, (20, 12), True), (3, (12, 7, 9), True)])
def test_time_step_of_a_boundary_that_computes_it(dim, n, mhd, nstages):
    """A boundary that calls ComputeTimestep in the first of two cycles leaves the cycles' own time
    steps as they are, also where the second one's signals are slower than those it saw."""
    import torch
    a = _block(dim, n, mhd, nstages, [])
    calls = []
    b = _block(dim, n, mhd, nstages, calls)
    prs = 1 + dim
    for q in range(4):
        calls[:] = ["compute_timestep"] if q % 2 == 0 else []
        a.cycle()
        b.cycle()
        assert a.dt == b.dt
        for g in (a, b):
            g.Vc[1:prs + 1] *= 0.25  # velocities and pressure
    assert torch.equal(a.interior(a.Vc), b.interior(b.Vc))


@pytest.mark.parametrize("nstages", [2, 3])
def test_time_step_of_a_boundary_that_checks_divb(nstages):
    """Nor does CheckDivB, whose result comes back through the same pinned block, change them."""
    a = _block(2, (20, 12), True, nstages, [])
    b = _block(2, (20, 12), True, nstages, ["check_divb", "compute_timestep", "check_divb"])
    for _ in range(3):
        a.cycle()
        b.cycle()
        assert a.dt == b.dt
