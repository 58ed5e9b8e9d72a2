"""idfx_cycle's schedules (idfx_ctx_set_fusion): switching between them, and what they leave in
the caller's arrays."""
import pytest

from idefix_amd import problems
from tests.pairs import cfg_kwargs, interior_faces, make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nstages,bc", [((70,), 2, "outflow"), ((70,), 3, "periodic"), ((20, 9), 2, "reflective"),
                                          ((12, 7, 9), 3, "outflow")])
def test_hydro_schedule_switches_both_ways(n, nstages, bc):
    """Hydro takes levels 0, 1 and 2 in any order, a cycle at each: every bit of the state and
    the time step as at level 0 throughout."""
    import torch
    kw = cfg_kwargs(len(n), n, mhd=False, solver="hllc", recon="plm", bc=bc, gamma=1.4, cfl=0.3,
                    nstages=nstages)
    _, g = make_pair(kw, problems.random_hd)
    _, h = make_pair(kw, problems.random_hd)
    h.set_fusion(0)
    for level in (0, 1, 2, 0, 2, 1):
        g.set_fusion(level)
        g.cycle()
        h.cycle()
        assert g.dt == h.dt
        assert torch.equal(g.interior(g.Vc), h.interior(h.Vc))
        assert torch.equal(g.interior(g.Uc), h.interior(h.Uc))


@pytest.mark.parametrize("kw", [dict(dim=1, nx=(40,), comps=2), dict(dim=2, nx=(20, 9), mhd=False, solver="hllc", ntracer=1),
                                dict(dim=1, nx=(40,), mhd=False, solver="roe")])
def test_levels_without_a_schedule_are_refused(kw):
    """1-D MHD, hydro with tracers and the 1-D Roe hydro solver have level 0 only."""
    from idefix_amd.datablock import DataBlock
    g = DataBlock(**kw)
    g.set_fusion(0)
    for level in (1, 2):
        with pytest.raises(Exception):
            g.set_fusion(level)


SHORT = [(2, (2, 9), False, "reflective"), (2, (2, 9), True, "reflective"),
         (2, (9, 2), True, ["outflow", ("reflective", "outflow")]), (2, (1, 8), False, [("outflow", "reflective"), "periodic"]),
         (3, (66, 3, 2), False, ["outflow", "periodic", "reflective"]), (3, (5, 2, 7), True, "reflective"),
         (3, (66, 3, 2), True, ["outflow", "periodic", "reflective"])]


@pytest.mark.parametrize("dim,n,mhd,bc", SHORT)
def test_reflection_in_a_direction_shorter_than_its_ghost_zone(dim, n, mhd, bc):
    """The left side mirrors ghost cells of the right one as the last fill left them, the right
    side those of the left one, just filled: every bit of cells and faces, over three fills,
    as the oracle fills side by side in one array."""
    import numpy as np
    kw = cfg_kwargs(dim, n, mhd=mhd, solver="hlld" if mhd else "hllc", recon="ppm", bc=bc, gamma=1.4)
    o, g = make_pair(kw, problems.random_mhd if mhd else problems.random_hd)
    for _ in range(3):
        o.set_boundaries()
        g.set_boundaries()
        Vc, Vs = g.download()
        assert np.array_equal(Vc, o.Vc)
        assert not mhd or np.array_equal(Vs, o.Vs)
        # other values inside, exact in both
        o.interior(o.Vc)[...] *= 0.75
        g.interior(g.Vc).mul_(0.75)


@pytest.mark.parametrize("nstages", [2, 3])
@pytest.mark.parametrize("dim,n,mhd,bc", SHORT)
def test_short_directions_at_every_level(dim, n, mhd, bc, nstages):
    """Stages that need the last fill's ghost cells keep to one array: every bit, over three
    cycles, as with a kernel per step."""
    import torch
    kw = cfg_kwargs(dim, n, mhd=mhd, solver="hlld" if mhd else "hllc", recon="ppm", bc=bc, gamma=1.4,
                    cfl=0.3, nstages=nstages)
    _, g = make_pair(kw, problems.random_mhd if mhd else problems.random_hd)
    _, h = make_pair(kw, problems.random_mhd if mhd else problems.random_hd)
    h.set_fusion(0)
    for _ in range(3):
        g.cycle()
        h.cycle()
        assert g.dt == h.dt
    assert torch.equal(g.interior(g.Vc), h.interior(h.Vc))
    if mhd:
        for a, b in zip(interior_faces(g, g.download()[1]), interior_faces(h, h.download()[1])):
            assert (a == b).all()


@pytest.mark.parametrize("n,fused", [((203, 150, 97), True), ((320, 200, 42), True), ((30, 300, 300), False),
                                     ((16, 16, 10300), False), ((128, 128, 160), False), ((64, 60, 60), False)])
def test_which_constrained_transport(n, fused):
    """Level 1 takes the fused kernel where a block of enough cells fills its tiles; the other two
    on narrow ones.  Every bit is that of the fused kernel, which level 2 takes."""
    import torch
    from idefix_amd.datablock import DataBlock
    blocks = []
    for level in (1, 2):
        g = DataBlock(3, n, recon="plm", cfl=0.3, first_dt=1e-7)
        gen = torch.Generator(device="cuda")
        gen.manual_seed(3)
        g.Vc.copy_(torch.rand(g.Vc.shape, generator=gen, device="cuda", dtype=torch.float64) * 0.3 + 0.5)
        g.Vs.copy_(torch.rand(g.Vs.shape, generator=gen, device="cuda", dtype=torch.float64) * 0.2)
        g.set_fusion(level)
        g.set_profiling(True)
        for _ in range(2):
            g.cycle()
        assert ("ct_fused" in g.region_times()) == (fused or level == 2)
        blocks.append(g)
    a, b = blocks
    assert a.dt == b.dt
    assert torch.equal(a.interior(a.Vc), b.interior(b.Vc))
    for x, y in zip(interior_faces(a, a.Vs), interior_faces(b, b.Vs)):
        assert torch.equal(x, y)
