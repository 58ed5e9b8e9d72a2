"""Sweeps at the sizes where their lane mapping can go wrong: the sites of an x sweep and the
columns of a y or z sweep are dealt to waves of 64 lanes across row ends, so rows shorter
than a wave, rows that end at or next to a wave's last lanes, and last waves with one site
are compared with the oracle cell by cell (FP64 bar of tests/pairs.py)."""
import pytest

from idefix_amd import problems
from tests.pairs import cfg_kwargs, compare_state, interior_faces, make_pair

pytestmark = pytest.mark.gpu

# a wave of the x sweep solves 62 sites (PLM) or 61 (PPM); a row holds nx + 2 or nx + 3
SIZES_3D = [(4, 5, 3), (7, 4, 6), (58, 3, 4), (59, 4, 3), (61, 3, 3), (64, 3, 4), (121, 3, 3),
            (125, 4, 3), (130, 3, 3), (3, 33, 18)]


@pytest.mark.parametrize("recon,nstages", [("plm", 2), ("ppm", 3)])
@pytest.mark.parametrize("n", SIZES_3D)
def test_mhd_3d(n, recon, nstages):
    kw = cfg_kwargs(3, n, emf="uct_contact", recon=recon, nstages=nstages, cfl=0.3)
    o, g = make_pair(kw, problems.random_mhd)
    o.set_boundaries()
    assert o.cycle() == 0
    g.cycle()
    compare_state(o, g, what="%s %s" % (recon, n))
    assert g.dt == pytest.approx(o.dt, rel=1e-12)


@pytest.mark.parametrize("recon", ["plm", "ppm"])
@pytest.mark.parametrize("n", [(5, 40), (58, 9), (60, 7), (122, 6), (128, 5)])
def test_mhd_2d_three_components(n, recon):
    kw = cfg_kwargs(2, n, comps=3, emf="uct_contact", recon=recon, nstages=3, cfl=0.3)
    o, g = make_pair(kw, problems.random_mhd)
    o.set_boundaries()
    assert o.cycle() == 0
    g.cycle()
    compare_state(o, g, what="%s %s" % (recon, n))


@pytest.mark.parametrize("recon", ["plm", "ppm"])
@pytest.mark.parametrize("n", [(3,), (59,), (61,), (62,), (123,), (124,), (125,), (1000,)])
def test_hd_1d(n, recon):
    kw = cfg_kwargs(1, n, mhd=False, solver="hllc", recon=recon, bc="outflow", gamma=1.4, cfl=0.3)
    o, g = make_pair(kw, problems.random_hd)
    o.set_boundaries()
    assert o.cycle() == 0
    g.cycle()
    compare_state(o, g, what="%s %s" % (recon, n))


@pytest.mark.parametrize("n", [(3, 4, 5), (60, 5, 4), (62, 3, 3), (64, 4, 4)])
def test_hd_3d_outflow(n):
    kw = cfg_kwargs(3, n, mhd=False, solver="hllc", recon="plm", bc="outflow", gamma=1.4, cfl=0.3)
    o, g = make_pair(kw, problems.random_hd)
    o.set_boundaries()
    assert o.cycle() == 0
    g.cycle()
    compare_state(o, g, what="%s" % (n,))


@pytest.mark.parametrize("nstages", [2, 3])
@pytest.mark.parametrize("n", [(3, 5, 4), (61, 6, 3), (62, 7, 3), (63, 5, 4), (124, 12, 3), (125, 13, 3),
                               (5, 3, 40)])
def test_ct3d_tiles(n, nstages):
    """The fused constrained transport (fusion level 2: at every size) at the edges of its
    tiles of 62 x 6 faces and of its k segments."""
    kw = cfg_kwargs(3, n, emf="uct_contact", recon="ppm" if min(n) >= 3 else "plm", nstages=nstages,
                    cfl=0.3)
    o, g = make_pair(kw, problems.random_mhd)
    g.set_fusion(2)
    o.set_boundaries()
    for _ in range(2):
        assert o.cycle() == 0
        g.cycle()
    compare_state(o, g, what="ct3d %s" % (n,))


@pytest.mark.parametrize("nstages", [2, 3])
@pytest.mark.parametrize("n,csiso", [((61,), None), ((61,), 0.9), ((130,), None), ((60, 7), None),
                                     ((60, 7), 0.9), ((9, 66), None), ((5, 4, 6), None),
                                     ((61, 4, 3), None)])
def test_hydro_ping_pong_equals_in_place(n, nstages, csiso):
    """Hydro stages whose last sweep converts the state (the default) against the schedule
    with ConsToPrim as a kernel of its own: every bit of Vc and Uc, and dt, over three
    cycles; and the oracle."""
    import torch
    kw = cfg_kwargs(len(n), n, mhd=False, solver="hllc", recon="plm", bc="outflow" if len(n) < 3 else
                    "periodic", gamma=1.4, cfl=0.3, nstages=nstages, csiso=csiso)
    o, g = make_pair(kw, problems.random_hd)
    _, h = make_pair(kw, problems.random_hd)
    h.set_fusion(0)
    o.set_boundaries()
    for _ in range(3):
        assert o.cycle() == 0
        g.cycle()
        h.cycle()
    assert g.dt == h.dt
    assert torch.equal(g.interior(g.Vc), h.interior(h.Vc))
    assert torch.equal(g.interior(g.Uc), h.interior(h.Uc))
    compare_state(o, g, what="hydro %s" % (n,))


@pytest.mark.parametrize("n,recon,nstages,bc", [
    (n, r, s, b) for n, r, s in [(2, "plm", 2), (3, "ppm", 2), (61, "plm", 3), (62, "ppm", 2),
                                 (250, "plm", 2), (500, "ppm", 3)]
    for b in ("periodic", "outflow", "reflective", [("reflective", "outflow")])] +
    [(2, "ppm", 3, "periodic"), (2, "ppm", 3, "outflow"), (16384, "plm", 2, "outflow"),
     (16385, "plm", 2, "outflow"), (16385, "plm", 3, "periodic")])
def test_hd_1d_sides_in_the_sweep(n, recon, nstages, bc):
    """1-D hydro sweeps that fill the ghost zones and hand over the time step themselves, at the
    shortest grids (two PPM cells: one less than a ghost zone) and around a wave and a block,
    against the schedule with a kernel for each: every bit of Vc, and dt, over three cycles; and
    the oracle."""
    import torch
    kw = cfg_kwargs(1, (n,), mhd=False, solver="hllc", recon=recon, bc=bc, gamma=1.4, cfl=0.3,
                    nstages=nstages, first_dt=1e-4 if n < 10000 else 1e-6)
    o, g = make_pair(kw, problems.random_hd)
    _, h = make_pair(kw, problems.random_hd)
    h.set_fusion(0)
    o.set_boundaries()
    for _ in range(3):
        assert o.cycle() == 0
        g.cycle()
        h.cycle()
        assert g.dt == h.dt
    assert torch.equal(g.interior(g.Vc), h.interior(h.Vc))
    compare_state(o, g, what="%s %s %s" % (n, recon, bc))


@pytest.mark.parametrize("bc", [["outflow", "reflective", "periodic"], ["reflective", "outflow", "outflow"],
                                ["periodic", "outflow", "reflective"]])
@pytest.mark.parametrize("n", [(4,), (3, 5), (64, 7), (2, 2), (4, 3, 5), (33, 6, 2)])
def test_hd_box_ghost_zones(n, bc):
    """The ghost zones of a hydro box in one kernel, corners included: every bit as the oracle
    fills them direction by direction."""
    kw = cfg_kwargs(len(n), n, mhd=False, solver="hllc", recon="plm", bc=bc[:len(n)], gamma=1.4)
    o, g = make_pair(kw, problems.random_hd)
    o.set_boundaries()
    g.set_boundaries()
    assert (g.download()[0] == o.Vc).all()


@pytest.mark.parametrize("mhd,recon,precision", [(True, "plm", "fp64"), (True, "plm", "fp32"),
                                                 (True, "ppm", "fp32"), (True, "limo3", "fp64"),
                                                 (False, "plm", "fp64"),
                                                 (False, "ppm", "fp64")])
@pytest.mark.parametrize("n", [(4, 3, 5), (3, 37, 4), (52, 4, 3), (54, 5, 3), (56, 4, 3), (58, 3, 3), (60, 5, 2),
                               (62, 3, 3), (114, 4, 3), (118, 5, 3), (57, 130, 3)])
def test_sweep_xy_equals_two_sweeps(n, mhd, recon, precision):
    """x and y sweeps in one kernel (60 or 58 of a wave's 64 lanes own a cell, rows dealt across
    their ends, several segments along y) against a kernel for each: every bit of Vc, Vs and
    dt over two cycles; and the oracle."""
    import torch
    kw = cfg_kwargs(3, n, mhd=mhd, solver="hlld" if mhd else "hllc", emf="uct_contact", recon=recon,
                    cfl=0.3, nstages=2)
    ic = problems.random_mhd if mhd else problems.random_hd
    o, g = make_pair(kw, ic, precision=precision)
    _, h = make_pair(kw, ic, precision=precision)
    if recon == "ppm" and mhd:
        g.set_fusion(2)  # large grids only by default
    h.set_fusion(0)
    o.set_boundaries()
    for _ in range(2):
        assert o.cycle() == 0
        g.cycle()
        h.cycle()
        assert g.dt == h.dt
    assert torch.equal(g.interior(g.Vc), h.interior(h.Vc))
    if mhd:
        for a, b in zip(interior_faces(o, g.download()[1]), interior_faces(o, h.download()[1])):
            assert (a == b).all()
    if precision == "fp64":
        compare_state(o, g, what="xy %s %s" % (recon, n))


@pytest.mark.parametrize("emf,recon", [("uct_hlld", "plm"), ("uct_hlld", "ppm"), ("uct_contact", "plm"),
                                       ("uct_contact", "ppm"), ("uct0", "plm"), ("arithmetic", "ppm")])
@pytest.mark.parametrize("n", [(4, 3), (57, 4), (60, 5), (62, 3), (63, 9), (124, 4), (20, 70)])
def test_mhd_2d_fused(n, emf, recon):
    """The fused second half of a 2-D stage at the edges of its waves' columns (57 to 62 of 64
    lanes own one) and at the one-cell segments small grids take."""
    kw = cfg_kwargs(2, n, emf=emf, recon=recon, nstages=2, cfl=0.3)
    o, g = make_pair(kw, problems.random_mhd)
    o.set_boundaries()
    for _ in range(2):
        assert o.cycle() == 0
        g.cycle()
    compare_state(o, g, what="%s %s %s" % (emf, recon, n))
