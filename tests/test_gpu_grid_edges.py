"""Grids that the other tests do not reach: cell widths that vary along every direction, the
rows of faces at which the fused constrained transport's tiles end, and the batches at which
the training kernel's blocks start to loop."""
import ctypes

import numpy as np
import pytest

from idefix_amd import datablock, problems
from oracle.oracle import OracleGrid, lib
from tests import test_gpu_mlp_train_edges
from tests.pairs import cfg_kwargs, compare_state, interior_faces, make_oracle, make_pair

pytestmark = pytest.mark.gpu


def _stretched(kw, ic, monkeypatch, count):
    """An oracle and `count` blocks whose widths vary by up to a half from cell to cell."""
    o = make_oracle(kw)
    rng = np.random.default_rng(11)
    dx = []
    for d in range(3):
        n = o.np_tot[d]
        view = np.ctypeslib.as_array(ctypes.cast(lib().orc_coord(o._h, d, 3), ctypes.POINTER(ctypes.c_double)), (n,))
        if d < kw["dim"]:
            view *= rng.uniform(0.75, 1.25, n)
        dx.append(view.copy())
    real = datablock.make_grid
    monkeypatch.setattr(datablock, "make_grid", lambda *a: real(*a)[:3] + (dx,))
    Vc, Vs = ic(OracleGrid(o))
    o.Vc[...] = Vc
    if kw["mhd"]:
        o.Vs[...] = Vs
    blocks = []
    for _ in range(count):
        g = datablock.DataBlock(kw["dim"], kw["nx"], mhd=kw["mhd"], comps=kw["comps"], recon=kw["recon"],
                                solver=kw["solver"], emf=kw["emf"], bc=kw["bc"], gamma=kw["gamma"], cfl=kw["cfl"],
                                nstages=kw["nstages"], first_dt=kw["first_dt"])
        g.upload(Vc, Vs)
        blocks.append(g)
    return o, blocks


@pytest.mark.parametrize("n,mhd,recon,emf,nstages,bc", [
    ((70,), False, "plm", "uct_contact", 2, "outflow"), ((70,), False, "ppm", "uct_contact", 3, "periodic"),
    ((61, 9), False, "plm", "uct_contact", 2, "outflow"), ((12, 7, 9), False, "ppm", "uct_contact", 3, "outflow"),
    ((61, 9), True, "plm", "uct_hlld", 2, "periodic"), ((20, 12), True, "ppm", "uct_contact", 3, "periodic"),
    ((12, 7, 9), True, "plm", "uct_contact", 2, "periodic"), ((62, 5, 4), True, "limo3", "uct_contact", 2, "outflow"),
    ((12, 11, 9), True, "ppm", "uct_contact", 3, "periodic")])
def test_cell_widths_that_vary(n, mhd, recon, emf, nstages, bc, monkeypatch):
    """Every level of idfx_ctx_set_fusion: every bit of level 0, whose cells and dt are the
    oracle's to 1e-12."""
    import torch
    kw = cfg_kwargs(len(n), n, mhd=mhd, solver="hlld" if mhd else "hllc", emf=emf, recon=recon, bc=bc,
                    cfl=0.3, nstages=nstages)
    o, (g, h, q) = _stretched(kw, problems.random_mhd if mhd else problems.random_hd, monkeypatch, 3)
    assert len(set(g.dx[0])) == g.np_tot[0]
    h.set_fusion(0)
    q.set_fusion(2)
    o.set_boundaries()
    for _ in range(2):
        assert o.cycle() == 0
        for b in (g, h, q):
            b.cycle()
        assert g.dt == h.dt == q.dt
    assert h.dt == pytest.approx(o.dt, rel=1e-12)
    compare_state(o, h, what="stretched %s %s" % (recon, n))
    for b in (g, q):
        assert torch.equal(b.interior(b.Vc), h.interior(h.Vc))
        assert torch.equal(b.interior(b.Uc), h.interior(h.Uc))
        if mhd:
            for x, y in zip(interior_faces(o, b.download()[1]), interior_faces(o, h.download()[1])):
                assert (x == y).all()


@pytest.mark.parametrize("n", [(61, 8, 3), (61, 9, 3), (62, 10, 4), (20, 11, 3), (63, 19, 3), (62, 20, 4), (4, 21, 3)])
def test_ct3d_rows(n):
    """The fused constrained transport at the ends of its tiles of 62 x 10 faces."""
    kw = cfg_kwargs(3, n, emf="uct_contact", recon="ppm", nstages=3, cfl=0.3)
    o, g = make_pair(kw, problems.random_mhd)
    g.set_fusion(2)
    o.set_boundaries()
    for _ in range(2):
        assert o.cycle() == 0
        g.cycle()
    compare_state(o, g, what="ct3d %s" % (n,))


@pytest.mark.parametrize("batch", [8192, 8193])
def test_training_blocks_that_loop(batch):
    """256 blocks of 32 rows, and one row more."""
    test_gpu_mlp_train_edges.test_loss_and_gradient(batch, 0)
