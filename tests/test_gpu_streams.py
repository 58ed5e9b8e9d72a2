"""Calls on streams that do not wait for the null stream (torch's side streams): the first
cycles of a block, which use memory that the library has just allocated and cleared, and the
time step that the host polls for, with one context and with two in flight."""
import threading

import pytest

from idefix_amd import problems

pytestmark = pytest.mark.gpu


def _block(dim, n, mhd, recon, nstages, bc="periodic"):
    from idefix_amd.datablock import DataBlock
    g = DataBlock(dim, n, mhd=mhd, recon=recon, solver="hlld" if mhd else "hllc", bc=bc, cfl=0.3,
                  nstages=nstages, first_dt=1e-5)
    g.upload(*(problems.random_mhd if mhd else problems.random_hd)(g))
    return g


def _cycles(g, n=3):
    import torch
    dts = []
    for _ in range(n):
        g.cycle()
        dts.append(g.dt)
    torch.cuda.current_stream().synchronize()
    return dts


def _equal(a, b):
    import torch
    assert torch.equal(a.interior(a.Vc), b.interior(b.Vc))
    assert torch.equal(a.interior(a.Uc), b.interior(b.Uc))
    if a.mhd:
        assert torch.equal(a.interior(a.Vs), b.interior(b.Vs))


@pytest.mark.parametrize("nstages", [2, 3])
@pytest.mark.parametrize("dim,n,mhd,recon", [(1, (1000,), False, "plm"), (1, (20000,), False, "plm"),
                                             (2, (256, 256), True, "ppm"), (2, (256, 200), False, "plm"),
                                             (3, (40, 36, 32), True, "plm"),
                                             (3, (48, 40, 36), False, "ppm")])
def test_first_cycles_on_a_side_stream(dim, n, mhd, recon, nstages):
    """A block created and stepped on a side stream from its first cycle on (the first RK3 cycle
    allocates): every bit as on the default stream."""
    import torch
    a = _block(dim, n, mhd, recon, nstages)
    want = _cycles(a)
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):
        b = _block(dim, n, mhd, recon, nstages)
        got = _cycles(b)
    torch.cuda.synchronize()
    assert got == want
    _equal(a, b)


def test_two_contexts_in_flight():
    """Two threads, each with its own stream and blocks of its own: every cycle's time step and
    the states as when one runs after the other."""
    import torch
    kinds = [[(1, (3000,), False, "plm", 2), (2, (128, 96), True, "plm", 2)],
             [(3, (24, 20, 16), False, "plm", 3), (1, (20000,), False, "plm", 3)]]
    want = [[(g, _cycles(g, 5)) for g in (_block(*k) for k in ks)] for ks in kinds]
    torch.cuda.synchronize()
    got, errors = [None, None], []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                blocks = [_block(*k) for k in kinds[i]]
                dts = [[] for _ in blocks]
                for _ in range(5):
                    for g, d in zip(blocks, dts):
                        g.cycle()
                        d.append(g.dt)
                torch.cuda.current_stream().synchronize()
                got[i] = list(zip(blocks, dts))
        except Exception as e:  # reported by the main thread
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for w, r in zip(want, got):
        for (a, da), (b, db) in zip(w, r):
            assert da == db
            _equal(a, b)


def test_new_weights_behind_a_running_cycle():
    """The learned limiter's weights replaced right after a cycle returned on a side stream, its
    last stages still running: they take the old weights."""
    import numpy as np
    import torch
    from idefix_amd import learned
    from idefix_amd.datablock import DataBlock
    p = learned.init_params(8)
    q = p + np.random.default_rng(9).normal(0, 0.05, p.shape).astype(np.float32)
    out = []
    for late in (False, True):
        with torch.cuda.stream(torch.cuda.Stream()):
            g = DataBlock(2, (512, 384), comps=3, mhd=True, recon="mlp", precision="fp32", cfl=0.3,
                          nstages=3, first_dt=1e-5)
            g.upload(*problems.random_mhd(g))
            g.set_mlp_params(q)
            g.cycle()
            if not late:
                torch.cuda.current_stream().synchronize()
            g.set_mlp_params(p)
            torch.cuda.current_stream().synchronize()
            out.append(g)
    torch.cuda.synchronize()
    _equal(*out)


def test_training_on_a_side_stream():
    """A trainer created, stepped, read and given new parameters on a side stream without waits
    of the caller's: every parameter as on the default stream."""
    import contextlib

    import numpy as np
    import torch
    from idefix_amd import learned
    rng = np.random.default_rng(2)
    B = 20000
    X = rng.uniform(-1, 1, (B, 72)).astype(np.float32)
    tau = rng.uniform(-0.5, 0.5, (B, 8)).astype(np.float32)
    p = learned.pack({k: v + 0.05 * rng.standard_normal(np.shape(v))
                      for k, v in learned.unpack(learned.init_params(3)).items()})
    got = []
    for side in (False, True):
        with torch.cuda.stream(torch.cuda.Stream()) if side else contextlib.nullcontext():
            x, t = torch.from_numpy(X).cuda(), torch.from_numpy(tau).cuda()
            torch.cuda.synchronize()
            tr = learned.Trainer(B, p)
            for _ in range(20):
                tr.step(x, t, 1e-3)
            first = tr.params()
            for _ in range(20):
                tr.step(x, t, 1e-3)
            tr.set_params(p)
            for _ in range(5):
                tr.step(x, t, 1e-3)
            got.append((first, tr.params()))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    assert not np.array_equal(got[0][0], p)
