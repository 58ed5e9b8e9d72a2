"""Values near the end of FP64's range.  A transverse velocity of 1e-310 rides on a uniform flow
(density 1, so that momenta and velocities are the same numbers and every other variable keeps
its bits): its curvatures are subnormal, its PPM limiter has an extremum in every cell."""
import numpy as np
import pytest

from tests.pairs import cfg_kwargs, make_pair

pytestmark = pytest.mark.gpu


def _tail(g, amp):
    rng = np.random.default_rng(5)
    Vc = np.zeros((2 + g.dim, g.np_tot[2], g.np_tot[1], g.np_tot[0]))
    Vc[0], Vc[1], Vc[1 + g.dim] = 1.0, 0.5, 1.0
    Vc[2] = amp * np.round(rng.uniform(-1, 1, Vc.shape[1:]) * 16)
    return Vc, None


@pytest.mark.parametrize("amp", [1e-3, 2.0 ** -960, 2.0 ** -1010, 2.0 ** -1035])
@pytest.mark.parametrize("n", [(70, 5), (20, 9), (14, 7, 5)])
def test_ppm_limits_values_whose_curvature_is_subnormal(n, amp):
    """Against the oracle, whose quotients are IEEE's: 1e-12 of the amplitude, or four steps of
    the subnormal grid, where each of the two stages rounds two quotients once more at most."""
    kw = cfg_kwargs(len(n), n, mhd=False, solver="hllc", recon="ppm", gamma=1.4, cfl=0.3, nstages=2,
                    first_dt=1e-3)
    o, g = make_pair(kw, lambda gg: _tail(gg, amp))
    o.set_boundaries()
    assert o.cycle() == 0
    g.cycle()
    got, want = g.interior(g.Vc).cpu().numpy(), o.interior(o.Vc)
    for v in (0, 1, 1 + len(n)):
        assert np.array_equal(got[v], want[v])
    assert np.abs(want[2]).max() > amp
    assert np.abs(got[2] - want[2]).max() <= max(1e-12 * amp, 4 * 2.0 ** -1074)
