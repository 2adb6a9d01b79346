"""The field gather of the plasma push against the oracle, bit for bit, where the O + 1 cells of the
shape function change place in the stencil: particles on nodes, cell centres, the points in
between and one ulp beside them, and stencils that leave the guarded plane.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from helpers import random_plasma, random_store, small_config  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [31, 64])
def test_gather_windows(order, n):
    from hipace2_amd.simulation import Simulation
    from oracle.oracle import OracleSim
    cfg = small_config(n=n, order=order, dtype=2 if order > 0 else 1)
    sim, orc = Simulation(cfg), OracleSim(cfg)
    st = random_store(sim.ncomp, sim.ldy, sim.ldx, seed=order)
    sim.store.copy_(torch.as_tensor(st))
    orc.set_store(st)
    d = random_plasma(cfg, sim.np, seed=n)
    rng = np.random.default_rng(order)
    for k, lo, hi, step in (("x_prev", cfg.xlo, cfg.xhi, cfg.dx), ("y_prev", cfg.ylo, cfg.yhi, cfg.dy)):
        at = np.round((d[k] - lo) / step * 4.0) / 4.0 * step + lo
        # one in eight out at the box's edge, or beyond it by less than the guard cells
        at = np.where(rng.uniform(size=at.size) < 0.125, rng.choice([lo, hi, lo - step, hi + step], at.size), at)
        d[k] = np.nextafter(at, at + rng.choice([-1.0, 0.0, 1.0], at.size))
    orc.set_plasma(d)
    sim.set_plasma(d)
    sim.advance_plasma_particles()
    orc.push_plasma()
    g, o = sim.plasma_host(), orc.plasma()
    for k in g:
        assert np.array_equal(g[k], o[k]), k
