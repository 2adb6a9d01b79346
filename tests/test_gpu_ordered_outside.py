"""The ordered plasma depositions against the oracle, bit for bit, with particles up to eight cells
outside the box on all sides: those whose stencil reaches the guard cells deposit there, the others
nothing. Grids with every remainder of a deposition block's width and height, for all three block
sizes.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_ordered import COMPS, _config, _lattice  # noqa: E402

pytestmark = pytest.mark.gpu


def _outside(cfg, d, rng):
    """A third of the particles in the frame of eight cells around the box."""
    n = d["x"].size
    k = n // 3
    w = rng.choice(n, size=k, replace=False)
    x, y = rng.uniform(-8, cfg.nx + 8, k), rng.uniform(-8, cfg.ny + 8, k)
    side = rng.integers(0, 4, k)
    far = rng.uniform(0, 8, k)
    x = np.where(side == 0, -far, np.where(side == 1, cfg.nx + far, x))
    y = np.where(side == 2, -far, np.where(side == 3, cfg.ny + far, y))
    d["x"][w], d["y"][w] = cfg.xlo + x * cfg.dx, cfg.ylo + y * cfg.dy
    d["x_prev"], d["y_prev"] = d["x"].copy(), d["y"].copy()


# blocks of 8 x 4 cells, then 8 x 8, then 16 x 8
SIZES = [(57, 59), (58, 62), (59, 57), (60, 58), (61, 63), (62, 60), (63, 61), (64, 64),
         (365, 365), (366, 358), (523, 509), (509, 523)]


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("order,dtype", [(0, 1), (1, 2), (2, 1), (2, 2), (3, 0), (3, 2)])
def test_particles_outside_the_box(nx, ny, order, dtype):
    from helpers import random_store
    from hipace2_amd.simulation import Simulation
    from oracle.oracle import OracleSim
    cfg = _config(nx, ny, order, dtype, 32)
    d = _lattice(cfg, 1, 0.5, 0, seed=nx)
    _outside(cfg, d, np.random.default_rng(ny))
    sim, orc = Simulation(cfg), OracleSim(cfg)
    st = random_store(sim.ncomp, sim.ldy, sim.ldx, seed=2)
    sim.store.copy_(torch.as_tensor(st))
    orc.set_store(st)
    orc.set_plasma(d)
    sim.set_plasma(d)
    comps = [c if sim.layout[c] >= 0 else -1 for c in COMPS]
    for cs in (comps, ["jx", "jy", -1, -1, "chi", "rhomjz"]):
        assert sim.deposit_current(cs) == orc.deposit_plasma(cs)
    sim.explicit_deposition()
    orc.explicit_deposit()
    g, o = sim.store_host(), orc.store()
    for name in ("jx", "jy", "rho", "chi", "rhomjz", "Sx", "Sy"):
        assert np.array_equal(g[sim.layout[name]], o[orc.layout[name]]), name
