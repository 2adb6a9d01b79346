"""The multigrid against the oracle, bit for bit, where its launches change: the tiles of the fine
levels (remainders, several rows of points per thread), and the coarse levels in one workgroup (one
or two points per thread, levels of a single wavefront, one level alone, a bottom level too large
for it), node- and cell-centred, square and not.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from helpers import random_store  # noqa: E402
from hipace2_amd.inputs import SliceConfig  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [
    (7, 7), (15, 31), (63, 63), (127, 63), (129, 127), (261, 259), (391, 391), (511, 127),   # node-centred
    (4, 8), (64, 66), (100, 100), (128, 256), (130, 130), (262, 130), (384, 96), (640, 512),   # cell-centred
    (1151, 1151)])
def test_mg_sizes(nx, ny):
    from hipace2_amd.simulation import Simulation
    from oracle.oracle import OracleSim
    cfg = SliceConfig(nx=nx, ny=ny, nz=2, xlo=-4.0, xhi=4.0, ylo=-4.0, yhi=4.0, zlo=0.0, zhi=1.0)
    sim, orc = Simulation(cfg), OracleSim(cfg)
    st = random_store(sim.ncomp, sim.ldy, sim.ldx, seed=nx)
    rng = np.random.default_rng(ny)
    for tol, maxiter in [(1e-4, 30), (1e-300, 2), (1e-6, 3)]:
        # new coefficients for every solve: nothing of the last one's may be left
        st[orc.layout["chi"]] = rng.uniform(0.0, 2.0, st[0].shape)
        orc.set_store(st)
        sim.store.copy_(torch.as_tensor(st))
        rc_g, it_g = sim.mg_solve1(tol_rel=tol, maxiter=maxiter)
        rc_o, it_o = orc.mg_solve1(tol_rel=tol, maxiter=maxiter)
        assert (rc_g, it_g) == ({0: 0, 1: 3, 2: 4}[rc_o], it_o)
        g, o = sim.store_host(), orc.store()
        for name in ("Bx", "By"):
            assert np.array_equal(g[sim.layout[name]], o[orc.layout[name]]), (tol, maxiter, name)
