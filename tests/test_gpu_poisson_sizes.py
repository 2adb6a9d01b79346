"""The transverse Poisson solves against the oracle, bit for bit, at sizes without a power-of-two
transform: remainders of the 32 x 32 tiles of the matrix path in every place, one direction by FFT
and the other by sums, rows of several fields in one tile.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from helpers import random_store  # noqa: E402
from hipace2_amd.inputs import SliceConfig  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(7, 9), (31, 33), (33, 31), (32, 64), (65, 63), (63, 47), (96, 40), (100, 130),
                                   (257, 95)])
def test_poisson_sizes(nx, ny):
    from hipace2_amd.simulation import Simulation
    from oracle.oracle import OracleSim
    cfg = SliceConfig(nx=nx, ny=ny, nz=2, xlo=-4.0, xhi=4.0, ylo=-3.0, yhi=3.0, zlo=0.0, zhi=1.0, has_plasma=False)
    sim, orc = Simulation(cfg), OracleSim(cfg)
    st = random_store(sim.ncomp, sim.ldy, sim.ldx, seed=nx)
    sim.store.copy_(torch.as_tensor(st))
    orc.set_store(st)
    sim.solve_poisson_psi_exmby_eypbx_ez_bz()
    orc.solve_poisson_psi_ez_bz()
    g, o = sim.store_host(), orc.store()
    for name in ("Psi", "Ez", "Bz", "ExmBy", "EypBx"):
        assert np.array_equal(g[sim.layout[name]], o[orc.layout[name]]), name
