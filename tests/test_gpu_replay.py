"""Depositions recorded into a HIP graph and replayed: every replay adds what the oracle adds, with
eager depositions of the same context between the replays and with particles that have moved since
the recording (plasma in lattice and in random order, the beam of a slice).
"""
import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from helpers import random_store  # noqa: E402
from hipace2_amd.inputs import BeamSpec, make_beam  # noqa: E402
from test_gpu_ordered import COMPS, _config, _lattice  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,order,dtype,shuffled", [
    (63, 47, 2, 2, False), (61, 63, 1, 2, True), (127, 129, 3, 0, True)])
def test_depositions_replayed(nx, ny, order, dtype, shuffled):
    from hipace2_amd.simulation import Simulation
    from oracle.oracle import OracleSim
    cfg = _config(nx, ny, order, dtype, 32)
    beam = make_beam(cfg, BeamSpec(injection_type="fixed_weight", profile="gaussian", density=1.0,
                                   position_mean=(0.1, -0.2, 0.5), position_std=(0.4, 0.3, 0.3), num_particles=4000,
                                   u_mean=(0.0, 0.0, 100.0), seed=2))
    d = _lattice(cfg, 1, 2.0, 0, seed=nx)
    if shuffled:
        p = np.random.default_rng(1).permutation(d["x"].size)
        d = {k: np.ascontiguousarray(v[p]) for k, v in d.items()}
    sim, orc = Simulation(cfg, beam), OracleSim(cfg, beam)
    st = random_store(sim.ncomp, sim.ldy, sim.ldx, seed=2)
    st_gpu = torch.as_tensor(st).to(sim.device)
    comps = [c if sim.layout[c] >= 0 else -1 for c in COMPS]
    arr = (C.c_int32 * 6)(*[sim.layout.get(c, -1) if isinstance(c, str) else c for c in comps])

    def deposit():
        rc = sim.L.hpq_deposit_current(sim.ctx, C.byref(sim._pdesc), C.c_void_p(sim.store.data_ptr()), arr, 0, None)
        assert rc == 0
        sim.explicit_deposition()
        sim.deposit_current_slice(1, "jx_beam", "jy_beam", "jz_beam")

    def expected(state):
        orc.set_store(st)
        orc.set_plasma(state)
        orc.deposit_plasma(comps)
        orc.explicit_deposit()
        orc.deposit_beam(1, "jx_beam", "jy_beam", "jz_beam")
        return orc.store().copy()

    sim.set_plasma(d)
    sim.store.copy_(st_gpu)
    deposit()   # the scratch is in place before the recording
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        eager = sim.stream
        sim.set_stream(torch.cuda.current_stream())
        deposit()
    sim.set_stream(eager)
    want = expected(d)
    names = ("jx", "jy", "rho", "chi", "rhomjz", "Sx", "Sy", "jx_beam", "jy_beam", "jz_beam")
    for k in range(6):
        if k == 3:   # other cells than those of the recording
            d = dict(d, x=np.clip(d["x"] + 9.3 * cfg.dx, cfg.xlo, cfg.xhi - 0.1 * cfg.dx))
            want = expected(d)
            sim.set_plasma(d)
        if k % 2:
            deposit()
            torch.cuda.synchronize()
        sim.store.copy_(st_gpu)
        graph.replay()
        g = sim.store_host()
        for name in names:
            assert np.array_equal(g[sim.layout[name]], want[orc.layout[name]]), (k, name)
