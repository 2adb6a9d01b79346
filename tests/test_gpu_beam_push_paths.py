"""Time steps with a beam that is pushed and slips from slice to slice, against the oracle, over the
ways through the slice loop: both solvers, with and without transverse beam currents (the beam's
sequences are built one or two slices ahead of the push), ordered deposition bit for bit and atomic
deposition to its rounding.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from helpers import small_config  # noqa: E402
from hipace2_amd.inputs import BeamSpec, make_beam  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("explicit", [True, False], ids=["explicit", "pc"])
@pytest.mark.parametrize("jxjy", [True, False], ids=["jxjy", "jz"])
@pytest.mark.parametrize("deposition", ["ordered", "atomic"])
def test_pushed_beam(explicit, jxjy, deposition):
    from hipace2_amd.simulation import Simulation
    from oracle.oracle import OracleSim
    cfg = small_config(n=31, nz=16, order=2, explicit=explicit)
    cfg.do_beam_jx_jy, cfg.deposition = jxjy, deposition
    beam = make_beam(cfg, BeamSpec(injection_type="fixed_weight", profile="gaussian", density=0.3,
                                   position_std=(0.4, 0.3, 1.41), num_particles=8000, u_mean=(0.5, -0.3, 15.0),
                                   u_std=(0.5, 0.5, 2.0), seed=5))
    sim, orc = Simulation(cfg, beam), OracleSim(cfg, beam)
    n = beam.n
    moved = 0
    for step in range(3):
        if step > 0:
            before = np.array(sim.beam_host.off)
            sim.sort_beam()
            orc.sort_beam()
            moved += int(np.abs(np.array(sim.beam_host.off) - before).sum())
        names = ("Ez", "Bx", "Psi")
        cg, co = {k: sim.capture(k) for k in names}, {k: orc.capture(k) for k in names}
        sim.run_step_with_beam(4.0, 10)
        orc.begin_step()
        orc.run_step_with_beam(4.0, 10)
        torch.cuda.synchronize()
        assert sim.stats()["pc_iters"] == orc.stats()["pc_iters"]
        ob = orc.beam()
        got = {k: sim.beam[k][:n].cpu().numpy() for k in ("x", "y", "z", "ux", "uy", "uz", "w", "valid")}
        pairs = [(k, got[k], ob[k]) for k in got if k in ob] + [(k, cg[k].cpu().numpy(), co[k]) for k in names]
        for k, a, b in pairs:
            if deposition == "ordered":
                assert np.array_equal(a, b), (step, k)
            else:   # FP64 sums in hardware order, a few ulp per cell and slice
                assert np.abs(a - b).max() <= 1e-10 * np.abs(b).max(), (step, k)
        sim.clear_captures()
        orc.clear_captures()
    assert moved > 0
