"""The ordered beam deposition against the oracle, bit for bit, where the chunks of a cell's
contributions end: sequences from one below to one above the lengths that a wavefront reads and adds
at a time, and more long sequences than there are wavefronts.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from hipace2_amd.inputs import BeamArrays, SliceConfig  # noqa: E402

pytestmark = pytest.mark.gpu


def _check(cfg, x, y, seed):
    from hipace2_amd.simulation import Simulation
    from oracle.oracle import OracleSim
    rng = np.random.default_rng(seed)
    n = x.size
    z = np.full(n, cfg.zlo + 0.5 * cfg.dz)
    beam = BeamArrays(x=x, y=y, z=z, ux=rng.normal(0, 1, n), uy=rng.normal(0, 1, n), uz=rng.uniform(10, 20, n),
                      w=rng.uniform(0.5, 1.5, n), valid=(rng.uniform(size=n) > 0.05).astype(np.int32),
                      off=np.array([0] + [n] * cfg.nz, dtype=np.int64), charge=-1.0, mass=1.0)
    sim, orc = Simulation(cfg, beam), OracleSim(cfg, beam)
    st = rng.uniform(-1, 1, (sim.ncomp, sim.ldy, sim.ldx))
    sim.store.copy_(torch.as_tensor(st))
    orc.set_store(st)
    for args in (("jx_beam", "jy_beam", "jz_beam"), (-1, -1, "jz_beam"), ("jx_beam", "jy_beam", -1)):
        sim.deposit_current_slice(0, *args)
        orc.deposit_beam(0, *args)
    g, o = sim.store_host(), orc.store()
    for name in ("jx_beam", "jy_beam", "jz_beam"):
        assert np.array_equal(g[sim.layout[name]], o[orc.layout[name]]), name


def _config(n, order):
    return SliceConfig(nx=n, ny=n, nz=2, xlo=-n / 16, xhi=n / 16, ylo=-n / 16, yhi=n / 16, zlo=0.0, zhi=1.0,
                       depos_order=order, has_plasma=False)


@pytest.mark.parametrize("order", [0, 1, 2, 3])
def test_sequence_lengths(order):
    """One spot for every length, all of a spot's particles in one cell, in random index order."""
    cfg = _config(127, order)
    lengths = [c + d for c in (32, 40, 56, 64, 72, 128, 256, 320, 512) for d in (-1, 0, 1)]
    k = np.repeat(np.arange(len(lengths)), lengths)
    rng = np.random.default_rng(order)
    rng.shuffle(k)
    x = cfg.xlo + (8 + 16 * (k % 7) + rng.uniform(0.3, 0.7, k.size)) * cfg.dx
    y = cfg.ylo + (8 + 16 * (k // 7) + rng.uniform(0.3, 0.7, k.size)) * cfg.dy
    _check(cfg, x, y, order)


def test_more_long_sequences_than_wavefronts():
    cfg = _config(127, 2)
    rng = np.random.default_rng(4)
    n = 150_000   # 80 a cell over a third of the grid
    x, y = rng.uniform(cfg.xlo / 2, cfg.xhi / 2, n), rng.uniform(cfg.ylo / 3, cfg.yhi / 3, n)
    _check(cfg, x, y, 5)
