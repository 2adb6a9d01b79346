"""The ordered plasma depositions against the oracle, bit for bit, where their particle sequences can
go wrong: plasmas in lattice order (listed runs), with runs that span the domain (particles that
wrapped around), in random index order (runs found through the boxes), with more particles in a
window than are sequenced at a time, tiles narrower than a block and off its grid, remainders of
runs and of blocks.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from helpers import PLASMA_REALS, random_store  # noqa: E402
from hipace2_amd.inputs import SliceConfig  # noqa: E402

pytestmark = pytest.mark.gpu

COMPS = ["jx", "jy", "jz", "rho", "chi", "rhomjz"]


def _config(nx, ny, order, dtype, tile):
    return SliceConfig(nx=nx, ny=ny, nz=4, xlo=-nx / 16, xhi=nx / 16, ylo=-ny / 16, yhi=ny / 16, zlo=0.0, zhi=1.0,
                       depos_order=order, derivative_type=dtype, deposit_rho=True, tile_size=tile)


def _lattice(cfg, ppc, amp, wrapped, seed):
    """A displaced lattice in injection order; `wrapped` particles moved to random places."""
    rng = np.random.default_rng(seed)
    j, i, k = np.meshgrid(np.arange(cfg.ny), np.arange(cfg.nx), np.arange(ppc * ppc), indexing="ij")
    x = (i + (0.5 + k % ppc) / ppc).ravel()
    y = (j + (0.5 + k // ppc) / ppc).ravel()
    x = x + amp * np.sin(2 * np.pi * y / 13.0)
    y = y + amp * np.cos(2 * np.pi * x / 17.0)
    n = x.size
    w = rng.choice(n, size=min(wrapped, n), replace=False)
    x[w], y[w] = rng.uniform(0, cfg.nx, w.size), rng.uniform(0, cfg.ny, w.size)
    d = {"x": cfg.xlo + np.clip(x, 0.01, cfg.nx - 0.01) * cfg.dx, "y": cfg.ylo + np.clip(y, 0.01, cfg.ny - 0.01) * cfg.dy,
         "w": rng.uniform(0.5, 1.5, n), "ux": rng.normal(0, 0.2, n), "uy": rng.normal(0, 0.2, n),
         "psi": 1.0 + rng.uniform(-0.3, 0.3, n), "valid": (rng.uniform(size=n) > 0.02).astype(np.int32)}
    for k in PLASMA_REALS:
        d.setdefault(k, d[k.replace("_prev", "").replace("_half_step", "")])
    return d


# nx, ny, ppc, amp (cells), wrapped, shuffled, tile
CASES = [(63, 63, 1, 0.1, 0, False, 32), (45, 81, 2, 3.0, 0, False, 32), (64, 32, 2, 3.0, 5, False, 8),
         (63, 47, 2, 1.0, 700, False, 24), (31, 33, 7, 2.0, 0, False, 32), (33, 31, 7, 2.0, 30, False, 9),
         (79, 63, 1, 1.0, 0, True, 32), (127, 129, 1, 1.0, 0, True, 64)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(str(v) for v in c))
@pytest.mark.parametrize("order,dtype", [(0, 2), (1, 2), (2, 2), (3, 2), (2, 1), (3, 0)])
def test_ordered_depositions(case, order, dtype):
    from hipace2_amd import _abi
    from hipace2_amd.simulation import Simulation
    from oracle.oracle import OracleSim
    nx, ny, ppc, amp, wrapped, shuffled, tile = case
    cfg = _config(nx, ny, order, dtype, tile)
    d = _lattice(cfg, ppc, amp, wrapped, seed=nx)
    if shuffled:
        p = np.random.default_rng(1).permutation(d["x"].size)
        d = {k: np.ascontiguousarray(v[p]) for k, v in d.items()}
    sim, orc = Simulation(cfg), OracleSim(cfg)
    st = random_store(sim.ncomp, sim.ldy, sim.ldx, seed=2)
    sim.store.copy_(torch.as_tensor(st))
    orc.set_store(st)
    orc.set_plasma(d)
    sim.np = d["x"].size
    for k in PLASMA_REALS:
        sim.plasma[k] = torch.as_tensor(d[k], dtype=torch.float64).to(sim.device)
    sim.plasma["valid"] = torch.as_tensor(d["valid"]).to(sim.device)
    sim._pdesc = _abi.Plasma(*[sim.plasma[k].data_ptr() for k in PLASMA_REALS + ["valid"]], sim.np)
    comps = [c if sim.layout[c] >= 0 else -1 for c in COMPS]   # six sums, and the usual four
    for cs in (comps, ["jx", "jy", -1, -1, "chi", "rhomjz"]):
        assert sim.deposit_current(cs) == orc.deposit_plasma(cs)
    sim.explicit_deposition()
    orc.explicit_deposit()
    g, o = sim.store_host(), orc.store()
    for name in ("jx", "jy", "rho", "chi", "rhomjz", "Sx", "Sy"):
        assert np.array_equal(g[sim.layout[name]], o[orc.layout[name]]), name
