"""Shock flattening of single cells at the edges of the flags' 60 x 12 tiles and
of their chunks along x3, on grids down to the smallest: bit for bit against the
oracle, in whole stages and in the separate sweeps, and not the unflattened run.
"""
import numpy as np
import pytest

from phlegethon_amd import problems as P
from phlegethon_amd.config import (BC_OUTFLOW, BC_PERIODIC, BC_REFLECTIVE, HLLC_FLUX, LHLLD_FLUX,
                                   PPH_REC, PhlxConfig)

pytestmark = pytest.mark.gpu

WALLS = (BC_PERIODIC, BC_PERIODIC, BC_REFLECTIVE, BC_REFLECTIVE, BC_OUTFLOW, BC_OUTFLOW)


def _gpu(pb, nsteps, fused):
    from phlegethon_amd.runtime import Simulation
    sim = Simulation(pb.cfg)
    sim.setup(pb)
    sim.set_fused_sweep(fused)
    sim.init()
    sim.run(nsteps)
    st = sim.download()
    st.update(sim.scalars())
    sim.close()
    return st


def _oracle(pb, nsteps):
    import oracle
    r = oracle.OracleRun(pb)
    r.init()
    frac = float(r.shock_flags().mean())
    r.run(nsteps)
    st = r.state()
    st.update(time=r.scalar("time"))
    r.close()
    return st, frac


@pytest.mark.parametrize("flux", [HLLC_FLUX, LHLLD_FLUX], ids=["whole-stage", "separate"])
@pytest.mark.parametrize("shape", [(3, 3, 1), (119, 4, 1), (122, 26, 1), (3, 4, 3), (62, 14, 5),
                                   (64, 27, 19)], ids=lambda s: "x".join(map(str, s)))
def test_single_flattened_cells(oracle_mod, shape, flux):
    nx, ny, nz = shape
    sd = 2 if nz == 1 else 3
    cfg = PhlxConfig(sdims=sd, nx1=nx, nx2=ny, nx3=nz, x1u=nx / 32.0, x2u=ny / 32.0, x3u=nz / 32.0,
                     flux=flux, recon=PPH_REC, cfl=0.3, bc=WALLS, shock_flattening=True,
                     eps_sf=0.6).validate()
    pb = P.random_smooth(cfg, amp=0.02)
    # the neighbours of a pressure spike are marked, and what is around them
    spikes = [(i, j, k) for i in (0, 2, 57, 58, 60, 61, 118, 120) for j in (1, 10, 13, 24)
              for k in (0, 3, 10, 17) if i < nx and j < ny and k < nz]
    for n, (i, j, k) in enumerate(spikes):
        if n % 3 == 0 or min(nx, ny) <= 4:
            pb.prim[sd + 1, k, j, i] *= 1.8
    ref, frac = _oracle(pb, 2)
    print(f"flag fraction {frac:.3f}", flush=True)
    assert 0.0 < frac and (frac < 0.9 or min(nx, ny) <= 4)
    plain = pb.copy()
    plain.cfg = cfg.with_(shock_flattening=False)
    assert not np.array_equal(oracle_mod.run_problem(plain, 2)["prim"], ref["prim"])
    for fused in (True, False):
        got = _gpu(pb, 2, fused)
        assert got["time"] == ref["time"] and np.array_equal(got["prim"], ref["prim"])
