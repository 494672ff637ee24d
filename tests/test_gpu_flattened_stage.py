"""Shock flattening in the one-pass stage and the one-launch flags: runs equal
the CPU oracle and the separate sweeps bit for bit, on extents around the
flags' 60 x 12 tiles and the sweep's 16 x 15, with and without scalars, on
walls that mirror and that wrap, captured and not.
"""
import numpy as np
import pytest

from phlegethon_amd import problems as P
from phlegethon_amd.config import (BC_OUTFLOW, BC_PERIODIC, BC_REFLECTIVE, HLLC_FLUX, LHLLC_FLUX,
                                   LIM2ND_REC, PPH_REC, PhlxConfig)

pytestmark = pytest.mark.gpu

WALLS = (BC_PERIODIC, BC_PERIODIC, BC_REFLECTIVE, BC_REFLECTIVE, BC_OUTFLOW, BC_OUTFLOW)


def _run(pb, nsteps, fused, graph=False):
    from phlegethon_amd.runtime import Simulation
    sim = Simulation(pb.cfg)
    sim.setup(pb)
    sim.set_fused_sweep(fused)
    sim.set_step_graph(graph)
    sim.init()
    sim.run(nsteps - 2)
    sim.run(2)
    st = sim.download()
    st.update(sim.scalars())
    sim.close()
    return st


@pytest.mark.parametrize("nas", [0, 2])
@pytest.mark.parametrize("shape", [(3, 3, 1), (58, 11, 1), (60, 25, 1), (119, 4, 1), (3, 4, 3),
                                   (57, 10, 15), (59, 13, 31), (17, 23, 34)],
                         ids=lambda s: "x".join(map(str, s)))
def test_flattened_stage(oracle_mod, shape, nas):
    nx, ny, nz = shape
    cfg = PhlxConfig(sdims=2 if nz == 1 else 3, nx1=nx, nx2=ny, nx3=nz, x1u=nx / 32.0,
                     x2u=ny / 32.0, x3u=nz / 32.0, flux=HLLC_FLUX if nx % 2 else LHLLC_FLUX,
                     recon=PPH_REC if ny % 2 else LIM2ND_REC, cfl=0.4, bc=WALLS, nas=nas,
                     shock_flattening=True, eps_sf=0.25).validate()
    pb = P.blast(cfg) if min(shape[:cfg.sdims]) > 4 else P.random_smooth(cfg, amp=0.4)
    r = oracle_mod.OracleRun(pb)
    r.init()
    r.run(5)
    frac = float(r.shock_flags().mean())
    ref = r.state()
    time = r.scalar("time")
    r.close()
    print(f"flag fraction {frac:.3f}", flush=True)
    a = _run(pb, 5, True)
    assert a["time"] == time and np.array_equal(a["prim"], ref["prim"])
    for b in (_run(pb, 5, False), _run(pb, 5, True, graph=True)):
        for k, v in a.items():
            assert np.array_equal(v, b[k]), k
