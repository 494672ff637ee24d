"""2D ideal MHD: the fused sweep on any extents and the one-pass constrained
transport.  FP64 runs equal the CPU oracle bit for bit; fused, split and captured
runs, FP64 and mixed, equal each other, and steps past tmax leave both face
buffers with the current field.
"""
import numpy as np
import pytest

from phlegethon_amd import problems as P
from phlegethon_amd.config import (BC_OUTFLOW, BC_PERIODIC, BC_REFLECTIVE, HLLD_FLUX, LHLLD_FLUX,
                                   LIM2ND_REC, PPH_REC, PREC_FP64, PREC_MIXED, PhlxConfig)

pytestmark = pytest.mark.gpu

WALLS = [(BC_PERIODIC, BC_PERIODIC, BC_REFLECTIVE, BC_REFLECTIVE, 0, 0),
         (BC_REFLECTIVE, BC_OUTFLOW, BC_PERIODIC, BC_PERIODIC, 0, 0)]


def _run(pb, fused, graph=False):
    from phlegethon_amd.runtime import Simulation
    sim = Simulation(pb.cfg)
    sim.setup(pb)
    sim.set_fused_sweep(fused)
    sim.set_step_graph(graph)
    sim.init()
    sim.run(3)
    sim.hydro_step()
    sim.compute_hyperbolic_dt()
    sim.run(2)
    st = sim.download()
    st.update(sim.scalars())
    st["divb"] = sim.divb_max()
    sim.close()
    return st


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("walls", WALLS, ids=["walls2", "walls1"])
@pytest.mark.parametrize("shape,rk", [((2, 2), 2), ((3, 2), 3), ((16, 15), 2), ((17, 31), 3),
                                      ((65, 16), 2), ((130, 61), 3)],
                         ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else f"rk{s}")
def test_fused_equals_split_equals_oracle(oracle_mod, shape, rk, walls, prec):
    nx, ny = shape
    cfg = PhlxConfig(sdims=2, nx1=nx, nx2=ny, nx3=1, x1u=nx / 32.0, x2u=ny / 32.0,
                     flux=HLLD_FLUX if ny % 2 else LHLLD_FLUX, rk_stages=rk, cfl=0.4, bc=walls,
                     recon=PPH_REC if nx % 2 else LIM2ND_REC, precision=prec).validate()
    pb = P.random_smooth(cfg)
    for tmax in (1e30, None):
        if tmax is None:
            pb.cfg = cfg.with_(tmax=0.5 * a["time"])
        a = _run(pb, True)
        for b in (_run(pb, False), _run(pb, True, graph=True)):
            for k, v in a.items():
                assert np.array_equal(v, b[k]), k
        if tmax and prec == PREC_FP64:
            r = oracle_mod.OracleRun(pb)
            r.init()
            r.run(3)
            ref3 = r.state()
            r.close()
            from phlegethon_amd.runtime import Simulation
            sim = Simulation(pb.cfg)
            sim.setup(pb)
            sim.init()
            sim.run(3)
            got = sim.download()
            sim.close()
            for k in ("prim", "b_x1", "b_x2"):
                assert np.array_equal(got[k], ref3[k]), k
