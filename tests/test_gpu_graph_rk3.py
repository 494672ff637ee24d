"""Captured RK3 steps of whole-stage passes (phlx_set_step_graph): each step
ends in the other primitive buffer, so two graphs alternate.  Bit for bit the
eager launches, in chunks of odd and even length with eager steps, downloads
and changes of the sweep form between them; and in about the eager launches'
time, not the separate sweeps'.
"""
import time

import numpy as np
import pytest

from phlegethon_amd import problems as P
from phlegethon_amd.config import (HLLC_FLUX, LHLLC_FLUX, LIM2ND_REC, PREC_FP64, PREC_MIXED,
                                   PhlxConfig)

pytestmark = pytest.mark.gpu


def _problem(shape, prec, flux=LHLLC_FLUX, **kw):
    nx, ny, nz = shape
    cfg = PhlxConfig(sdims=2 if nz == 1 else 3, nx1=nx, nx2=ny, nx3=nz, rk_stages=3, flux=flux,
                     recon=LIM2ND_REC, cfl=0.4, precision=prec, **kw).validate()
    return P.random_smooth(cfg)


def _states(pb, graph):
    from phlegethon_amd.runtime import Simulation
    sim = Simulation(pb.cfg)
    sim.setup(pb)
    sim.set_step_graph(graph)
    sim.init()
    out = []
    for n, fused in ((1, None), (2, None), (3, False), (3, None), (5, None)):
        sim.set_fused_sweep(fused)
        sim.run(n)
        if n == 2:
            sim.hydro_step()
            sim.compute_hyperbolic_dt()
        st = sim.download()
        st.update(sim.scalars())
        out.append(st)
    sim.close()
    return out


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(37, 20, 1), (32, 15, 11)], ids=lambda s: "x".join(map(str, s)))
def test_bitwise(shape, prec):
    pb = _problem(shape, prec)
    for a, b in zip(_states(pb, False), _states(pb, True)):
        for k, v in a.items():
            assert np.array_equal(v, b[k]), k


def test_bitwise_flattened():
    pb = _problem((33, 17, 14), PREC_FP64, HLLC_FLUX, shock_flattening=True, eps_sf=0.05)
    for a, b in zip(_states(pb, False), _states(pb, True)):
        for k, v in a.items():
            assert np.array_equal(v, b[k]), k


def test_captured_form():
    """128^3, best of 6 runs of 10 steps each way in turn: the separate sweeps
    take more than 1.3 times as long."""
    from phlegethon_amd.runtime import Simulation
    best = {}
    sims = {}
    for graph in (False, True):
        sim = Simulation(_problem((128, 128, 128), PREC_FP64).cfg)
        sim.setup(_problem((128, 128, 128), PREC_FP64))
        sim.set_step_graph(graph)
        sim.init()
        sim.run(4)
        sim.synchronize()
        sims[graph] = sim
    for _ in range(6):
        for graph, sim in sims.items():
            t = time.perf_counter()
            sim.run(10)
            sim.synchronize()
            t = time.perf_counter() - t
            best[graph] = min(best.get(graph, t), t)
    for sim in sims.values():
        sim.close()
    print(f"eager {best[False] * 1e5:.1f} us/step, captured {best[True] * 1e5:.1f}", flush=True)
    assert best[True] < 1.15 * best[False]
