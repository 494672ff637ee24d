"""The diffusion's stages keep e_0 in place and alternate two buffers, the first
takes T from p or from the last step's array and the last one ends the step: two
steps in a row, with odd and even stage counts, on grids that no block divides
and next to every kind of wall, equal the CPU oracle bit for bit.
"""
import numpy as np
import pytest

from phlegethon_amd.config import BC_OUTFLOW, BC_REFLECTIVE, PhlxConfig

from test_gpu_diffusion import _random_T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ratio,stages", [(0.5, 3), (5.0, 5), (8.0, 6), (12.0, 7)])
@pytest.mark.parametrize("dims", [(67, 9, 1), (33, 21, 1), (35, 10, 7), (130, 5, 4)])
def test_two_steps_bitwise(oracle_mod, dims, ratio, stages):
    from phlegethon_amd.runtime import Simulation
    sdims = 3 if dims[2] > 1 else 2
    bc = (BC_REFLECTIVE, BC_OUTFLOW, 0, 0, BC_OUTFLOW, BC_REFLECTIVE) if sdims == 3 else \
        (0, 0, BC_OUTFLOW, BC_REFLECTIVE, 0, 0)
    fix = (None, 1.2e7, None, None, 0.9e7, None) if sdims == 3 else \
        (None, None, 1.1e7, None, None, None)
    cfg = PhlxConfig(sdims=sdims, nx1=dims[0], nx2=dims[1], nx3=dims[2], x1u=1e8, x2u=8e7,
                     x3u=6e7, bc=bc, thermal_diffusion=True, fix_temperature=fix)
    pb = _random_T(cfg, amp=0.02)
    r = oracle_mod.OracleRun(pb)
    r.init()
    dtp = r.parabolic_dt()
    r.set_scalar("dt", ratio * dtp)
    sim = Simulation(cfg)
    sim.setup(pb)
    sim.init()
    assert sim.parabolic_dt() == dtp
    sc = sim.scalars()
    sim.set_scalars(sc["time"], ratio * dtp, sc["smax"], sc["step"])
    for n in (1, 2):
        r.diffusion_step(n)
        sim.diffusion_step(n)
        assert sim.diffusion_stages() == stages
        got, ref = sim.download(), r.state()
        for name in ("eint", "temp", "prim"):
            assert np.array_equal(got[name], ref[name]), (n, name)
    sim.close()
    r.close()


@pytest.mark.parametrize("dims", [(33, 9, 1601), (64, 16, 1024)])
def test_marching_chunks_bitwise(oracle_mod, dims):
    """3D grids large enough for chunks of two and three planes, the last one
    short: the carried x3 flux and the prefetched planes, walls and wraps."""
    from phlegethon_amd.runtime import Simulation
    wall = dims[0] % 2 == 1
    bc = (BC_REFLECTIVE, BC_OUTFLOW, 0, 0, BC_OUTFLOW, BC_REFLECTIVE) if wall else (0,) * 6
    fix = (None, 1.2e7, None, None, 0.9e7, None) if wall else None
    cfg = PhlxConfig(sdims=3, nx1=dims[0], nx2=dims[1], nx3=dims[2], x1u=1e8, x2u=8e7, x3u=1e9,
                     bc=bc, thermal_diffusion=True, fix_temperature=fix)
    pb = _random_T(cfg, amp=0.02)
    r = oracle_mod.OracleRun(pb)
    r.init()
    dtp = r.parabolic_dt()
    r.set_scalar("dt", 5.0 * dtp)
    sim = Simulation(cfg)
    sim.setup(pb)
    sim.init()
    sc = sim.scalars()
    assert sim.parabolic_dt() == dtp
    sim.set_scalars(sc["time"], 5.0 * dtp, sc["smax"], sc["step"])
    r.diffusion_step(1)
    sim.diffusion_step(1)
    got, ref = sim.download(), r.state()
    sim.close()
    r.close()
    for name in ("eint", "temp", "prim"):
        assert np.array_equal(got[name], ref[name]), name
