"""Grid shapes at the edges of the kernels' tilings: rows shorter and longer
than a wave, segments of one face up to the longest, grids smaller than a
block, odd extents on every axis.

FP64 runs meet the parity bar of tests/test_gpu_parity.py against the oracle
(rel. L1 <= 1e-12 per field); mixed runs the 1e-6 bar of
tests/test_gpu_mixed.py (smooth flow at Mach ~0.2, no well-balancing, so the
FP32 fluxes' ~1e-7 is the whole error).
"""
import numpy as np
import pytest

from phlegethon_amd import problems as P
from phlegethon_amd.config import (BC_DIODE, BC_OUTFLOW, BC_PERIODIC, BC_REFLECTIVE, HLLC_FLUX,
                                   HLLD_FLUX, LHLLC_FLUX, LIM2ND_REC, PPH_REC, PREC_FP64, PREC_MIXED,
                                   PhlxConfig)

pytestmark = pytest.mark.gpu

TOL = {PREC_FP64: 1e-12, PREC_MIXED: 1e-6}
WALLS = (BC_PERIODIC, BC_PERIODIC, BC_REFLECTIVE, BC_REFLECTIVE, BC_OUTFLOW, BC_OUTFLOW)

SHAPES = [(2, 2, 1), (3, 130, 1), (65, 4, 1), (101, 93, 1), (2, 2, 2), (63, 5, 3), (65, 9, 26),
          (16, 17, 49), (130, 2, 7)]


def _check(pb, oracle_mod, nsteps=3):
    from phlegethon_amd.runtime import Simulation
    sim = Simulation(pb.cfg)
    sim.setup(pb)
    sim.init()
    sim.run(nsteps)
    got = sim.download()
    got.update(sim.scalars())
    sim.close()
    ref = oracle_mod.run_problem(pb, nsteps, nthreads=8)
    tol = TOL[pb.cfg.precision]
    assert got["step"] == ref["step"] == nsteps
    assert abs(got["time"] - ref["time"]) <= tol * ref["time"]
    # velocities share one scale: a component may start at zero
    vel = np.abs(ref["prim"][1:1 + pb.cfg.sdims]).sum()
    for v in range(pb.cfg.nvars):
        den = vel if 1 <= v <= pb.cfg.sdims else np.abs(ref["prim"][v]).sum()
        err = np.abs(got["prim"][v] - ref["prim"][v]).sum() / den
        assert err <= tol, (v, err)
    if pb.cfg.mhd:
        den = sum(np.abs(ref[f"b_x{d + 1}"]).sum() for d in range(pb.cfg.sdims))
        for d in range(pb.cfg.sdims):
            err = np.abs(got[f"b_x{d + 1}"] - ref[f"b_x{d + 1}"]).sum() / den
            assert err <= tol, (d, err)


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("flux", [LHLLC_FLUX, HLLD_FLUX], ids=["lhllc", "hlld"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_sweep_shapes(oracle_mod, shape, flux, prec):
    nx, ny, nz = shape
    cfg = PhlxConfig(sdims=2 if nz == 1 else 3, nx1=nx, nx2=ny, nx3=nz, x1u=nx / 32.0,
                     x2u=ny / 32.0, x3u=nz / 32.0, flux=flux, cfl=0.4, bc=WALLS,
                     recon=PPH_REC if ny % 2 else LIM2ND_REC, precision=prec).validate()
    _check(P.random_smooth(cfg), oracle_mod)


@pytest.mark.parametrize("shape", [(5, 65, 1), (67, 30, 1), (7, 33, 9)],
                         ids=lambda s: "x".join(map(str, s)))
def test_flattened_sweep_shapes(oracle_mod, shape):
    nx, ny, nz = shape
    cfg = PhlxConfig(sdims=2 if nz == 1 else 3, nx1=nx, nx2=ny, nx3=nz, flux=HLLC_FLUX,
                     recon=PPH_REC, cfl=0.4, bc=WALLS, shock_flattening=True,
                     eps_sf=0.25).validate()
    _check(P.blast(cfg), oracle_mod)


def _state(pb, nsteps, fused, graph=False):
    from phlegethon_amd.runtime import Simulation
    sim = Simulation(pb.cfg)
    sim.setup(pb)
    sim.set_fused_sweep(fused)
    sim.set_step_graph(graph)
    sim.init()
    # two calls: the second starts from whichever buffers the first left
    sim.run(nsteps - 2)
    sim.hydro_step()
    sim.compute_hyperbolic_dt()
    sim.run(2)
    st = sim.download()
    st.update(sim.scalars())
    sim.close()
    return st


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape,rk", [((2, 2, 1), 2), ((17, 16, 1), 3), ((101, 31, 1), 2),
                                      ((2, 3, 2), 2), ((15, 46, 13), 3), ((33, 14, 25), 2)],
                         ids=lambda s: "x".join(map(str, s)) if isinstance(s, tuple) else f"rk{s}")
def test_whole_stage_pass(oracle_mod, shape, rk, prec):
    """Ideal hydro: the one-pass stage equals the separate sweeps and update
    bit for bit on ragged tiles (with WB, gravity, ETOT, heating, diode and
    outflow walls, an odd number of stages), and steps past tmax leave the
    state alone whichever buffer holds it."""
    nx, ny, nz = shape
    base = P.lowmach_box(n=8, mach=1e-2, sdims=2 if nz == 1 else 3).cfg
    walls = (BC_OUTFLOW, BC_OUTFLOW, BC_DIODE, BC_DIODE, BC_PERIODIC, BC_PERIODIC)
    cfg = base.with_(nx1=nx, nx2=ny, nx3=nz, rk_stages=rk, recon=PPH_REC if ny % 2 else LIM2ND_REC,
                     bc=walls, precision=prec, cfl=0.4).validate()
    pb = P.random_smooth(cfg)
    y = np.linspace(0.0, 1.0, ny)
    yf = np.linspace(0.0, 1.0, ny + 1)
    pb.profiles.update(eq_rho_cc=1.0 - 0.2 * y, eq_p_cc=1.0 - 0.1 * y, eq_rho_f=1.0 - 0.2 * yf,
                       eq_p_f=1.0 - 0.1 * yf, grav_cc=np.full(ny, -0.1), phi_cc=0.1 * y,
                       phi_f=0.1 * yf, edot_cc=0.01 * np.sin(6.0 * y))
    for tmax in (1e30, None):
        if tmax is None:
            pb.cfg = cfg.with_(tmax=0.6 * a["time"])
        a, b = _state(pb, 6, True), _state(pb, 6, False)
        c = _state(pb, 6, True, graph=True)
        for other in (b, c):
            for k, v in a.items():
                assert np.array_equal(v, other[k]), k


@pytest.mark.parametrize("prec", [PREC_FP64, PREC_MIXED], ids=["fp64", "mixed"])
def test_ragged_fused_helmholtz(oracle_mod, prec):
    """The FASTEOS slab on tiles that divide neither axis: fused equals
    separate sweeps bit for bit."""
    from phlegethon_amd import helmholtz as H
    table = H.default_table()
    pb = P.helm_slab(oracle_mod.OracleHelm(table), table, n=21, ny=34, sdims=3)
    pb.cfg = pb.cfg.with_(precision=prec)
    a, b = _state(pb, 5, True), _state(pb, 5, False)
    for k, v in a.items():
        assert np.array_equal(v, b[k]), k
