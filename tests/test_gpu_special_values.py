"""Zeros, infinities and subnormal intermediate values in the FP64 kernels
against the oracle's plain IEEE operations, bit for bit (NaN where it has NaN):
EoS targets that no temperature reaches, cells without pressure, opaque cells
of the thermal diffusion, velocities whose squares underflow.
"""
import numpy as np
import pytest

from phlegethon_amd import helmholtz as H
from phlegethon_amd import problems as P
from phlegethon_amd.config import (BC_OUTFLOW, BC_REFLECTIVE, HLLC_FLUX, HLLD_FLUX, LHLLC_FLUX,
                                   LHLLD_FLUX, LIM2ND_REC, PPH_REC, PhlxConfig)

from test_gpu_diffusion import _one_step, _random_T
from test_gpu_parity import TOL, rel_l1

pytestmark = pytest.mark.gpu

WALLS = (0, 0, BC_REFLECTIVE, BC_REFLECTIVE, BC_OUTFLOW, BC_OUTFLOW)


def _equal(a, b):
    return np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("ret", [True, False])
def test_unreachable_eos_targets(oracle_mod, ret):
    """An infinite target takes T out of the table at the first step, which
    resets it to the start value and ends the loop."""
    from phlegethon_amd.runtime import HelmEoS
    table = H.default_table()
    eos, orc = HelmEoS(table), oracle_mod.OracleHelm(table)
    n = 130
    r = np.random.default_rng(5)
    rho, T0 = 10.0 ** r.uniform(2, 8, n), 10.0 ** r.uniform(6, 9, n)
    abar = r.uniform(4, 16, n)
    zbar = 0.5 * abar
    p, e, _, _ = orc.full(rho, T0, abar, zbar)
    for x in (p, e):
        x[0::5] = np.inf
        x[1::5] = -np.inf
        x[2::15] = 0.0
        x[3::15] = np.nan
    try:
        for got, ref in ((eos.rhoe_given(rho, e, abar, zbar, T0, ret),
                          orc.rhoe_given(rho, e, abar, zbar, T0, ret)),
                         (eos.rhoP_given(rho, p, abar, zbar, T0, ret),
                          orc.rhoP_given(rho, p, abar, zbar, T0, ret))):
            for k in (0, 1):
                assert np.array_equal(got[0][k::5], T0[k::5]) and np.all(got[3][k::5] == 1)
            for a, b in zip(got, ref):
                assert _equal(a, b)
    finally:
        eos.close()


def test_eos_of_no_matter_and_no_limit(oracle_mod):
    """rho = 0 (an infinite specific energy and c_v from the radiation), T = 0,
    and infinite ones."""
    from phlegethon_amd.runtime import HelmEoS
    table = H.default_table()
    eos, orc = HelmEoS(table), oracle_mod.OracleHelm(table)
    v = np.array([0.0, 1.0, 1e7, np.inf])
    rho, T = (x.ravel() for x in np.meshgrid(v, v))
    abar, zbar = np.full(rho.size, 12.0), np.full(rho.size, 6.0)
    try:
        got, ref = eos.full(rho, T, abar, zbar), orc.full(rho, T, abar, zbar)
        assert np.any(np.isinf(ref[1])) and np.any(np.isfinite(ref[1]))
        for a, b in zip(got, ref):
            assert _equal(a, b)
    finally:
        eos.close()


def _run_both(pb, oracle_mod, nsteps=1):
    from phlegethon_amd.runtime import Simulation
    out = []
    for fused in (True, False):
        sim = Simulation(pb.cfg)
        sim.setup(pb)
        sim.set_fused_sweep(fused)
        sim.init()
        sim.run(nsteps)
        out.append(sim.download())
        sim.close()
    return out, oracle_mod.run_problem(pb, nsteps)


@pytest.mark.parametrize("sdims", [2, 3])
@pytest.mark.parametrize("flux,recon", [(HLLC_FLUX, LIM2ND_REC), (LHLLC_FLUX, LIM2ND_REC),
                                        (LHLLC_FLUX, PPH_REC), (HLLD_FLUX, LIM2ND_REC),
                                        (LHLLD_FLUX, LIM2ND_REC)])
def test_cells_without_pressure(oracle_mod, flux, recon, sdims):
    """Single cells of zero pressure, at rest and moving: a face with a zero
    sound speed on one side, whose Mach number there is infinite or NaN."""
    cfg = PhlxConfig(sdims=sdims, nx1=32, nx2=21, nx3=10 if sdims == 3 else 1, flux=flux,
                     recon=recon, cfl=0.3, bc=WALLS).validate()
    pb = P.random_smooth(cfg, amp=0.3)
    pb.prim[1:1 + sdims, :, :9, :] = 0.0
    pb.prim[sdims + 1, slice(1, None, 4) if sdims == 3 else 0, 2::4, 2::4] = 0.0
    if pb.b_faces is not None:
        pb.b_faces = [None if b is None else 0.0 * b for b in pb.b_faces]
    got, ref = _run_both(pb, oracle_mod)
    assert np.isfinite(ref["prim"]).mean() > 0.5
    for g in got:
        assert _equal(g["prim"], ref["prim"])


@pytest.mark.parametrize("ratio", [0.7, 40.0])
@pytest.mark.parametrize("sdims", [2, 3])
def test_opaque_cells(oracle_mod, sdims, ratio):
    """Single cells of the largest opacity conduct nothing: rho kappa overflows
    or nearly does, K is zero or subnormal and so is the flux of their faces."""
    cfg = PhlxConfig(sdims=sdims, nx1=20, nx2=16, nx3=12 if sdims == 3 else 1, x1u=1e8, x2u=8e7,
                     x3u=6e7, thermal_diffusion=True)
    pb = _random_T(cfg)
    k = 5 if sdims == 3 else 0
    for i, j in ((3, 4), (9, 9), (15, 6)):
        pb.kappa[k, j + 1, i + 1] = 1.7e308
    got, ref, _ = _one_step(pb, ratio, oracle_mod)
    assert np.all(np.isfinite(ref["eint"]))
    for name in ("eint", "temp"):
        assert rel_l1(got[name], ref[name]) <= TOL, name
        assert got[name][max(k - 1, 0), 4, 3] == ref[name][max(k - 1, 0), 4, 3]


@pytest.mark.parametrize("flux,speed", [(LHLLC_FLUX, 1e-157), (LHLLC_FLUX, 1e-146),
                                        (LHLLD_FLUX, 1e-79), (HLLC_FLUX, 1e-161)])
def test_vanishing_velocities(oracle_mod, flux, speed):
    """Roots of subnormal squares and quotients of subnormal products."""
    cfg = PhlxConfig(sdims=3, nx1=20, nx2=17, nx3=9, flux=flux, recon=LIM2ND_REC, cfl=0.3,
                     bc=WALLS).validate()
    pb = P.random_smooth(cfg, amp=0.3)
    r = np.random.default_rng(2)
    pb.prim[1:4] = speed * r.uniform(-1.0, 1.0, pb.prim[1:4].shape)
    pb.prim[0] = pb.prim[4] = 1.0
    if pb.b_faces is not None:
        pb.b_faces = [0.0 * b for b in pb.b_faces]
    got, ref = _run_both(pb, oracle_mod, 2)
    for g in got:
        assert np.array_equal(g["prim"][0], ref["prim"][0])
        assert np.array_equal(g["prim"][4], ref["prim"][4])
        for v in (1, 2, 3):
            assert np.abs(g["prim"][v] - ref["prim"][v]).max() <= TOL * speed
