"""The FP64 kernels' own quotients, square roots and table-cell lookup
(Recip, dsqrt, helm_index in phlx_helm.hpp) give the bits of the IEEE
operations and of the FP64 log10 form: runs and batch calls equal the CPU
oracle, which uses those, bit for bit.
"""
import numpy as np
import pytest

from phlegethon_amd import helmholtz as H
from phlegethon_amd import problems as P
from phlegethon_amd.config import (HLLC_FLUX, HLLD_FLUX, LHLLC_FLUX, LHLLD_FLUX, LIM2ND_REC,
                                   PhlxConfig)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flux", [HLLC_FLUX, LHLLC_FLUX, HLLD_FLUX, LHLLD_FLUX])
@pytest.mark.parametrize("scale", [1.0, 1e-30, 1e30], ids=["unit", "small", "large"])
def test_solvers_bitwise(oracle_mod, flux, scale):
    """Density and pressure (and the field's square) scaled together: the same
    flow with every quotient and root at another exponent."""
    from phlegethon_amd.runtime import Simulation
    cfg = PhlxConfig(sdims=3, nx1=37, nx2=22, nx3=19, flux=flux, recon=LIM2ND_REC).validate()
    pb = P.random_smooth(cfg, amp=0.6)
    pb.prim[0] *= scale
    pb.prim[4] *= scale
    pb.prim[1:4, 3:9] = 0.0  # a gas at rest: roots and quotients of zero
    if pb.b_faces is not None:
        pb.b_faces = [b * np.sqrt(scale) for b in pb.b_faces]
    sim = Simulation(cfg)
    sim.setup(pb)
    sim.init()
    sim.run(4)
    got = sim.download()
    got.update(sim.scalars())
    sim.close()
    ref = oracle_mod.run_problem(pb, 4, nthreads=8)
    assert got["time"] == ref["time"] and got["dt"] == ref["dt"]
    assert np.array_equal(got["prim"], ref["prim"])
    if pb.b_faces is not None:
        for d in range(3):
            assert np.array_equal(got[f"b_x{d + 1}"], ref[f"b_x{d + 1}"])


@pytest.fixture(scope="module")
def eos_pair(oracle_mod):
    from phlegethon_amd.runtime import HelmEoS
    table = H.default_table()
    eos = HelmEoS(table)
    yield eos, oracle_mod.OracleHelm(table), table
    eos.close()


@pytest.mark.parametrize("n", [1, 63, 257, 20000])
def test_eos_batch_bitwise(eos_pair, n):
    eos, orc, _ = eos_pair
    r = np.random.default_rng(n)
    rho, T = 10.0 ** r.uniform(-2, 9, n), 10.0 ** r.uniform(5, 9.5, n)
    abar = r.uniform(4, 16, n)
    zbar = abar * r.uniform(0.45, 0.5, n)
    full = orc.full(rho, T, abar, zbar)
    for a, b in zip(eos.full(rho, T, abar, zbar), full):
        assert np.array_equal(a, b)
    T0 = T * r.uniform(0.9, 1.1, n)  # leaves the cell in most solves
    for a, b in zip(eos.rhoe_given(rho, full[1], abar, zbar, T0),
                    orc.rhoe_given(rho, full[1], abar, zbar, T0)):
        assert np.array_equal(a, b)
    for a, b in zip(eos.rhoP_given(rho, full[0], abar, zbar, T0),
                    orc.rhoP_given(rho, full[0], abar, zbar, T0)):
        assert np.array_equal(a, b)


def test_cell_lookup_beside_nodes(eos_pair):
    """Points within the estimate's doubt of a node take the FP64 logarithm;
    points just outside it the estimate: both sides of both limits, bit for bit
    where the distance from the node exceeds the rounding of log10 itself
    (which may fall to either cell on either machine; there the two cells'
    interpolants agree to third order in the distance)."""
    eos, orc, t = eos_pair
    i = np.arange(1, t.nrho - 1, 7)
    j = np.arange(1, t.nT - 1, 5)
    for d in (0.0, 1e-9, 4e-7, 6e-7, 2e-6, 1e-4):
        for sx, sy in ((1, 1), (-1, 1), (1, -1), (-1, -1)):
            rho = (t.rho_nodes[i] * 10.0 ** (sx * d))[:, None] * np.ones(j.size)
            T = np.ones(i.size)[:, None] * (t.T_nodes[j] * 10.0 ** (sy * d))
            rho, T = rho.ravel(), T.ravel()
            one = np.ones_like(rho)
            a, b = eos.full(rho, T, one, one), orc.full(rho, T, one, one)
            for x, y in zip(a[:2], b[:2]):
                if d > 0.0:
                    assert np.array_equal(x, y)
                else:
                    assert np.max(np.abs(x - y) / np.abs(y)) < 1e-6
