"""The mixed Helmholtz update is built once per EoS solve: the surrogate's
start alone, or the form that also counts iterations.  Both make the same
solve, so a run is the same bit for bit with and without the counting, in the
split and in the swept update, with and without a field.
"""
import os
import tempfile

import numpy as np
import pytest

from phlegethon_amd import helmholtz as H
from phlegethon_amd import problems as P
from phlegethon_amd.config import PREC_MIXED

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def slab_table():
    p = os.path.join(tempfile.mkdtemp(), "t.bin")
    H.generate(141, 81, 0.0, 7.0, 6.0, 6.0 + 80 * 10.0 / 270.0, path=p)
    return H.load(p)


@pytest.mark.parametrize("beta", [None, 1e5], ids=["hydro", "mhd"])
@pytest.mark.parametrize("fused", [False, True], ids=["split", "fused"])
def test_surrogate_start_with_and_without_counting(oracle_mod, slab_table, beta, fused):
    import mlp_oracle as M
    from phlegethon_amd.runtime import Simulation
    orc = oracle_mod.OracleHelm(slab_table)
    pb = P.helm_slab(orc, slab_table, n=64, ny=8, sdims=3, mhd_beta=beta)
    theta = M.init_params(5).astype(np.float32)
    norm = np.array([3.5, 15.0, 10.0, 5.0, 0.3, 0.2, 0.15, 0.3, 7.5, 1.4], dtype=np.float32)
    got = []
    for count in (False, True):
        sim = Simulation(pb.cfg.with_(precision=PREC_MIXED))
        sim.setup(pb)
        sim.mlp_set_params(theta, norm)
        sim.set_eos_guess("mlp", count=count)
        sim.set_fused_sweep(fused)
        sim.init()
        sim.run(4)
        st = sim.download()
        st.update(sim.scalars())
        if count:
            assert sim.eos_stats()["solves"] == 2 * 4 * 64 * 8 * 64
        sim.close()
        got.append(st)
    a, b = got
    assert a["step"] == b["step"] == 4 and a["time"] == b["time"] and a["dt"] == b["dt"]
    assert np.array_equal(a["prim"], b["prim"])
    assert np.array_equal(a["temp"], b["temp"])
    for d in range(3 if beta else 0):
        assert np.array_equal(a[f"b_x{d + 1}"], b[f"b_x{d + 1}"])
