"""3D Helmholtz runs without FASTEOS, whose column sweeps (a T(rho, P) Newton per
face state) number the columns flat, so that a wave holds cells of several rows:
with and without shock flattening, at the parity bar of
tests/test_gpu_flattening.py against the oracle.
"""
import numpy as np
import pytest

from phlegethon_amd import helmholtz as H
from phlegethon_amd import problems as P
from phlegethon_amd.config import HLLC_FLUX, LHLLC_FLUX, LIM2ND_REC, PPH_REC

from test_gpu_parity import TOL

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def table(tmp_path_factory):
    p = str(tmp_path_factory.mktemp("helm_sf3") / "t.bin")
    H.generate(141, 81, 0.0, 7.0, 6.0, 6.0 + 80 * 10.0 / 270.0, path=p)
    return H.load(p)


@pytest.mark.parametrize("sf", [True, False], ids=["flattened", "plain"])
@pytest.mark.parametrize("recon,flux,beta,n,ny", [
    (LIM2ND_REC, LHLLC_FLUX, None, 21, 24), (PPH_REC, HLLC_FLUX, None, 13, 33),
    (PPH_REC, LHLLC_FLUX, None, 70, 24), (LIM2ND_REC, LHLLC_FLUX, 1e3, 11, 24),
    (PPH_REC, LHLLC_FLUX, 1e3, 19, 24)],
    ids=["lim2nd", "pph", "pph-wide", "lim2nd-mhd", "pph-mhd"])
def test_face_newton_3d(table, oracle_mod, recon, flux, beta, n, ny, sf):
    from phlegethon_amd.runtime import Simulation
    pb = P.helm_slab(oracle_mod.OracleHelm(table), table, n=n, ny=ny, sdims=3, recon=recon,
                     flux=flux, mhd_beta=beta, fasteos=False)
    if n > 64:   # a thinner box of the same rows
        pb.cfg = pb.cfg.with_(nx3=5, x3u=pb.cfg.x3u * 5 / n)
        pb.prim, pb.temp = pb.prim[:, :5].copy(), pb.temp[:5].copy()
    pb.prim[4][..., n // 3: 2 * n // 3] *= 5.0
    if sf:
        pb.cfg = pb.cfg.with_(shock_flattening=True, eps_sf=1.5)
        r = oracle_mod.OracleRun(pb)
        frac = float(r.shock_flags().mean())
        r.close()
        print(f"flag fraction {frac:.3f}", flush=True)
        assert 0.05 < frac < 0.95
    sim = Simulation(pb.cfg)
    sim.setup(pb)
    sim.init()
    sim.run(4)
    got = sim.download()
    got.update(sim.scalars())
    sim.close()
    ref = oracle_mod.run_problem(pb, 4, nthreads=8)
    assert got["step"] == ref["step"] == 4
    assert abs(got["time"] - ref["time"]) <= 1e-14 * abs(ref["time"])
    for v in range(pb.cfg.nvars):
        a, b = got["prim"][v], ref["prim"][v]
        r = np.abs(a - b).sum() / max(np.abs(b).sum(), 1e-300)
        assert r <= TOL, (v, r)
    np.testing.assert_allclose(got["temp"], ref["temp"], rtol=1e-11)
