"""A device allocation that fails inside a library call: the call reports it,
later calls see no error of it, and the same call made again gets everything it
needs (phlx_set_thermal_diffusion kept the buffers it had and took the rest
for granted).  Without a GPU, over stand-ins for the HIP calls.
"""
import ctypes
import os
import subprocess
import sys

import pytest

from phlegethon_amd.runtime import LIB_PATH

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
E_NOMEM = -4


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    if not os.path.exists(LIB_PATH):
        pytest.skip("libphlx.so not built (run __graft_entry__.build())")
    so = str(tmp_path_factory.mktemp("hip") / "stub.so")
    subprocess.run(["gcc", "-O1", "-fPIC", "-shared", "-o", so, os.path.join(HERE, "hip_stub.c")],
                   check=True)
    return so


def _child(code, stub):
    env = dict(os.environ, LD_PRELOAD=stub, PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", code, stub], env=env, capture_output=True, text=True,
                       timeout=110)
    assert r.returncode == 0, r.stdout + r.stderr


PRELUDE = """
import ctypes, sys
from phlegethon_amd.config import *
from phlegethon_amd.runtime import load_library
lib, stub = load_library(), ctypes.CDLL(sys.argv[1])
def create(**kw):
    c, ctx = PhlxConfig(sdims=3, nx1=6, nx2=5, nx3=4, **kw).validate().to_c(), ctypes.c_void_p()
    return lib.phlx_create(ctypes.byref(c), ctypes.byref(ctx)), ctx
"""


def test_thermal_diffusion(stub):
    _child(PRELUDE + f"""
for fail in range(5):
    rc, ctx = create()
    assert rc == 0
    n = stub.stub_allocs()
    stub.stub_fail_after(fail)
    assert lib.phlx_set_thermal_diffusion(ctx, 1, 1, None) == {E_NOMEM}
    assert lib.phlx_init(ctx) == 0, fail
    for again in range(2):
        assert lib.phlx_set_thermal_diffusion(ctx, 1, 1, None) == 0
        # kappa, two stages, M e_0, T
        assert stub.stub_allocs() - n == 5, (fail, stub.stub_allocs() - n)
    assert lib.phlx_destroy(ctx) == 0
""", stub)


def test_create(stub):
    _child(PRELUDE + f"""
rc, ctx = create()
for fail in range(10):
    stub.stub_fail_after(fail)
    assert create()[0] == {E_NOMEM}
    assert lib.phlx_init(ctx) == 0, fail
""", stub)
