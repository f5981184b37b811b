"""The rules that choose a call's kernel form (csrc/dispatch.hpp, built here
for the host exactly as the launchers include it)."""
import ctypes
import shutil
import subprocess
from collections import namedtuple
from pathlib import Path

import pytest
from scipy import stats

ROOT = Path(__file__).resolve().parent
Plan = namedtuple("Plan", "tile_rows gate_up_shape down_shape glu chunk blocks stream")


def build_rules(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    so = tmp_path_factory.mktemp("dispatch") / "libdispatch.so"
    subprocess.run([gxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-o", str(so),
                    str(ROOT / "native" / "dispatch_host.cpp")], check=True)
    lib = ctypes.CDLL(str(so))
    lib.expected_tiles.argtypes = [ctypes.c_int64, ctypes.c_int32, ctypes.c_int]
    lib.expected_tiles.restype = ctypes.c_double
    lib.grouped_plan.argtypes = [ctypes.c_int64] + [ctypes.c_int32] * 4 + [ctypes.c_void_p]
    return lib


def grouped_plan(rules, tokens, E, top_k, hidden, inter, tiled=True):
    out = (ctypes.c_int32 * 7)()
    rules.grouped_plan(tokens * top_k, E, hidden, inter, int(tiled), out)
    return Plan(*out)


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    return build_rules(tmp_path_factory)


@pytest.mark.parametrize("P,E", [(1, 256), (232, 256), (8168, 256), (32768, 256), (90, 4),
                                 (5000, 6), (900, 1)])
@pytest.mark.parametrize("rows", [16, 32, 64])
def test_expected_tiles_is_the_poisson_expectation(rules, P, E, rows):
    lam = P / E
    n = int(lam + 12 * lam ** 0.5 + 40)
    want = E * sum(stats.poisson.pmf(k, lam) * -(-k // rows) for k in range(n))
    assert rules.expected_tiles(P, E, rows) == pytest.approx(want, rel=1e-6)
