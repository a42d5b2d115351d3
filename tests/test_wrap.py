"""Node coordinates on periodic axes (hemocell_amd/csrc/hc_wrap.h) for positions of any finite size, on the CPU: the wall
contact of a vertex reads the type of the node they name, so they have to lie on the axis."""
import ctypes
import math
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("wrap") / "libwrap.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-o", out,
                           os.path.join(HERE, "native", "wrap_shim.cpp")])
    L = ctypes.CDLL(out)
    for f in (L.wrap_node, L.wrap_far):
        f.argtypes, f.restype = [ctypes.c_double, ctypes.c_int], ctypes.c_int
    return L


@pytest.mark.parametrize("n", [1, 2, 3, 50, 97, 256, 1291, 2 ** 31 - 1])
def test_any_finite_node(lib, n):
    rng = random.Random(n)
    edges = [0, 1, n - 1, n, n + 1, 2 ** 52, 2 ** 53 - 1, 2 ** 53, 2 ** 53 + 2, 10 ** 16, 2 ** 62, 2 ** 63, 2 ** 64]
    far = [math.floor(10.0 ** rng.uniform(0, 308)) for _ in range(3000)]
    for fl in edges + far + [1.7976931348623157e308]:
        for x in (float(fl), -float(fl)):
            assert lib.wrap_far(x, n) == int(x) % n, (x, n)
            assert abs(x) > 2.0 ** 52 or lib.wrap_node(x, n) == int(x) % n, (x, n)
    for x in (math.inf, -math.inf, math.nan):
        lib.wrap_far(x, n)  # no node, but it returns
