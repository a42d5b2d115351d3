"""The layout a per-cell launch takes (cell_lds_layout of hemocell_amd/csrc/hc_lds_plan.h), on the CPU: it follows from the
mesh, not from the spread scratch that the launch asks for, which grows with the layout's room only; what is accepted
with the smallest scratch is accepted with any."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
RBC, PLT, WBC = 0, 1, 2
IN_LDS, AS_DOUBLES, GLOBAL = 0, 1, 2
LEAST = 12288
SCRATCH = [LEAST, 16384, 21504, 24576, 45056, 69632]
SIZES = [12, 66, 162, 227, 228, 455, 642, 1442, 1962, 2190, 2200, 2562, 3600, 3900, 4197, 4269, 4270, 5700, 6200, 10242,
         40962, 45953, 58000, 65534, 70000, 74600]
DEVICE, STATIC, MARGIN = 163840, 1408, 256


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("lds") / "libldslayout.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", out,
                           os.path.join(HERE, "native", "lds_layout_shim.cpp")])
    L = ctypes.CDLL(out)
    i64, c = ctypes.c_int64, ctypes.c_int
    L.layout.argtypes, L.layout.restype = [c, c, c, i64, i64, i64, i64, c, ctypes.POINTER(i64)], None
    L.mech_bytes.argtypes, L.mech_bytes.restype = [c, c, i64], i64
    L.edge_bytes.argtypes, L.edge_bytes.restype = [c, i64], i64
    return L


def _layout(L, model, nv, psize, box, pos):
    out = (ctypes.c_int64 * 7)()
    L.layout(model, nv, int(model != RBC), psize, box, DEVICE, STATIC, pos, out)
    return dict(zip(("ok", "staged", "fixed", "region", "lists", "dyn", "nodes"), (int(v) for v in out)))


@pytest.mark.parametrize("pos", [IN_LDS, AS_DOUBLES, GLOBAL])
@pytest.mark.parametrize("psize", [4, 8])
@pytest.mark.parametrize("model", [RBC, PLT, WBC])
def test_the_layout_follows_from_the_mesh(lib, model, psize, pos):
    for nv in SIZES:
        least = _layout(lib, model, nv, psize, LEAST, pos)
        room = 0
        for box in [6144] + SCRATCH:
            p = _layout(lib, model, nv, psize, box, pos)
            assert p["dyn"] == p["fixed"] + p["region"] + p["lists"]
            if box >= LEAST:
                assert (p["ok"], p["staged"], p["fixed"]) == (least["ok"], least["staged"], least["fixed"]), (nv, box)
            if not p["ok"]:
                continue
            assert p["dyn"] + STATIC + MARGIN <= DEVICE and 24 * p["nodes"] <= p["region"]
            assert p["region"] >= room  # never less for asking more
            room = p["region"]
            free = DEVICE - MARGIN - STATIC - p["dyn"]
            assert p["region"] >= box or free < 16, (nv, box)
            if p["staged"]:
                assert pos != GLOBAL and not (pos == AS_DOUBLES and psize == 4)
                assert p["region"] >= lib.mech_bytes(model, nv, psize)
        if pos == GLOBAL and nv <= 74000:
            assert least["ok"]


@pytest.mark.parametrize("psize", [4, 8])
def test_a_platelets_edge_terms_fit_the_region(lib, psize):
    for nv in (12, 66, 162, 227, 228, 455, 456):
        edges = 6 * (3 * nv - 6) * psize  # of a closed surface without holes
        assert lib.edge_bytes(nv, psize) in (0, 18 * nv * psize)
        assert (lib.edge_bytes(nv, psize) == 0) == (18 * nv * psize > 32768)
        for box in [6144] + SCRATCH:
            p = _layout(lib, PLT, nv, psize, box, IN_LDS)
            assert p["ok"] and p["staged"]
            if lib.edge_bytes(nv, psize):
                assert p["region"] >= edges
