"""Host replay of the schedule of regions on levels: every dependency is in a
level group's LDS ring, or in memory behind a barrier that waits for stores,
before its reader's level starts; in spread levels it is a row of a level
launched before (tests/schedule_replay.cpp)."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import test_level_sweeps as ls

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "multiregionfoam_amd", "csrc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("schedule") / "libschedule.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", so, os.path.join(HERE, "schedule_replay.cpp"),
                    *(os.path.join(CSRC, f) for f in ("layout.cpp", "case_builder.cpp", "dictionary.cpp"))], check=True)
    return C.CDLL(so)


def replay(lib, R, waves, no_waits=0):
    out, why = (C.c_longlong * 5)(), C.create_string_buffer(200)
    p = lambda a: a.ctypes.data_as(C.POINTER(C.c_int32))  # noqa: E731
    rc = lib.replay(R["nCells"], R["nFaces"], p(R["lAddr"]), p(R["uAddr"]), waves, no_waits, out, why, len(why))
    return rc, why.value.decode(), dict(zip(("ring", "far", "barriers", "stored", "spread"), out))


@pytest.mark.parametrize("waves", [1, 3, 16])
@pytest.mark.parametrize("name", list(ls.CASES))
def test_dependencies_are_where_their_codes_say(lib, name, waves):
    regions = ls.CASES[name]()
    kinds = ls.KINDS.get(name, ["levels"] * len(regions))
    for R, kind in zip(regions, kinds):
        rc, why, n = replay(lib, R, waves)
        if kind not in ("levels", "spread"):
            assert rc == 2 and why == "no levels: " + kind
            continue
        assert rc == 0, why
        assert (n["spread"] > 0) == (kind == "spread")
        # barriers that wait for stores: none without far rows, and no more
        # than two for each ring of rows in either direction (or one a level)
        rows = 64 * -(-R["nCells"] // 64) + 64 * n["barriers"] // 2
        assert n["stored"] <= (min(n["barriers"], 4 * (rows // 16384) + 2) if n["far"] else 0)


def test_far_rows_of_narrow_levels_are_reached(lib):
    # levels far narrower than the ring, and rows far beyond it: none of them
    # may rest on how long ago they were stored
    for R in ls.CASES["far_rows_of_narrow_levels"]():
        rc, why, n = replay(lib, R, 16)
        assert rc == 0 and n["far"] > 1000 and n["stored"] >= 2
        rc, why, n = replay(lib, R, 16, no_waits=1)
        assert rc == 1 and why.startswith("far row not in memory yet")
