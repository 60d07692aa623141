"""The list room a first construction makes (mdacp_amd/csrc/room.hpp, compiled here for the host) against
the slots that the list of a uniform fluid takes, counted in numpy: rows of each brick by length in
steps of 8, 64 rows to a slice, a slice 64 times its longest row rounded up to 8."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from mdacp_amd.lattice import fcc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SL = 3.0


@pytest.fixture(scope="module")
def expected_slots(tmp_path_factory):
    d = tmp_path_factory.mktemp("room")
    (d / "room.cpp").write_text('#include "room.hpp"\nextern "C" double expected_slots(double rows, double mean, '
                                'double bricks) { return mdgpu::expected_slots(rows, mean, bricks); }\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "mdacp_amd", "csrc"),
                    str(d / "room.cpp"), "-o", str(d / "room.so")], check=True)
    f = ctypes.CDLL(str(d / "room.so")).expected_slots
    f.argtypes, f.restype = [ctypes.c_double] * 3, ctypes.c_double
    return f


def slots_of(q, L, brick):
    from scipy.spatial import cKDTree

    n = cKDTree(q, boxsize=L).query_ball_point(q, SL, return_length=True) - 1
    ms = int(L / SL)
    b = (q * (ms / L)).astype(int) // np.array(brick)
    key = (b[:, 2] * 1000 + b[:, 1]) * 1000 + b[:, 0]
    total = 0
    for k in np.unique(key):
        rows = n[key == k]
        rows = rows[np.argsort(-((rows + 7) // 8), kind="stable")]
        total += sum(64 * ((rows[s:s + 64].max() + 7) // 8 * 8) for s in range(0, len(rows), 64))
    return int(total)


@pytest.mark.parametrize("brick", [(1, 1, 1), (2, 2, 1), (4, 4, 3)])
@pytest.mark.parametrize("rho", [0.3, 0.5, 0.9])
@pytest.mark.parametrize("L", [12.0, 16.0, 30.0])
def test_room_for_the_list_of_a_uniform_fluid(expected_slots, L, rho, brick):
    rng = np.random.default_rng(1)
    q = fcc(L, rho)
    q = np.mod(q + rng.uniform(-0.25, 0.25, q.shape), L)
    need = slots_of(q, L, brick)
    bricks = int(np.prod([-(-int(L / SL) // b) for b in brick]))
    room = expected_slots(len(q), len(q) / L ** 3 * 4.0 / 3.0 * np.pi * SL ** 3, bricks)
    print(len(q), brick, need, room)
    assert need <= room <= 3 * need + 65536
