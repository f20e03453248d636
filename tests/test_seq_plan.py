"""The choices that a portion's kernels are launched with (csrc/seq_plan.hpp), on the host."""
import ctypes
import os
import random
import subprocess

import pytest

from clusterfusionplus_amd import build

CUS, PER_CU, ROOM = 256, 2, 1 << 24
SOURCE = """
#include "seq_plan.hpp"
using namespace cfpp;
extern "C" int attn_splits(int T, int R, int G, int pos0, int chunk, int keys, int bf16, int per_cu, long floats, int cus, long room, int* columns) {
    const AttnPlan p = plan_attn({T, R, G, pos0, chunk, keys, bf16 != 0, per_cu, (size_t)floats}, cus, (size_t)room);
    *columns = p.two ? 128 : 64;
    return p.splits;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{build.CSRC}", str(d / "plan.cpp"), "-o", str(d / "plan.so")], check=True)
    lib = ctypes.CDLL(str(d / "plan.so"))
    lib.attn_splits.argtypes = [ctypes.c_int] * 8 + [ctypes.c_long, ctypes.c_int, ctypes.c_long, ctypes.POINTER(ctypes.c_int)]
    return lib


def splits(plan, T, R, G, pos, chunk, keys=64, room=ROOM, vdim=128):
    columns = ctypes.c_int()
    floats = T * R * G * (vdim + 2)
    n = plan.attn_splits(T, R, G, pos, chunk, keys, keys == 64, PER_CU, floats, CUS, room, ctypes.byref(columns))
    assert 1 <= n <= 16 and (n == 1 or n * floats <= room)
    return n, columns.value


def walks(T, R, pos, chunk, keys, columns):
    """Tiles of keys that every workgroup's columns walk."""
    out = []
    for c0 in range(0, T * R, columns):
        first, last = pos + c0 // R, pos + min(T - 1, (c0 + columns - 1) // R)
        out.append((last + 1 - (first // chunk * chunk if chunk else 0) + keys - 1) // keys)
    return out


@pytest.mark.parametrize("pos, chunk, want", [(8192, 8192, 1), (8193, 8192, 1), (8192 + 219, 8192, 2), (1990, 8192, 16), (8192 + 1990, 8192, 16), (8150, 8192, 16),
                                              (8170, 8192, 16), (0, 0, 1), (1990, 0, 16), (100, 40, 1), (1000, 300, 1)])
def test_splits_follow_what_a_short_portion_sees(plan, pos, chunk, want):
    """37 tokens, four query heads to each of eight key heads: a chunk's first tokens see that chunk only."""
    assert splits(plan, 37, 4, 8, pos, chunk)[0] == want


def test_every_split_of_the_longest_walk_has_two_tiles(plan):
    rng = random.Random(3)
    for _ in range(3000):
        T, R, G = rng.choice([2, 5, 37, 64, 65, 150, 301, 700]), rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 8, 16, 32])
        chunk, keys = rng.choice([0, 1, 7, 100, 1000, 8192]), rng.choice([32, 64])
        pos = rng.randrange(0, 20000)
        n, columns = splits(plan, T, R, G, pos, chunk, keys)
        assert n == 1 or n <= max(walks(T, R, pos, chunk, keys, columns)) // 2, (T, R, G, pos, chunk, keys, n)
