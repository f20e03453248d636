"""csrc/seq_plan.hpp compiled for the host: what a portion's kernels are launched with on a card of 256 compute units."""
import ctypes
import functools
import os
import subprocess
import tempfile

from clusterfusionplus_amd import build

CUS = 256
SOURCE = """
#include "seq_plan.hpp"
using namespace cfpp;
static int code(int shape, int splits, bool bf16) { const GemmShape& s = shapes_of(bf16)[shape]; return ((s.rows * 1024 + s.tokens) * 4 + s.resident) * 32 + splits; }
extern "C" int attn(int T, int R, int G, int pos0, int chunk, int keys, int bf16, int per_cu, long floats, int cus, long room, int* columns, int* up, int* swap) {
    const AttnPlan p = plan_attn({T, R, G, pos0, chunk, keys, bf16 != 0, per_cu, (size_t)floats}, cus, (size_t)room);
    *columns = p.two ? 128 : 64;
    *up = p.up;
    *swap = p.swap;
    return p.splits;
}
extern "C" int block(int row, int rows, int up, int swap) { return attn_block(row, rows, up, swap); }
extern "C" int product(int n, int m, int kbytes, int ldy, long room, int bf16, int cus) {
    const GemmPlan p = plan_gemm({n, m, kbytes, ldy, (size_t)room}, bf16 != 0, cus);
    return code(p.shape, p.splits, bf16);
}
extern "C" int experts(int n, int top, int experts, int ff, int xbytes, int bf16, int cus, int* once) {
    const ExpertPlan p = plan_experts({n, top, experts, ff, xbytes}, bf16 != 0, cus);
    *once = p.once;
    return code(p.shape, 1, bf16);
}
extern "C" int beside(int n, int top, int experts, int ff, int xbytes, int rows, int kbytes, int shared_rows, int shared_kbytes, int ldy, long room, int bf16, int cus) {
    const ExpertSizes e{n, top, experts, ff, xbytes};
    return plan_beside(e, plan_experts(e, bf16 != 0, cus), rows, kbytes, {shared_rows, n, shared_kbytes, ldy, (size_t)room}, bf16 != 0, cus);
}
extern "C" int turn(int n, int pos, int heads, int dim, int rot, int vdim, int kbytes, int rank, int bf16, long room, int cus, int* sets, int* tokens) {
    const LatentTurn t = plan_latent_turn({n, pos, heads, dim, rot, vdim, kbytes, rank, bf16 != 0, (size_t)room}, cus);
    *sets = t.sets;
    *tokens = t.tokens;
    return t.splits;
}
extern "C" int tile(int shape, int bf16) { return code(shape, 1, bf16 != 0); }
extern "C" float estimate(int n, int m, int kbytes, int shape, int splits, int bf16, int cus) { return gemm_cost({n, m, kbytes, n, 0}, shapes_of(bf16)[shape], splits, cus); }
"""


@functools.lru_cache(maxsize=None)
def lib():
    with tempfile.TemporaryDirectory() as d:
        src, so = os.path.join(d, "plan.cpp"), os.path.join(d, "plan.so")
        with open(src, "w") as f:
            f.write(SOURCE)
        subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{build.CSRC}", src, "-o", so], check=True)
        lib = ctypes.CDLL(so)
    i, l, p = ctypes.c_int, ctypes.c_long, ctypes.POINTER(ctypes.c_int)
    lib.attn.argtypes = [i] * 8 + [l, i, l, p, p, p]
    lib.block.argtypes = [i] * 4
    lib.product.argtypes = [i] * 4 + [l, i, i]
    lib.experts.argtypes = [i] * 7 + [p]
    lib.beside.argtypes = [i] * 10 + [l, i, i]
    lib.turn.argtypes = [i] * 9 + [l, i, p, p]
    lib.tile.argtypes = [i, i]
    lib.estimate.argtypes, lib.estimate.restype = [i] * 7, ctypes.c_float
    return lib


def attention(T, R, G, pos, chunk, keys, floats, room, per_cu=2):
    """(splits of the keys, columns of a workgroup)"""
    return attention_plan(T, R, G, pos, chunk, keys, floats, room, per_cu)[:2]


def attention_plan(T, R, G, pos, chunk, keys, floats, room, per_cu=2):
    """(splits of the keys, columns of a workgroup, blocks of columns in the order of the workgroups' rows)"""
    columns, up, swap = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    splits = lib().attn(T, R, G, pos, chunk, keys, keys == 64, per_cu, floats, CUS, room, ctypes.byref(columns), ctypes.byref(up), ctypes.byref(swap))
    rows = -(-T * R // columns.value)
    return splits, columns.value, [lib().block(row, rows, up.value, swap.value) for row in range(rows)]


def _decode(code):
    """(rows, tokens, workgroups per compute unit, splits of k)"""
    return code // (32 * 4 * 1024), code // (32 * 4) % 1024, code // 32 % 4, code % 32


def tile(shape, bf16):
    return _decode(lib().tile(shape, bf16))[:3]


def row_bytes(k, bf16):
    return (k * (2 if bf16 else 4) + 127) // 128 * 128


def room(portion, width):
    """Floats behind a product of `width` rows for partial results, in a model with passes of `portion` tokens."""
    floats = portion * ((width + 3) // 4 * 4)
    return max(floats, min(8 * floats, 16 << 20))


def product(n, m, k, bf16, floats=0):
    """Tile and splits of a product of n rows of k values with m tokens, with room for so many floats of partial results."""
    return _decode(lib().product(n, m, row_bytes(k, bf16), n, floats, bf16, CUS))


def experts(n, top, count, ff, width, bf16):
    """Tile of the products of `count` experts of which every one of n tokens takes `top`, and whether an expert's tokens fit one."""
    once = ctypes.c_int()
    return _decode(lib().experts(n, top, count, ff, row_bytes(width, bf16), bf16, CUS, ctypes.byref(once)))[:3] + (bool(once.value),)


def turn(n, pos, mixer, bf16, floats):
    """Splits (0: keys and values are made), sets of columns in a block, and the merge's tokens of a portion of n tokens at pos with latent attention."""
    m, out = mixer, [ctypes.c_int() for _ in range(2)]
    splits = lib().turn(n, pos, m["heads"], m["dim"], m["rot_dim"], m["vdim"], row_bytes(m["kv_rank"], bf16), (m["kv_rank"] + 15) // 16 * 16, bf16, floats, CUS,
                        *map(ctypes.byref, out))
    return (splits, *(x.value for x in out))
