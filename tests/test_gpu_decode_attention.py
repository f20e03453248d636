"""Attention of one token: rows that fill a tile's columns and rows that do not, at the edges of tiles, waves and splits."""
import functools

import pytest
import torch

from tests import nibotar_models as M
from tests.test_gpu_nibotar import DTYPES, IDS, LIMIT, build

pytestmark = pytest.mark.gpu
# heads, key / value heads, key and value dims
SHAPES = {"64": (4, 2, 64, 64), "48_40": (6, 2, 48, 40), "128": (4, 1, 128, 128), "128_tail": (3, 3, 100, 128), "20_heads": (20, 1, 96, 80),
          "256": (2, 1, 256, 256), "200_256": (2, 2, 200, 256)}


@functools.lru_cache(maxsize=None)
def reference(shape, n):
    heads, kv, dim, vdim = SHAPES[shape]
    cfg = M.model(64, 97, [(M.attn(heads, kv, dim, vdim), M.dense(64)), (M.attn(heads, kv, dim, vdim, v_mix=True), M.dense(64))])
    w, toks = M.weights(cfg, 5), M.prompt(cfg, n, 6)
    return cfg, w, toks, M.oracle(cfg, w, toks)


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("shape", list(SHAPES))
def test_steps_at_the_edges(shape, dtype):
    """Steps at the first positions, at tiles of 16 and 32 keys and at the first position of a second split, behind what a portion left."""
    cfg, w, toks, want = reference(shape, 131)
    m = build(cfg, w, dtype)
    for first in (0, 15, 31, 63, 127):
        if first:
            m.forward(0, toks[:first], 0, [first - 1])
        got = torch.cat([m.forward(0, [toks[i]], i, [0]) for i in range(first, first + 4)])
        assert M.error(got, want[first:first + 4]) < LIMIT[dtype], f"from position {first}"


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
def test_more_splits_than_travel_together(dtype):
    cfg, w, toks, want = reference("128", 4198)
    m = build(cfg, w, dtype, capacity=4300, max_portion=4300)
    m.forward(0, toks[:4195], 0, [4194])
    got = torch.cat([m.forward(0, [toks[i]], i, [0]) for i in range(4195, 4198)])
    assert M.error(got, want[4195:]) < LIMIT[dtype]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("heads, dim, vdim", [(128, 24, 20), (128, 72, 88), (128, 136, 72)], ids=str)
def test_several_tiles_per_wave(heads, dim, vdim, dtype):
    """So many heads that the keys are in few splits: every wave goes on to further tiles, the last of them short, in rows that do not fill the columns."""
    cfg = M.model(64, 97, [(M.attn(heads, heads, dim, vdim), M.dense(64))])
    w, toks = M.weights(cfg, 5), M.prompt(cfg, 1101, 6)
    want = M.oracle(cfg, w, toks)
    m = build(cfg, w, dtype, capacity=1110, max_portion=1110)
    for first in (700, 1023, 1097):
        m.forward(0, toks[:first], 0, [first - 1])
        got = torch.cat([m.forward(0, [toks[i]], i, [0]) for i in range(first, first + 4)])
        assert M.error(got, want[first:first + 4]) < LIMIT[dtype], f"from position {first}"
