"""The matrix products of a portion at the edges of their tiles, in models small enough for the oracle.

Sizes are chosen so that every tile is taken (one layer whose feed-forward and vocabulary make the product that decides): tokens
at and one past a tile's columns, rows that end inside a tile, one step of k and several, split and whole."""
import functools

import pytest
import torch

from tests import nibotar_models as M
from tests.test_gpu_nibotar import DTYPES, IDS, LIMIT, build

pytestmark = pytest.mark.gpu

# (tokens, width, feed-forward, vocabulary): tile rows x tokens of the up rows in bf16; the down rows are split in most
DENSE = [(2, 300, 2001, 333),        # 64 x 16
         (16, 1500, 2000, 51),
         (17, 130, 9001, 51),        # 64 x 32
         (33, 60, 20003, 51),        # 64 x 64, one step of k
         (64, 130, 20001, 51),
         (65, 60, 20001, 51),        # 64 x 96
         (65, 60, 33001, 51),        # 256 x 96
         (97, 130, 29999, 777),      # 128 x 64
         (97, 260, 17001, 17001),    # 96 x 128, in the head as well
         (97, 60, 33001, 51),        # 128 x 128, two per compute unit (fp32 too)
         (97, 390, 25001, 51),       # 128 x 128, one
         (129, 60, 22001, 22001),    # 96 x 160, in the head as well
         (129, 60, 33001, 51),       # 192 x 160
         (129, 130, 25001, 25001),   # 128 x 192, in the head as well
         (193, 390, 25001, 51),      # 256 x 128
         (257, 60, 20000, 51),
         (129, 520, 29999, 51),
         (700, 300, 4001, 51),       # 64 x 96 in the down rows, split
         (257, 520, 29999, 51),      # 256 x 256
         (513, 130, 20001, 20001)]   # one token and one row in the last tiles


@functools.lru_cache(maxsize=1)
def dense(n, width, ff, vocab):
    cfg = M.model(width, vocab, [(M.attn(2, 1, 16, 16), M.dense(ff))])
    w, toks, res = M.weights(cfg, 7), M.prompt(cfg, n, 8), []
    return cfg, w, toks, M.oracle(cfg, w, toks, res), res[0]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("sizes", DENSE, ids=str)
def test_dense_products(sizes, dtype):
    cfg, w, toks, want, res = dense(*sizes)
    logits, layers = build(cfg, w, dtype, capacity=sizes[0]).forward(0, toks, 0, range(sizes[0]), residuals=True)
    assert M.error(layers[0], res) < LIMIT[dtype]
    assert M.error(logits, want) < LIMIT[dtype]


# (tokens, top, experts, feed-forward of one): one tile per expert, several, experts without tokens
EXPERTS = [(9, 2, 40, 500), (60, 2, 3, 9000), (150, 2, 3, 4000), (97, 2, 3, 9001), (400, 2, 3, 4000), (300, 3, 4, 7001)]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("sizes", EXPERTS, ids=str)
def test_expert_products(sizes, dtype):
    n, top, experts, ff = sizes
    cfg = M.model(100, 64, [(M.attn(2, 1, 16, 16), M.moe(ff, experts, top, shared=40))])
    w, toks, res = M.weights(cfg, 9), M.prompt(cfg, n, 10), []
    if experts > top:                # most tokens go to the same experts, so that these have several tiles and others none
        w["l0.mlp.table"][:48] = torch.arange(top, dtype=torch.int32)
    want = M.oracle(cfg, w, toks, res)
    logits, layers = build(cfg, w, dtype, capacity=n).forward(0, toks, 0, range(n), residuals=True)
    assert M.error(layers[0], res[0]) < LIMIT[dtype]
    assert M.error(logits, want) < LIMIT[dtype]
