"""The matrix products of a portion at the edges of their tiles, in models small enough for the oracle.

Sizes are chosen so that every tile is taken by every kind of product that a model has (one layer, whose product that decides is
large): tokens at and one past a tile's columns, rows that end inside a tile, one step of k and several, split and whole.  The tile
in bf16, (rows, tokens, workgroups per compute unit), and the splits of k that a case is for stand with it; tests/test_seq_plan.py
holds the lists to that."""
import functools

import pytest
import torch

from tests import kagapel_models as K
from tests import nibotar_models as M
from tests.test_gpu_nibotar import DTYPES, IDS, LIMIT, build

pytestmark = pytest.mark.gpu


def build_latent(cfg, w, dtype, capacity):
    from clusterfusionplus_amd import kagapel
    return kagapel.from_tensors(cfg, w, dtype, capacity=capacity)


# (tokens, width, feed-forward, vocabulary): tile of the up rows in bf16; the down rows are split in all but the narrowest tiles' cases
DENSE = [(2, 300, 2001, 333),        # 64 x 16
         (16, 1500, 2000, 51),
         (17, 130, 9001, 51),        # 64 x 32
         (33, 60, 20003, 51),        # 64 x 64, one step of k
         (64, 130, 20001, 51),
         (65, 60, 20001, 51),        # 64 x 96
         (65, 60, 33001, 51),        # 256 x 96
         (97, 130, 29999, 777),      # 128 x 64
         (97, 260, 17001, 17001),    # 96 x 128, in the head as well
         (97, 60, 33001, 51),        # 128 x 128, two per compute unit
         (97, 390, 25001, 51),       # 128 x 128, one (fp32: 128 x 128)
         (129, 60, 22001, 22001),    # 96 x 160, in the head as well
         (129, 60, 33001, 51),       # 192 x 160
         (129, 130, 25001, 25001),   # 128 x 192, in the head as well
         (193, 390, 25001, 51),      # 256 x 128
         (257, 60, 20000, 51),       # 256 x 96, three of them over the tokens
         (129, 520, 29999, 51),      # 128 x 192
         (700, 300, 4001, 51),       # 64 x 96 in the down rows, split
         (257, 520, 29999, 51),      # 256 x 256, nine steps of k
         (513, 130, 20001, 20001)]   # 128 x 192: 129 tokens and 33 rows in the last tiles
DENSE_TILES = [(64, 16, 2), (64, 16, 2), (64, 32, 2), (64, 64, 2), (64, 64, 2), (64, 96, 2), (256, 96, 1), (128, 64, 2), (96, 128, 1), (128, 128, 2),
               (128, 128, 1), (96, 160, 1), (192, 160, 1), (128, 192, 1), (256, 128, 1), (256, 96, 1), (128, 192, 1), (64, 96, 2), (256, 256, 1), (128, 192, 1)]


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


# (tokens, width, feed-forward), tile and splits of the down rows, with room for up to 16: the products that the residual sums read
SPLIT = [((2, 257, 4100), (64, 16, 2, 16)), ((17, 700, 4100), (64, 32, 2, 16)), ((33, 700, 4100), (64, 64, 2, 16)), ((65, 1030, 4100), (64, 96, 2, 12)),
         ((33, 2052, 8000), (128, 64, 2, 12)), ((97, 8196, 1500), (128, 128, 1, 3)), ((97, 2052, 8000), (128, 128, 1, 12)), ((193, 700, 8000), (96, 128, 1, 16)),
         ((129, 1501, 8000), (96, 160, 1, 16)), ((161, 4097, 4100), (128, 192, 1, 6)), ((129, 4100, 8000), (192, 160, 1, 8)), ((65, 6000, 8000), (256, 96, 1, 8)),
         ((193, 8196, 3000), (256, 128, 1, 3)), ((193, 8196, 6000), (256, 256, 1, 6))]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("sizes", [s for s, _ in SPLIT], ids=str)
def test_split_products(sizes, dtype):
    cfg, w, toks, want, res = dense(*sizes, 51)
    logits, layers = build(cfg, w, dtype, capacity=4 * sizes[0]).forward(0, toks, 0, range(sizes[0]), residuals=True)
    assert M.error(layers[0], res) < LIMIT[dtype]
    assert M.error(logits, want) < LIMIT[dtype]


# (tokens, width, feed-forward), tile of the gate and up rows; the down rows, with a bias, are split (the last two: 256 x 256)
GATED = [((17, 130, 4500), (64, 32, 2)), ((50, 60, 10000), (64, 64, 2)), ((65, 60, 10001), (64, 96, 2)), ((65, 60, 16500), (256, 96, 1)), ((97, 130, 15000), (128, 64, 2)),
         ((97, 200, 10001), (96, 128, 1)), ((97, 60, 16500), (128, 128, 2)), ((97, 390, 12500), (128, 128, 1)), ((129, 520, 10000), (96, 160, 1)),
         ((129, 70, 12500), (128, 192, 1)), ((129, 60, 16500), (192, 160, 1)), ((193, 390, 12500), (256, 128, 1)), ((193, 130, 24999), (256, 256, 1)),
         ((193, 8196, 6000), (96, 128, 1)), ((400, 8196, 4500), (128, 192, 1))]


@functools.lru_cache(maxsize=1)
def latent(n, width, vocab, streams, mixer, ff):
    cfg = K.model(width, vocab, [K.gated(*mixer, ff=ff)], streams=streams, positions=n)
    w, toks, res = K.weights(cfg, 7), M.prompt(cfg, n, 8), []
    return cfg, w, toks, K.oracle(cfg, w, toks, res), res[0]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("sizes", [s for s, _ in GATED], ids=str)
def test_gated_products(sizes, dtype):
    n, width, ff = sizes
    cfg, w, toks, want, res = latent(n, width, 51, 2, (2, 16, 8, 16, 24), ff)
    logits, layers = build_latent(cfg, w, dtype, n).forward(0, toks, 0, range(n), residuals=True)
    assert M.error(layers[0], res) < LIMIT[dtype]
    assert M.error(logits, want) < LIMIT[dtype]


# (heads, dimensions, of values, latent values, positions), tile of the product that makes the keys and values of all positions
HEADS = [((48, 100, 72, 130, 17), (64, 32, 2)), ((48, 192, 200, 60, 33), (64, 64, 2)), ((64, 100, 72, 130, 65), (64, 96, 2)), ((48, 192, 200, 200, 97), (96, 128, 1)),
         ((48, 192, 200, 512, 129), (96, 160, 1)), ((48, 191, 200, 60, 97), (128, 64, 2)), ((64, 192, 200, 512, 97), (128, 128, 1)), ((64, 192, 200, 60, 193), (128, 128, 2)),
         ((64, 190, 199, 130, 129), (128, 192, 1)), ((48, 192, 200, 130, 300), (192, 160, 1)), ((64, 192, 200, 60, 129), (256, 96, 1)), ((64, 192, 200, 512, 193), (256, 128, 1)),
         ((64, 192, 200, 512, 385), (256, 256, 1)), ((64, 193, 198, 512, 385), (256, 256, 1))]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("sizes", [s for s, _ in HEADS], ids=str)
def test_products_of_latents(sizes, dtype):
    heads, dim, vdim, rank, n = sizes
    cfg, w, toks, want, _ = latent(n, 64, 51, 1, (heads, dim, 16, vdim, rank), None)
    m = build_latent(cfg, w, dtype, n)
    logits = torch.cat([m.forward(0, toks[:n - 3], 0, range(n - 3)), m.forward(0, toks[n - 3:], n - 3, range(3))])
    assert M.error(logits, want) < LIMIT[dtype]


# (tokens, top, experts, feed-forward of one, width), tile, and whether it is meant to hold an expert's tokens
EXPERT_TILES = [((33, 1, 3, 300, 60), (64, 16, 2, True)), ((65, 2, 8, 701, 100), (64, 32, 2, True)), ((97, 1, 3, 4000, 60), (64, 64, 2, True)), ((97, 2, 3, 4000, 60), (64, 96, 2, True)),
                ((150, 2, 3, 4000, 260), (96, 128, 1, True)), ((200, 2, 3, 4000, 520), (96, 160, 1, True)), ((150, 2, 2, 4000, 61), (128, 64, 2, False)),
                ((400, 2, 8, 2000, 60), (128, 128, 1, True)), ((700, 2, 3, 2000, 60), (128, 128, 2, False)), ((1000, 1, 3, 2000, 100), (128, 192, 1, False)),
                ((200, 2, 3, 8000, 60), (192, 160, 1, True)), ((97, 2, 3, 8000, 60), (256, 96, 1, True)), ((700, 2, 8, 2000, 520), (256, 128, 1, False)),
                ((300, 3, 4, 8000, 60), (256, 256, 1, True)), ((700, 2, 3, 4000, 259), (256, 256, 1, False))]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("sizes", [s for s, _ in EXPERT_TILES], ids=str)
def test_expert_tiles(sizes, dtype):
    n, top, experts, ff, width = sizes
    cfg, w, toks, want, res = routed(*sizes)
    logits, layers = build(cfg, w, dtype, capacity=n).forward(0, toks, 0, range(n), residuals=True)
    assert M.error(layers[0], res) < LIMIT[dtype]
    assert M.error(logits, want) < LIMIT[dtype]


@functools.lru_cache(maxsize=1)
def routed(n, top, experts, ff, width):
    cfg = M.model(width, 64, [(M.attn(2, 1, 16, 16), M.moe(ff, experts, top))])
    w, toks, res = M.weights(cfg, 9), M.prompt(cfg, n, 10), []
    return cfg, w, toks, M.oracle(cfg, w, toks, res), res[0]


# (tokens, width, vocabulary), tile of the head
HEAD = [((193, 130, 50001), (256, 256, 1)), ((193, 390, 25001), (256, 128, 1)), ((65, 60, 33001), (256, 96, 1)), ((129, 60, 33003), (192, 160, 1)), ((97, 60, 33003), (128, 128, 2)),
        ((97, 390, 25001), (128, 128, 1)), ((97, 130, 29999), (128, 64, 2)), ((65, 60, 20001), (64, 96, 2)), ((33, 60, 20003), (64, 64, 2)), ((17, 130, 9001), (64, 32, 2))]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("sizes", [s for s, _ in HEAD], ids=str)
def test_heads(sizes, dtype):
    n, width, vocab = sizes
    cfg = M.model(width, vocab, [(M.attn(2, 1, 16, 16), None)])
    w, toks = M.weights(cfg, 7), M.prompt(cfg, n, 8)
    assert M.error(build(cfg, w, dtype, capacity=n).forward(0, toks, 0, range(n)), M.oracle(cfg, w, toks)) < LIMIT[dtype]


# widths at the edges of what the kernels between the products hold in registers, rows of whole groups of four and others; the
# down rows are split, so that they have parts to add
WIDTHS = [2048, 2052, 4096, 4097, 4100, 8192, 8196]
STREAMS = [(2048, 1), (2048, 4), (2052, 2), (4096, 1), (4096, 3), (4096, 4), (4098, 2), (5120, 4), (2052, 8)]
ROWS = (41, 1500)                # tokens, feed-forward


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("width", WIDTHS)
def test_rows_of_wide_models(width, dtype):
    n, ff = ROWS
    cfg = M.model(width, 51, [(M.attn(2, 1, 16, 16), M.dense(ff)), (M.attn(2, 1, 16, 16), M.moe(40, 5, 3, shared=600))])
    w, toks, res = M.weights(cfg, 7), M.prompt(cfg, n, 8), []
    want = M.oracle(cfg, w, toks, res)
    logits, layers = build(cfg, w, dtype, capacity=100).forward(0, toks, 0, range(n), residuals=True)
    for got, r in zip(layers, res):
        assert M.error(got, r) < LIMIT[dtype]
    assert M.error(logits, want) < LIMIT[dtype]


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("width, streams", STREAMS)
def test_streams_of_wide_models(width, streams, dtype):
    n, ff = ROWS
    cfg, w, toks, want, res = latent(n, width, 51, streams, (2, 16, 8, 16, 24), ff)
    logits, layers = build_latent(cfg, w, dtype, 100).forward(0, toks, 0, range(n), residuals=True)
    assert M.error(layers[0], res) < LIMIT[dtype]
    assert M.error(logits, want) < LIMIT[dtype]
