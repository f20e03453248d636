"""Attention of a portion: keys shared among workgroups, tiles of keys that begin and end anywhere, scores of either sign."""
import functools

import pytest
import torch

from tests import kagapel_models as K
from tests import nibotar_models as N
from tests.test_gpu_nibotar import DTYPES, IDS, LIMIT

pytestmark = pytest.mark.gpu


def grouped(scale=None, chunk=None, dims=(40, 56)):
    return N, N.model(64, 51, [(N.attn(6, 2, *dims, scale=scale, chunk=chunk, rot=8), None)])


def latent(scale=None, dims=(40, 16, 56, 48)):
    return K, K.model(64, 51, [K.gated(3, *dims, scale=scale), K.sunk(3, *dims, scale=scale, kv_from=0)], positions=1400)


MODELS = {"grouped": grouped(), "grouped_chunks": grouped(chunk=400), "grouped_small": grouped(dims=(16, 32)), "grouped_large": grouped(dims=(200, 250)),
          "latent": latent(), "latent_wide": latent(dims=(128, 64, 128, 96)), "latent_large": latent(dims=(160, 64, 200, 96)),
          "negative": grouped(scale=-0.2), "zero": grouped(scale=0.0), "latent_negative": latent(scale=-0.2)}


# (context, tokens): one and two tiles (64 keys in bf16, 32 in fp32) per workgroup and fewer than that, first and last keys of a
# tile, several column tiles, the edge of a chunk inside the portion
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("name", list(MODELS))
def test_portions_far_into_a_sequence(name, dtype):
    from clusterfusionplus_amd import kagapel, nibotar
    M, cfg = MODELS[name]
    w, toks, res = M.weights(cfg, 5), M.prompt(cfg, 1300, 6), []
    want = M.oracle(cfg, w, toks, res)
    m = (nibotar if M is N else kagapel).from_tensors(cfg, w, dtype, capacity=1300)
    pos = 0
    for n in (64, 63, 2, 127, 129, 3, 37, 70, 300, 5, 200, 2, 290, 8):
        logits, layers = m.forward(0, toks[pos:pos + n], pos, range(n), residuals=True)
        assert N.error(layers[-1], res[-1][pos:pos + n]) < LIMIT[dtype], (pos, n)
        assert N.error(logits, want[pos:pos + n]) < LIMIT[dtype], (pos, n)
        pos += n
    assert pos == 1300


# short portions that begin with a chunk, just behind its edge and just before it: they see a tile or two, far into the sequence
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
def test_short_portions_at_the_edge_of_a_chunk(dtype):
    from clusterfusionplus_amd import nibotar
    cfg = grouped(chunk=400)[1]
    w, toks = N.weights(cfg, 5), N.prompt(cfg, 1300, 6)
    want = N.oracle(cfg, w, toks)
    m = nibotar.from_tensors(cfg, w, dtype, capacity=1300)
    pos = 0
    for n in (400, 37, 63, 300, 2, 5, 130, 263, 3, 37, 60):
        assert N.error(m.forward(0, toks[pos:pos + n], pos, range(n)), want[pos:pos + n]) < LIMIT[dtype], (pos, n)
        pos += n
    assert pos == 1300


# a scale that is no number: no logit is one, in one split of the keys and in several
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("kind", [grouped, latent])
def test_scale_that_is_no_number(kind, dtype):
    from clusterfusionplus_amd import kagapel, nibotar
    M, cfg = kind(scale=float("nan"))
    toks = M.prompt(cfg, 600, 6)
    m = (nibotar if M is N else kagapel).from_tensors(cfg, M.weights(cfg, 5), dtype, capacity=600)
    for pos, n in ((0, 30), (30, 560), (590, 5)):
        assert m.forward(0, toks[pos:pos + n], pos, range(n)).isnan().all(), (pos, n)


# projections of up to 8192 and 16384 values, and of more; heads that are no whole groups of four; values mixed; padded heads
PROJECTIONS = {"12k": [N.attn(64, 16, 128, 128)], "17k": [N.attn(128, 4, 128, 128)], "mixed_12k": [N.attn(48, 12, 100, 132, v_mix=True, chunk=31), N.attn(48, 12, 100, 132, v_mix=True)],
               "no_fours": [N.attn(6, 2, 42, 30, v_mix=True), N.attn(6, 2, 40, 30, v_mix=True), N.attn(10, 5, 42, 12, v_mix=True)]}


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("name", list(PROJECTIONS))
def test_projection_sizes(name, dtype):
    from clusterfusionplus_amd import nibotar
    cfg = N.model(64, 51, [(m, None) for m in PROJECTIONS[name]])
    w, toks = N.weights(cfg, 5), N.prompt(cfg, 90, 6)
    want = N.oracle(cfg, w, toks)
    m = nibotar.from_tensors(cfg, w, dtype, capacity=100)
    logits = torch.cat([m.forward(0, toks[:33], 0, range(33)), m.forward(0, toks[33:62], 33, range(29)), m.forward(0, toks[62:], 62, range(28))])
    assert N.error(logits, want) < LIMIT[dtype]


# enough columns for blocks of 32 (512 workgroups of 128; tests/test_seq_plan.py): every size of tile, heads that share keys, chunks, a last block that is not full, keys of
# the portion and of the context before it, scores of either sign and scores that are no numbers
BLOCKS = {"small": (N, N.attn(64, 64, 16, 32)), "middle": (N, N.attn(64, 64, 72, 80, rot=8)), "large": (N, N.attn(64, 64, 200, 250)),
          "groups": (N, N.attn(96, 48, 40, 56, rot=8)), "chunks": (N, N.attn(64, 64, 40, 56, chunk=400)), "negative": (N, N.attn(64, 64, 40, 56, scale=-0.2)),
          "keys_192": (N, N.attn(64, 64, 160, 96)), "latent": (K, K.gated(64, 40, 16, 56, 48)), "latent_middle": (K, K.sunk(64, 72, 32, 88, 48)),
          "latent_wide": (K, K.sunk(64, 128, 64, 128, 96)), "latent_large": (K, K.gated(64, 160, 64, 200, 96)), "nan": (N, N.attn(64, 64, 40, 56, scale=float("nan")))}


@pytest.mark.parametrize("name", list(BLOCKS))
def test_columns_in_blocks_of_32(name):
    from clusterfusionplus_amd import kagapel, nibotar
    M, mixer = BLOCKS[name]
    cfg = M.model(64, 51, [mixer], positions=1900) if M is K else M.model(64, 51, [(mixer, None)])
    w, toks = M.weights(cfg, 5), M.prompt(cfg, 1807, 6)
    m = (nibotar if M is N else kagapel).from_tensors(cfg, w, torch.bfloat16, capacity=1807)
    got = torch.cat([m.forward(0, toks[:900], 0, range(900)), m.forward(0, toks[900:], 900, range(907))])
    if name == "nan":
        assert got.isnan().all()
    else:
        assert N.error(got, M.oracle(cfg, w, toks)) < LIMIT[torch.bfloat16]


# more workgroups than are resident, by less than one per compute unit: 10 rows of 64 heads; 5 of them in front
LEFT_OVER = {"grouped": (N, N.attn(64, 64, 40, 56, rot=8)), "chunks": (N, N.attn(64, 64, 40, 56, chunk=1000)), "latent": (K, K.sunk(64, 40, 16, 56, 48)), "middle": (N, N.attn(64, 64, 128, 128))}
LEFT_OVER_TOKENS = (320, 625)


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("name", list(LEFT_OVER))
def test_workgroups_left_over(name, dtype):
    from clusterfusionplus_amd import kagapel, nibotar
    M, mixer = LEFT_OVER[name]
    first, n = LEFT_OVER_TOKENS
    cfg = M.model(64, 51, [mixer], positions=1000) if M is K else M.model(64, 51, [(mixer, None)])
    w, toks = M.weights(cfg, 5), M.prompt(cfg, first + n, 6)
    m = (nibotar if M is N else kagapel).from_tensors(cfg, w, dtype, capacity=first + n)
    got = torch.cat([m.forward(0, toks[:first], 0, range(first)), m.forward(0, toks[first:], first, range(n))])
    assert N.error(got, M.oracle(cfg, w, toks)) < LIMIT[dtype]


# more heads than workgroups are resident: one row of them
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("kind", ["grouped", "latent"])
def test_one_row_of_many_heads(kind, dtype):
    from clusterfusionplus_amd import kagapel, nibotar
    cfg = K.model(64, 51, [K.sunk(600, 8, 8, 8, 16)]) if kind == "latent" else N.model(64, 51, [(N.attn(600, 600, 8, 8), None)])
    M, make = (K, kagapel) if kind == "latent" else (N, nibotar)
    w, toks = M.weights(cfg, 5), M.prompt(cfg, 30, 6)
    m = make.from_tensors(cfg, w, dtype, capacity=30)
    got = torch.cat([m.forward(0, toks[:20], 0, range(20)), m.forward(0, toks[20:], 20, range(10))])
    assert N.error(got, M.oracle(cfg, w, toks)) < LIMIT[dtype]


# latent projections of up to 4096, 8192 and 12288 values, and of more; in one part (64 columns) and in several (512); rows and gates that are no whole
# groups of four; a layer that reads the latents of another
LATENTS = {"1k": (5, 128, 64, 56, 48), "4k": (19, 128, 64, 56, 384), "4k_more": (19, 128, 64, 56, 388), "6k": (24, 128, 64, 56, 48), "12k": (48, 128, 64, 56, 48), "16k": (64, 128, 64, 56, 48), "no_fours": (3, 41, 16, 55, 49), "gates_no_fours": (3, 44, 16, 55, 48)}


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("width", [64, 512])
@pytest.mark.parametrize("name", list(LATENTS))
def test_latent_projection_sizes(name, width, dtype):
    from clusterfusionplus_amd import kagapel
    dims = LATENTS[name]
    cfg = K.model(width, 51, [K.gated(*dims), K.sunk(*dims, kv_from=0), K.gated(*dims), K.sunk(*dims)])
    w, toks = K.weights(cfg, 5), K.prompt(cfg, 90, 6)
    want = K.oracle(cfg, w, toks)
    m = kagapel.from_tensors(cfg, w, dtype, capacity=100)
    logits = torch.cat([m.forward(0, toks[:33], 0, range(33)), m.forward(0, toks[33:62], 33, range(29)), m.forward(0, toks[62:], 62, range(28))])
    assert N.error(logits, want) < LIMIT[dtype]


# projections of up to 4096, 8192 and more values whose products are split over k, by (values, width): partial rotation, padded heads, values kept by
# the first layer and mixed in by the second; 2 to 8 parts over these portions (tests/test_seq_plan.py)
PARTS_ROWS = {4096: (16, 8, 128, 128), 4100: (25, 5, 116, 124), 8192: (32, 16, 128, 128), 8196: (33, 3, 208, 236)}
PARTS_WIDTHS, PARTS_TOKENS = (1024, 2048), (5, 17, 33)


@functools.lru_cache(maxsize=1)
def in_parts(values, width):
    cfg = N.model(width, 51, [(N.attn(*PARTS_ROWS[values], rot=rot, v_mix=True), None) for rot in (64, 100)])
    w, toks = N.weights(cfg, 5), N.prompt(cfg, sum(PARTS_TOKENS), 6)
    return cfg, w, toks, N.oracle(cfg, w, toks)


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("width", PARTS_WIDTHS)
@pytest.mark.parametrize("values", list(PARTS_ROWS))
def test_projections_in_parts(values, width, dtype):
    from clusterfusionplus_amd import nibotar
    cfg, w, toks, want = in_parts(values, width)
    m, pos = nibotar.from_tensors(cfg, w, dtype, capacity=100), 0
    for n in PARTS_TOKENS:
        assert N.error(m.forward(0, toks[pos:pos + n], pos, range(n)), want[pos:pos + n]) < LIMIT[dtype], n
        pos += n
