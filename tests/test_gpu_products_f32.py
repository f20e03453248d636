"""fp32 products of 64 tokens and more, whose values are taken apart into bf16 parts: every tile in every kind of product, one to many steps of k,
values that bf16 does not hold, infinities and NaN.

Limit: a product's value is kept to 2^-24 and sums are rounded in fp32, which over the sums of these sizes gives 1e-6 of the outputs' spread in
the products alone; attention and norms, in fp32 as before, add as much."""
import functools

import pytest
import torch

from tests import kagapel_models as K
from tests import nibotar_models as M
from tests import seq_plan as P

LIMIT = 4e-6
S, T, B = (64, 64), (128, 64), (128, 128)

UP = [((97, 61, 16001), S), ((257, 93, 6001), S), ((97, 125, 10001), T), ((65, 221, 16001), T), ((65, 29, 24001), B), ((129, 93, 16001), B)]
DOWN = [((97, 1030, 4100), (*S, 6)), ((193, 3000, 700), (*T, 2)), ((129, 3000, 1500), (*T, 3)), ((65, 2052, 4100), (*T, 6)), ((193, 2052, 2500), (*B, 6))]
GATED = [((129, 60, 5001), S), ((97, 130, 5001), T), ((65, 93, 12001), B)]
HEADS = [((24, 100, 72, 512, 129), S), ((24, 192, 200, 130, 97), T), ((24, 192, 200, 60, 200), B)]
EXPERTS = [((200, 2, 8, 2000, 29), S), ((200, 2, 3, 2000, 61), S), ((150, 1, 3, 4001, 125), T), ((300, 1, 2, 2000, 125), T), ((150, 2, 3, 4001, 29), B), ((300, 2, 3, 2000, 29), B)]
UP_SIZES = [s for s, _ in UP]
HEAD = [((97, 61, 16001), S), ((97, 125, 10001), T), ((97, 29, 20001), B)]


def test_tiles():
    for (n, width, ff), tile in UP + HEAD:
        assert P.product(ff, n, width, False)[:2] == tile
    for (n, width, ff), tile in DOWN:
        rows, tokens, _, parts = P.product(width, n, ff, False, P.room(n, width))
        assert (rows, tokens, parts) == tile
    for (n, width, ff), tile in GATED:
        assert P.product(2 * ff, n, width, False)[:2] == tile
    for (heads, dim, vdim, rank, n), tile in HEADS:
        assert P.product(heads * (dim + vdim), n, rank, False)[:2] == tile
    for sizes, tile in EXPERTS:
        assert P.experts(*sizes, False)[:2] == tile
    for cases in (UP, GATED, HEADS, EXPERTS, HEAD):
        assert {t for _, t in cases} == {S, T, B}
    assert {t[:2] for _, t in DOWN} == {S, T, B}


def fp32(w):
    """Weights of 24 bits from those of 8."""
    g = torch.Generator().manual_seed(11)
    return {k: v if not v.dtype.is_floating_point or v.numel() < 4 else v.float() * (1 + 2.0 ** -8 * torch.rand(v.shape, generator=g)) for k, v in w.items()}


@functools.lru_cache(maxsize=1)
def dense(n, width, ff, vocab=51, softcap=20.0):
    cfg = M.model(width, vocab, [(M.attn(2, 1, 16, 16), M.dense(ff) if ff else None)], softcap=softcap)
    w, toks, res = fp32(M.weights(cfg, 7)), M.prompt(cfg, n, 8), []
    return cfg, w, toks, M.oracle(cfg, w, toks, res), res[0]


def nibotar(cfg, w, n, capacity=None):
    from clusterfusionplus_amd import nibotar
    return nibotar.from_tensors(cfg, w, torch.float32, capacity=capacity or n)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [s for s, _ in UP + DOWN], ids=str)
def test_dense_products(sizes):
    cfg, w, toks, want, res = dense(*sizes)
    logits, layers = nibotar(cfg, w, sizes[0]).forward(0, toks, 0, range(sizes[0]), residuals=True)
    assert M.error(layers[0], res) < LIMIT
    assert M.error(logits, want) < LIMIT


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [s for s, _ in GATED] + [(n, 64, None, mixer) for *mixer, n in [s for s, _ in HEADS]], ids=str)
def test_gated_products_and_products_of_latents(sizes):
    n, width, ff, (heads, dim, vdim, rank) = (*sizes, (2, 16, 16, 24))[:4]
    cfg = K.model(width, 51, [K.gated(heads, dim, 16, vdim, rank, ff=ff)], streams=2, positions=n)
    w, toks = fp32(K.weights(cfg, 7)), M.prompt(cfg, n, 8)
    from clusterfusionplus_amd import kagapel
    got = kagapel.from_tensors(cfg, w, torch.float32, capacity=n).forward(0, toks, 0, range(n))
    assert M.error(got, K.oracle(cfg, w, toks)) < LIMIT


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [s for s, _ in EXPERTS], ids=str)
def test_expert_products(sizes):
    n, top, experts, ff, width = sizes
    cfg = M.model(width, 64, [(M.attn(2, 1, 16, 16), M.moe(ff, experts, top))])
    w, toks, res = fp32(M.weights(cfg, 9)), M.prompt(cfg, n, 10), []
    want = M.oracle(cfg, w, toks, res)
    logits, layers = nibotar(cfg, w, n).forward(0, toks, 0, range(n), residuals=True)
    assert M.error(layers[0], res[0]) < LIMIT
    assert M.error(logits, want) < LIMIT


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["ordinary", "infinite", "not a number", "near the largest", "1e-36"])
@pytest.mark.parametrize("sizes", [s for s, _ in HEAD], ids=str)
def test_values_of_the_head(sizes, what):
    """What fp32 gives, whatever the values: logits without a cap."""
    n, width, vocab = sizes
    cfg, w, toks, _, _ = dense(n, width, 0, vocab, None)
    w = dict(w, head=w["head"].clone())
    rows = [0, 70, vocab // 2, vocab - 1]
    if what == "1e-36":
        w["head"] *= 1e-36
    elif what != "ordinary":
        w["head"][rows, width // 3] = {"infinite": float("inf"), "not a number": float("nan"), "near the largest": 3.4e38}[what]
    got, want = nibotar(cfg, w, n).forward(0, toks, 0, range(n)).cpu(), M.oracle(cfg, w, toks)
    for same in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(same(got), same(want.float()))
    if what in ("infinite", "not a number", "near the largest"):
        huge, exact = got[:, rows].double(), want[:, rows]
        live = torch.isfinite(huge)
        assert live.any() == (what == "near the largest")
        assert not live.any() or (huge[live] - exact[live]).abs().max().item() < 4 * LIMIT * 3.4e38      # (LIMIT is a root mean square)
        keep = [i for i in range(vocab) if i not in rows]
        got, want = got[:, keep], want[:, keep]
    assert M.error(got, want) < LIMIT


def by_row(got, want):
    """Root mean square of the difference of each row of the head, in units of its own spread."""
    d = got.double() - want
    return (d.pow(2).mean(0).sqrt() / want.std(0)).max().item()


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["rows", "inputs of 1e30", "inputs of 1e37", "inputs of 1e-7", "all small"])
@pytest.mark.parametrize("sizes", [s for s, _ in HEAD], ids=str)
def test_small_values_beside_others(sizes, what):
    """A value's error goes with the value: small rows of weights between ordinary ones, a column of inputs that are large where the weights are small,
    or the other way round, inputs and weights that are all small.  (2^-24 is the least that a final norm's factor 1 + w can be but for zero.)"""
    n, width, vocab = sizes
    cfg, w, toks, _, _ = dense(n, width, 0, vocab, None)
    w = dict(w, head=w["head"].clone())
    w["final.norm"] = w["final.norm"].clone()
    if what == "rows":
        for row, scale in zip([0, 1, 70, 71, vocab // 2, vocab - 1], [1e-30, 1e-33, 1e-35, 1e-36, 1e-34, 1e-37]):
            w["head"][row] *= scale
    elif what == "all small":
        w["final.norm"][:] = -1 + 2.0 ** -24
        w["head"] *= 1e-29
    else:
        factor = 2.0 ** -24 if what == "inputs of 1e-7" else float(what.split()[-1])
        w["final.norm"][width // 3] = factor if factor > 1 else factor - 1
        w["head"][:, width // 3] /= factor
    got, want = nibotar(cfg, w, n).forward(0, toks, 0, range(n)).cpu(), M.oracle(cfg, w, toks)
    assert by_row(got, want) < LIMIT


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [s for s, _ in UP[::2] + GATED] + [(n, 64, None, mixer) for *mixer, n in [s for s, _ in HEADS]] + [s for s, _ in EXPERTS[::3]], ids=str)
def test_a_token_that_is_no_number(sizes):
    """Every kind of product: it and the tokens behind it, which see its key, are no numbers; those before it are as they are, but for the ones
    whose keys share its tile of 32 in the attention (their weights for it are zero, and zero times its values is no number)."""
    if len(sizes) == 5:
        n, top, experts, ff, width = sizes
        cfg, made, lib = M.model(width, 64, [(M.attn(2, 1, 16, 16), M.moe(ff, experts, top))]), M, "nibotar"
    elif sizes in UP_SIZES:
        n, width, ff = sizes
        cfg, made, lib = M.model(width, 51, [(M.attn(2, 1, 16, 16), M.dense(ff))]), M, "nibotar"
    else:
        n, width, ff, (heads, dim, vdim, rank) = (*sizes, (2, 16, 16, 24))[:4]
        cfg, made, lib = K.model(width, 51, [K.gated(heads, dim, 16, vdim, rank, ff=ff)], streams=2, positions=n), K, "kagapel"
    import importlib
    lib = importlib.import_module(f"clusterfusionplus_amd.{lib}")
    w = fp32(made.weights(cfg, 9))
    w["embed"][0] = float("nan")
    toks, bad = [t or 1 for t in M.prompt(cfg, n, 10)], 2 * n // 3
    toks[bad] = 0
    got = lib.from_tensors(cfg, w, torch.float32, capacity=n).forward(0, toks, 0, range(n)).cpu()
    assert got[bad:].isnan().all()
    clean = bad // 32 * 32
    assert M.error(got[:clean], made.oracle(cfg, w, toks[:clean])) < LIMIT
