"""Portions of few tokens behind many positions, whose latent attention reads the cached latents: blocks of one, two and four sets of 16 columns, blocks and
workgroups that are not full, ranks of either kernel, heads of more dimensions than one pass takes, gates, sinks and shared latents."""
import functools

import pytest
import torch

from tests import kagapel_models as M
from tests import seq_plan as P
from tests.test_gpu_kagapel import DTYPES, IDS, LIMIT, build

# context, then the portions that follow one another
TURNS = {
    "heads_of_128": (M.model(200, 51, [M.gated(16, 128, 64, 128, 512)], positions=1700), 1600, (2, 7, 3)),
    "rank_of_100": (M.model(64, 51, [M.sunk(40, 64, 8, 100, 100)], positions=1700), 1500, (3, 6)),
    "large_heads": (M.model(64, 51, [M.gated(16, 180, 64, 250, 300)], positions=1300), 1200, (5, 17)),
    "odd_heads": (M.model(330, 41, [M.sunk(33, 100, 60, 131, 333), M.gated(33, 150, 60, 70, 333, kv_from=0)], positions=1300), 1200, (4, 5, 2)),
    "hundred_heads": (M.model(1024, 51, [M.sunk(100, 128, 64, 128, 512)], positions=1200), 1100, (11, 31)),
}


def plans(name, dtype):
    cfg, pos, turns = TURNS[name]
    bf16 = dtype == torch.bfloat16
    out = []
    for n in turns:
        out += [(n, *P.turn(n, pos, layer["mixer"], bf16, P.room(cfg["max_positions"], cfg["width"]))) for layer in cfg["layers"]]
        pos += n
    return out


def test_plans():
    for dtype in DTYPES:
        chosen = [p for name in TURNS for p in plans(name, dtype)]
        assert all(splits > 0 for _, splits, *_ in chosen if dtype == torch.bfloat16)
        assert {sets for _, splits, sets, *_ in chosen if splits} == {1, 2, 4}
    wide, small = {"heads": 128, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512}, {"heads": 2, "dim": 16, "rot_dim": 8, "vdim": 16, "kv_rank": 24}
    room = 16 << 20
    assert P.turn(20, 3000, wide, True, room)[0] > 0 and P.turn(120, 3000, wide, True, room)[0] == 0 and P.turn(500, 3000, wide, True, room)[0] == 0
    assert P.turn(2, 0, wide, True, room)[0] == 0 and P.turn(2, 100, small, True, room)[0] == 0 and P.turn(2, 100, small, False, room)[0] == 0
    assert P.turn(20, 3000, wide, True, 1000)[0] == 0                 # no room for partial results
    for n in (2, 17, 60):
        for pos in (100, 1000, 4000, 100000):
            splits, sets, tokens = P.turn(n, pos, wide, True, room)
            if splits:
                assert splits <= 64 and splits * n * 128 * 514 <= room and sets in (1, 2, 4) and 2 <= tokens <= 16


@functools.lru_cache(maxsize=1)
def reference(name):
    cfg, pos, turns = TURNS[name]
    w, toks = M.weights(cfg, 5), M.prompt(cfg, pos + sum(turns), 6)
    return w, toks, M.oracle(cfg, w, toks)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("name", TURNS)
def test_turns(name, dtype):
    cfg, pos, turns = TURNS[name]
    w, toks, want = reference(name)
    m = build(cfg, w, dtype, capacity=cfg["max_positions"])
    m.forward(0, toks[:pos], 0, [pos - 1])
    for n in turns:
        got = m.forward(0, toks[pos:pos + n], pos, range(n))
        assert M.error(got, want[pos:pos + n]) < LIMIT[dtype]
        pos += n


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
def test_large_latents(dtype):
    """A latent value near the end of the range, alike for all positions, which only small rows of W_uv read: weighted sums of it stay in range."""
    cfg, pos, _ = TURNS["rank_of_100"]
    w, toks, m = dict(M.weights(cfg, 5)), M.prompt(cfg, pos + 4, 6), "l0.mix."
    for n in ("embed", "pos"):
        w[n] = w[n].clone()
        w[n][:, 1] = 3.0 if n == "embed" else 0.0
    w[m + "dkv"][7] = 0
    w[m + "dkv"][7, 1] = 1.0
    w[m + "dkv.norm"][7], w[m + "uk"][:, 7] = 2.0 ** 124, 0
    w[m + "uv"][:, 7] = torch.sign(w[m + "uv"][:, 7].float()).bfloat16() * 2.0 ** -124
    assert P.turn(4, pos, cfg["layers"][0]["mixer"], dtype == torch.bfloat16, P.room(cfg["max_positions"], cfg["width"]))[0] > 0
    c = build(cfg, w, dtype, capacity=cfg["max_positions"])
    c.forward(0, toks[:pos], 0, [pos - 1])
    assert M.error(c.forward(0, toks[pos:], pos, range(4)), M.oracle(cfg, w, toks)[pos:]) < LIMIT[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
def test_values_that_are_not_finite_stay_in_their_sequence(dtype):
    """Heads whose keys end inside a unit of 16 bytes: what lies behind them in the keys' buffer meets zeros of the queries, and has to be finite."""
    cfg = M.model(64, 51, [M.sunk(40, 66, 8, 100, 100)], positions=1700)
    w, toks, pos = dict(M.weights(cfg, 5)), [t or 1 for t in M.prompt(cfg, 1500, 6)], 1500
    w["embed"] = w["embed"].clone()
    w["embed"][0] = float("inf")
    assert P.turn(6, pos, cfg["layers"][0]["mixer"], dtype == torch.bfloat16, P.room(cfg["max_positions"], cfg["width"]))[0] > 0
    m = build(cfg, w, dtype, capacity=cfg["max_positions"], slots=2)
    want = m.forward(0, toks, 0, range(pos))
    assert torch.isfinite(want).all()
    m.forward(1, toks, 0)
    assert not torch.isfinite(m.forward(1, [0] * 6, pos, range(6))).any()
    assert torch.equal(m.forward(0, toks, 0, range(pos)), want)
