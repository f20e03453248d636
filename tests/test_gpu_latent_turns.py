"""Portions of few tokens behind many positions, whose latent attention reads the cached latents: blocks of one, two and four sets of 16 columns for ranks of
either kernel, blocks and workgroups that are not full, more tokens than one workgroup turns into the latent space, heads of more dimensions than one pass
takes, gates, sinks, shared latents, slots, scales; single keys that decide everything, at the edges of tiles, splits and the portion."""
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
    "many_tokens": (M.model(512, 51, [M.gated(24, 192, 64, 256, 300)], positions=1700), 1500, (64, 40)),
    "small_rank": (M.model(256, 51, [M.sunk(61, 192, 64, 256, 64)], positions=700), 600, (33,)),
    "small_rank_few_tokens": (M.model(256, 51, [M.gated(64, 180, 64, 250, 100)], positions=500), 300, (3,)),
}
# heads, dimensions, rank, context and tokens of models with one key that decides everything; sets of columns in a block
FAR = [(32, (180, 64, 250), 300, 700, 5, 1), (48, (192, 64, 256), 300, 400, 24, 2), (24, (192, 64, 256), 300, 1500, 64, 4),
       (64, (180, 64, 250), 100, 300, 3, 1), (48, (192, 64, 256), 100, 400, 17, 2), (61, (192, 64, 256), 64, 600, 33, 4)]
WIDTH = 1024


def plans(name, dtype):
    cfg, pos, turns = TURNS[name]
    bf16 = dtype == torch.bfloat16
    out = []
    for n in turns:
        out += [(n, layer["mixer"]["kv_rank"], *P.turn(n, pos, layer["mixer"], bf16, P.room(cfg["max_positions"], cfg["width"]))) for layer in cfg["layers"]]
        pos += n
    return out


def far_plan(heads, dims, rank, pos, n, bf16):
    mixer = dict(zip(("dim", "rot_dim", "vdim"), dims), heads=heads, kv_rank=rank)
    return P.turn(n, pos, mixer, bf16, P.room(pos + n, WIDTH))


def test_plans():
    for dtype in DTYPES:
        chosen = [p for name in TURNS for p in plans(name, dtype)]
        assert all(splits > 0 for _, _, splits, *_ in chosen)
        assert {(rank <= 128, sets) for _, rank, _, sets, _ in chosen} == {(small, sets) for small in (False, True) for sets in (1, 2, 4)}
        assert {rank <= 128 for n, rank, *_ in chosen if n > 32} == {False, True}             # (more than a workgroup of k_seq_latent_absorb takes)
    for *sizes, sets in FAR:
        assert far_plan(*sizes, True)[0] > 1 and far_plan(*sizes, True)[1] == sets and far_plan(*sizes, False)[0] > 1
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


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("scale", [-0.05, 0.0])
def test_scales_and_slots(scale, dtype):
    cfg, pos, n = M.model(256, 51, [M.sunk(32, 180, 64, 250, 300, scale=scale)], positions=760), 700, 5
    assert P.turn(n, pos, cfg["layers"][0]["mixer"], dtype == torch.bfloat16, P.room(760, 256))[0] > 0
    w = M.weights(cfg, 5)
    m = build(cfg, w, dtype, capacity=760, slots=3)
    seqs = {slot: M.prompt(cfg, pos + n, 6 + slot) for slot in (1, 2)}
    for slot, toks in seqs.items():
        m.forward(slot, toks[:pos], 0)
    for slot, toks in seqs.items():
        assert M.error(m.forward(slot, toks[pos:], pos, range(n)), M.oracle(cfg, w, toks)[pos:]) < LIMIT[dtype]


def far_places(heads, dims, rank, pos, n):
    """Places of the key: first and last of a tile of the context and of a split (bf16), the last of the context, and the first, one and the last of the turn."""
    splits, tiles = far_plan(heads, dims, rank, pos, n, True)[0], (pos + n + 31) // 32
    edge = tiles * (splits // 2) // splits * 32
    return sorted({0, 31, 32, edge - 1, edge, pos - 1, pos, pos + n // 2, pos + n - 1})


@functools.lru_cache(maxsize=None)
def far(heads, dims, rank, pos, n, at, rotated):
    cfg, w, toks = M.far_key_model(heads, rank, pos + n, at, rotated, dims=dims, width=WIDTH)
    return cfg, w, toks, M.oracle(cfg, w, toks)[pos:]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("case", range(len(FAR) + 1))
def test_key_that_decides(case, dtype):
    sizes, rotated = FAR[case % len(FAR)][:5], case == len(FAR)
    *_, pos, n = sizes
    m = None
    for at in far_places(*sizes):
        cfg, w, toks, want = far(*sizes, at, rotated)
        m = m or build(cfg, w, dtype, capacity=pos + n)              # (the weights are the same for every place)
        m.forward(0, toks[:pos], 0)
        assert M.error(m.forward(0, toks[pos:], pos, range(n)), want) < LIMIT[dtype], f"key at {at}"
        # without it, whoever sees it has other logits
        toks, seen = [t or 1 for t in toks], max(at - pos, 0)
        m.forward(0, toks[:pos], 0)
        other = m.forward(0, toks[pos:], pos, range(n)).cpu()
        assert ((other - want)[seen:].pow(2).mean(-1).sqrt() / want.std()).min() > 0.2, f"key at {at}"
