"""The choices that a portion's kernels are launched with (csrc/seq_plan.hpp), on the host."""
import os
import random
import re

import pytest

from clusterfusionplus_amd import build
from tests import seq_plan as P
from tests import test_gpu_experts_beside as B
from tests import test_gpu_portion_attention as A
from tests import test_gpu_products as G

ROOM = 1 << 24


def splits(T, R, G, pos, chunk, keys=64, room=ROOM, vdim=128):
    floats = T * R * G * (vdim + 2)
    n, columns = P.attention(T, R, G, pos, chunk, keys, floats, room)
    assert 1 <= n <= 16 and (n == 1 or n * floats <= room)
    return n, columns


def walks(T, R, pos, chunk, keys, columns):
    """Tiles of keys that every workgroup's columns walk."""
    out = []
    for c0 in range(0, T * R, columns):
        first, last = pos + c0 // R, pos + min(T - 1, (c0 + columns - 1) // R)
        out.append((last + 1 - (first // chunk * chunk if chunk else 0) + keys - 1) // keys)
    return out


@pytest.mark.parametrize("pos, chunk, want", [(8192, 8192, 1), (8193, 8192, 1), (8192 + 219, 8192, 2), (1990, 8192, 16), (8192 + 1990, 8192, 16), (8150, 8192, 16),
                                              (8170, 8192, 16), (0, 0, 1), (1990, 0, 16), (100, 40, 1), (1000, 300, 1)])
def test_splits_follow_what_a_short_portion_sees(pos, chunk, want):
    """37 tokens, four query heads to each of eight key heads: a chunk's first tokens see that chunk only."""
    assert splits(37, 4, 8, pos, chunk)[0] == want


def test_every_split_of_the_longest_walk_has_two_tiles():
    rng = random.Random(3)
    for _ in range(3000):
        T, R, G = rng.choice([2, 5, 37, 64, 65, 150, 301, 700]), rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 8, 16, 32])
        chunk, keys = rng.choice([0, 1, 7, 100, 1000, 8192]), rng.choice([32, 64])
        pos = rng.randrange(0, 20000)
        n, columns = splits(T, R, G, pos, chunk, keys)
        assert n == 1 or n <= max(walks(T, R, pos, chunk, keys, columns)) // 2, (T, R, G, pos, chunk, keys, n)


def test_order_of_the_workgroups():
    """Every row of workgroups is there once.  Workgroups i and i + 256 share a compute unit: where all are resident, two such walks are little longer
    than the longest alone; where less than one per unit is left over and walks are alike, the younger of the two is the longer one and the shortest
    are left over; otherwise the longest are first."""
    rng, kinds = random.Random(4), set()
    for T, R, G, keys, pos, chunk in [(1000, 1, 16, 32, 0, 0), (1000, 4, 8, 32, 0, 0), (1500, 2, 5, 32, 0, 0), (700, 3, 4, 32, 0, 0), (3000, 1, 300, 64, 0, 0), (1150, 1, 32, 32, 1990, 0),
                                      (1500, 1, 32, 32, 1990, 0), (1500, 1, 32, 32, 1990, 3000), (1500, 1, 32, 32, 1990, 3490), (1500, 1, 32, 32, 749, 0), (1100, 1, 40, 64, 550, 0), (66, 1, 300, 64, 64, 0), (10, 1, 600, 64, 20, 0), (64, 1, 768, 32, 64, 0), (65, 1, 257, 32, 64, 0), (100, 1, 384, 64, 64, 0)] + \
            [(rng.randint(2, 4000), rng.choice([1, 2, 4, 8]), rng.choice([1, 2, 3, 5, 8, 12, 16, 32, 40]), rng.choice([32, 64]), rng.choice([0, 100, 1000, 3000]), rng.choice([0, 0, 2000, 8192])) for _ in range(600)] + \
            [(rng.randint(2, 200), 1, rng.randint(100, 4096), rng.choice([32, 64]), rng.choice([0, 100, 3000]), 0) for _ in range(300)]:
        n, columns, order = P.attention_plan(T, R, G, pos, chunk, keys, T * R * G * 130, ROOM)
        rows, what = len(order), (T, R, G, keys, pos, chunk)
        assert sorted(order) == list(range(rows)), what
        blocks = [block for block in order for _ in range(G * n)]
        alike = 2 * (pos - (pos // chunk * chunk if chunk else 0)) >= T and not (chunk and pos // chunk != (pos + T - 1) // chunk)
        if len(blocks) <= 2 * P.CUS:
            kinds.add("resident")
            assert max(blocks[i] + sum(blocks[i + P.CUS:i + P.CUS + 1]) for i in range(min(P.CUS, len(blocks)))) <= rows, what
        elif len(blocks) <= 3 * P.CUS and alike:
            kinds.add("left over")
            some = min(P.CUS // G or 1, rows // 2) * G
            assert n == 1 and all(blocks[i] < blocks[i + some] for i in range(some)) and max(blocks[2 * some:], default=-1) < min(blocks[:2 * some], default=rows), what
        else:
            kinds.add("many")
            assert n == 1 and blocks == sorted(blocks, reverse=True), what
    assert len(kinds) == 3


def test_attention_in_blocks_of_32():
    """The cases of its test take them, in every size of tile, and their keys are never split."""
    seen = set()
    for name, (model, mixer) in A.BLOCKS.items():
        m = mixer.get("mixer", mixer)
        R, G = (1, m["heads"]) if "mixer" in mixer else (m["heads"] // m["kv_heads"], m["kv_heads"])
        for n, pos in ((900, 0), (907, 900)):
            assert splits(n, R, G, pos, m.get("mask", {}).get("size", 0), vdim=m["vdim"])[1] == 128, name
        keys, values = m["dim"] + m.get("rot_dim", 0), m["vdim"]
        tile = next(t for t in ((64, 64), (128, 128), (192, 128), (256, 256)) if keys <= t[0] and values <= t[1])
        seen.add((*tile, "mixer" in mixer))
    assert seen == {(*t, latent) for t in ((64, 64), (128, 128), (192, 128), (256, 256)) for latent in (False, True)}
    rng = random.Random(6)
    for _ in range(500):
        n, columns = splits(rng.randint(2, 8000), rng.choice([1, 2, 4]), rng.choice([1, 8, 16, 32, 128]), rng.randrange(0, 9000), rng.choice([0, 8192]))
        assert columns == 64 or n == 1


def test_attention_with_workgroups_left_over():
    """What its test is for."""
    first, n = A.LEFT_OVER_TOKENS
    for keys in (32, 64):
        for chunk in (0, 1000):
            assert P.attention_plan(n, 1, 64, first, chunk, keys, n * 64 * 130, ROOM) == (1, 64, [5, 4, 3, 2, 9, 8, 7, 6, 1, 0])


# ---- the tiles that the products' tests are for --------------------------------------------------------------------------

@pytest.mark.parametrize("sizes, tile", list(zip(G.DENSE, G.DENSE_TILES)), ids=str)
def test_tiles_of_up_rows(sizes, tile):
    n, width, ff, vocab = sizes
    if sizes == (700, 300, 4001, 51):                # (here it is the down rows)
        assert P.product(width, n, ff, True, P.room(n, width))[:3] == tile
    else:
        assert P.product(ff, n, width, True) == (*tile, 1)
        if vocab > 10000:
            assert P.product(vocab, n, width, True) == (*tile, 1)


@pytest.mark.parametrize("sizes, tile", G.SPLIT, ids=str)
def test_tiles_of_split_rows(sizes, tile):
    n, width, ff = sizes
    assert P.product(width, n, ff, True, P.room(4 * n, width)) == tile
    assert P.product(width, n, ff, False, P.room(4 * n, width))[3] > 1


@pytest.mark.parametrize("sizes, tile", G.GATED, ids=str)
def test_tiles_of_gated_rows(sizes, tile):
    n, width, ff = sizes
    assert P.product(2 * ff, n, width, True) == (*tile, 1)
    down = P.product(width, n, ff, True, P.room(n, width))
    assert down[3] > 1 and (width < 8000 or down[:2] == (256, 256))


@pytest.mark.parametrize("sizes, tile", G.HEADS, ids=str)
def test_tiles_of_keys_and_values(sizes, tile):
    heads, dim, vdim, rank, n = sizes
    assert P.product(heads * (dim + vdim), n, rank, True) == (*tile, 1)


@pytest.mark.parametrize("sizes, tile", G.EXPERT_TILES, ids=str)
def test_tiles_of_experts(sizes, tile):
    assert P.experts(*sizes, True) == tile


@pytest.mark.parametrize("sizes, tile", G.HEAD, ids=str)
def test_tiles_of_the_head(sizes, tile):
    n, width, vocab = sizes
    assert P.product(vocab, n, width, True) == (*tile, 1)


def test_tiles_of_two_products_in_a_launch():
    """Every tile in which the shared expert's product is put beside the experts' has kernels for both, in either kind of product."""
    with open(build.SEQ_LIB, "rb") as f:
        kernels = {(m[1] != b"f", int(m[2]), int(m[3])) for m in re.finditer(rb"k_seq_gemm_besideI(\w+?)Li(\d+)ELi(\d+)E", f.read())}
    rng, beside = random.Random(7), set()
    for _ in range(4000):
        n, top, count = rng.choice([2, 5, 16, 17, 40, 64, 65, 129, 150, 300, 700, 2000]), rng.randint(1, 8), rng.choice([1, 2, 3, 8, 24, 64])
        ff, shared, width, bf16 = rng.choice([60, 700, 1408, 4000]), rng.choice([1, 60, 700, 2816, 6000]), rng.choice([60, 192, 2048, 4096]), rng.random() < 0.5
        a = (n, min(top, count), count, ff, P.row_bytes(width, bf16))
        for sizes in ((2 * ff, a[4], 2 * shared, a[4], 0, 0), (width, P.row_bytes(ff, bf16), width, P.row_bytes(shared, bf16), width, P.room(n, width))):
            if P.lib().beside(*a, *sizes, bf16, P.CUS):
                beside.add((bf16, *P.experts(n, a[1], count, ff, width, bf16)[:2]))
    assert beside == kernels, beside ^ kernels


def test_ways_of_shared_experts():
    """The ways that the shared experts' test is for."""
    for (shared, bf16), ways in B.WAYS.items():
        assert "".join(B.way(n, shared, bf16) for n in B.TOKENS) == ways, (shared, bf16)


def test_every_tile_is_tested_in_every_kind_of_product():
    tiles = {(64, 16, 2), (64, 32, 2), (64, 64, 2), (64, 96, 2), (256, 96, 1), (128, 128, 2), (256, 128, 1), (256, 256, 1), (128, 64, 2), (96, 128, 1), (128, 128, 1),
             (128, 192, 1), (192, 160, 1), (96, 160, 1)}
    assert {P.tile(i, True) for i in range(len(tiles))} == tiles
    small = {(64, 16, 2)}                            # (what everything takes in the other tests' small models)
    whole = {(128, 128, 2)}                          # (of its size, the tile that is alone on a compute unit is the one to split)
    head = {t for s, t in zip(G.DENSE, G.DENSE_TILES) if s[3] > 10000}
    for name, seen in (("up", set(G.DENSE_TILES)), ("split", {t[:3] for _, t in G.SPLIT} | whole), ("gated", {t for _, t in G.GATED} | small),
                       ("keys and values", {t for _, t in G.HEADS} | small), ("experts", {t[:3] for _, t in G.EXPERT_TILES}), ("head", head | {t for _, t in G.HEAD} | small)):
        assert seen == tiles, (name, tiles - seen)


def test_split_rows_of_wide_models():
    n, ff = G.ROWS
    for width in G.WIDTHS + [w for w, _ in G.STREAMS]:
        for bf16 in (True, False):
            assert P.product(width, n, ff, bf16, P.room(100, width))[3] > 1, (width, bf16)


def test_projections_in_parts():
    """The parts that every size of row has in its tests: some added in one round of three, some in two."""
    for values, (heads, kv_heads, dim, vdim) in A.PARTS_ROWS.items():
        assert heads * dim + kv_heads * (dim + vdim) == values
        for bf16 in (True, False):
            parts = {P.product(values, n, width, bf16, P.room(100, values))[3] for n in A.PARTS_TOKENS for width in A.PARTS_WIDTHS}
            assert 1 not in parts and len(parts) > (values < 8192) and (values > 4100 or max(parts) > 4), (values, bf16, parts)


def test_no_split_of_less_than_three_steps_or_more_than_its_room():
    rng = random.Random(5)
    for _ in range(3000):
        n, m, k, bf16 = rng.randint(1, 60000), rng.choice([2, 3, 17, 65, 100, 300, 1000, 4000]), rng.randint(1, 16000), rng.random() < 0.5
        floats = rng.choice([0, m * n, 4 * m * n, 16 << 20])
        rows, tokens, resident, sp = P.product(n, m, k, bf16, floats)
        assert sp == 1 or (sp * m * n <= floats and P.row_bytes(k, bf16) // 128 // sp >= 3)


def test_workgroups_that_share_a_compute_unit_fit_its_memory():
    """The table's workgroups per compute unit, and the LDS that the launches ask for (the figures of the resource report)."""
    with open(os.path.join(build.CSRC, "seq_kernels.hip")) as f:
        text = f.read()
    for bf16, part in ((True, text[text.index("switch (shape)"):text.index("} else {", text.index("switch (shape)"))]), (False, text[text.index("} else {", text.index("switch (shape)")):])):
        launches = {int(i): args for i, args in re.findall(r"case (\d+): return launch_gemm<T, ([\d, ]+), EPI>", part)}
        launches.setdefault(7 if bf16 else 3, None if bf16 else re.search(r"launch_gemm<T, (128, [\d, ]+), EPI>\(g", part)[1])
        assert len(launches) == (14 if bf16 else 4)
        for i, args in launches.items():
            rows, tokens, resident = P.tile(i, bf16)
            assert args is None or args.startswith(f"{rows}, {tokens}, ")
            lds, waves = build.launch_lds(f"k_seq_gemm<{'bf16' if bf16 else 'float'}, {args}, 0>" if args else "k_seq_gemm8<0>")
            assert resident * lds <= build.LDS_BYTES, (rows, tokens)


def test_lds_of_launches():
    assert build.launch_lds("k_seq_gemm<bf16, 96, 128, 2, 2, 5, 0>") == (143360, 4) and build.launch_lds("k_seq_gemm8<3>") == (131072, 8)
    assert build.launch_lds("k_seq_attn<bf16, 192, 128, 32, true>") == (81920, 4) and build.launch_lds("k_seq_attn<float, 256, 256, 16, false>") == (131072, 4)
    assert build.launch_lds("k_seq_latent_attn<bf16, 512, 4>") == (135168, 4)
    assert build.launch_lds("k_seq_latent_finish4<bf16, 12, 1>") == (49664, 4) and build.launch_lds("k_seq_latent_finish4<float, 4, 3>") == (16896, 4)
    assert build.launch_lds("k_seq_postnorm<bf16>")[0] is None and build.launch_lds("k_seq_postnorm4<bf16, 8>") is None and build.launch_lds("k_fused<1>") is None
