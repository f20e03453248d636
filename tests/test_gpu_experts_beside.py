"""The shared expert's products in the experts' launches and behind them: the oracle's results by either way.  Which way each case takes
stands with it; tests/test_seq_plan.py holds the table to the plan."""
import functools

import pytest
import torch

from tests import nibotar_models as M
from tests import seq_plan as P
from tests.test_gpu_nibotar import DTYPES, IDS, LIMIT, build

pytestmark = pytest.mark.gpu
WIDTH, FF, EXPERTS, TOP, PORTION = 192, 72, 24, 3, 1300
TOKENS = (2, 15, 16, 17, 64, 65, 129, 500, 1200)
# (the shared expert's inner size, bf16): for each of the counts, b: both of its products are beside the experts', u: the up rows only, -: neither
WAYS = {(1, True): "bbbbbbbbb", (40, True): "bbbbbbbbb", (72, True): "bbbbbbbbb", (900, True): "uuuuuuuu-", (2500, True): "uuuuuuu--",
        (1, False): "bbbbbbbbb", (40, False): "bbbbbbbbb", (72, False): "bbbbbbbbb", (900, False): "uuuuuuu-u", (2500, False): "uuuuuuu--"}


def way(n, shared, bf16):
    """What the library decides for a portion of n tokens."""
    x, h, hs = (P.row_bytes(k, bf16) for k in (WIDTH, FF, shared))
    up, down = (bool(P.lib().beside(n, TOP, EXPERTS, FF, x, *sizes, bf16, P.CUS)) for sizes in ((2 * FF, x, 2 * shared, x, 0, 0), (WIDTH, h, WIDTH, hs, WIDTH, P.room(PORTION, WIDTH))))
    return {(True, True): "b", (True, False): "u", (False, False): "-", (False, True): "d"}[up, down]


@functools.lru_cache(maxsize=None)
def reference(shared):
    cfg = M.model(WIDTH, 97, [(M.attn(2, 1, 64, 64), M.moe(FF, EXPERTS, TOP, shared=shared))] * 2)
    w, toks = M.weights(cfg, 7), M.prompt(cfg, 1200, 8)
    return cfg, w, toks, M.oracle(cfg, w, toks)


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("shared", sorted({shared for shared, _ in WAYS}))
def test_shared_beside_and_behind(shared, dtype):
    cfg, w, toks, want = reference(shared)
    m = build(cfg, w, dtype, capacity=PORTION, max_portion=PORTION)
    for n in TOKENS:
        assert M.error(m.forward(0, toks[:n], 0, range(n)), want[:n]) < LIMIT[dtype], f"{n} tokens"
