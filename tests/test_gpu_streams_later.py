"""Residual streams of portions of many tokens (32 MB and more), which are stored after the feed-forward only: two to four of them, in rows of two and of four
groups of values per thread, layers with and without a feed-forward, a portion on either side of the line."""
import pytest
import torch

from tests import kagapel_models as M
from tests.test_gpu_kagapel import DTYPES, IDS, LIMIT, build

SIZES = [(4, 1536, (1366, 1365)), (3, 2052, (1363, 1362)), (2, 2560, (1639, 1638)), (4, 4096, (513,))]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("streams,width,portions", SIZES, ids=str)
def test_streams(streams, width, portions, dtype):
    cfg = M.model(width, 51, [M.gated(2, 16, 8, 16, 24, ff=40), M.sunk(3, 16, 8, 16, 24), M.sunk(2, 16, 8, 24, 24, ff=24)], streams=streams, positions=1700)
    w, toks, res = M.weights(cfg, 5), M.prompt(cfg, max(portions), 6), []
    want = M.oracle(cfg, w, toks, res)
    assert {n * streams * width * 4 >= 32 << 20 for n in portions} == ({True, False} if len(portions) == 2 else {True})
    for n in portions:
        logits, layers = build(cfg, w, dtype, capacity=1700).forward(0, toks[:n], 0, range(n), residuals=True)
        assert M.error(logits, want[:n]) < LIMIT[dtype]
        for got, r in zip(layers, res):
            assert M.error(got, r[:n]) < LIMIT[dtype]
