"""Residual streams of portions of many tokens (32 MB and more), which are stored after the feed-forward only: two to four of them, in rows of two and of four
groups of values per thread, layers with and without a feed-forward and with experts, a portion on either side of the line."""
import pytest
import torch

from tests import kagapel_models as M
from tests import seq_plan as P
from tests.test_gpu_kagapel import DTYPES, IDS, LIMIT, build, grouped_layer_in_streams

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


def later(n, streams, width, portion, projected, mixed, bf16):
    """The streams of n tokens are large, and the mixer's whole output, a product of rows of `mixed` values, fits the buffer of `projected` values per token."""
    return n * streams * width * 4 >= 32 << 20 and n * width <= P.room(portion, projected) and P.product(width, n, mixed, bf16, P.room(portion, width))[3] == 1


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("streams,width,portions", SIZES, ids=str)
def test_streams_wait_in_a_wide_projection(streams, width, portions, dtype):
    mixers = [(20, 40, 8, 40, 24), (3, 16, 8, 16, 24), (2, 16, 8, 24, 24)]
    cfg = M.model(width, 51, [M.gated(*mixers[0], ff=40), M.sunk(*mixers[1]), M.sunk(*mixers[2], ff=24)], streams=streams, positions=1700)
    projected = 20 * 48 + 32 + 20 * 40
    w, toks, res = M.weights(cfg, 5), M.prompt(cfg, max(portions), 6), []
    want = M.oracle(cfg, w, toks, res)
    for heads, _, _, vdim, _ in mixers:
        assert [later(n, streams, width, 1700, projected, heads * vdim, dtype == torch.bfloat16) for n in portions] == [True, False][:len(portions)]
    for n in portions:
        logits, layers = build(cfg, w, dtype, capacity=1700).forward(0, toks[:n], 0, range(n), residuals=True)
        assert M.error(logits, want[:n]) < LIMIT[dtype]
        for got, r in zip(layers, res):
            assert M.error(got, r[:n]) < LIMIT[dtype]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
def test_streams_with_experts(dtype):
    from clusterfusionplus_amd.seq_model import SeqModel
    n, width, streams, capacity = 1400, 1536, 4, 1500
    pack, forward, vocab = grouped_layer_in_streams(width, streams, heads=40)
    assert later(n, streams, width, capacity, 40 * 24 + 2 * 40, 40 * 16, dtype == torch.bfloat16) and later(n, streams, width, capacity, 40 * 24 + 2 * 40, 2 * 16, dtype == torch.bfloat16)
    toks = torch.randint(0, vocab, (n,), generator=torch.Generator().manual_seed(4)).tolist()
    assert M.error(SeqModel(pack(dtype), capacity=capacity).forward(0, toks, 0, range(n)), forward(toks)) < LIMIT[dtype]
