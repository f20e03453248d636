"""Projections of latent attention of 256 MB and more, whose rows go from the last to the first and past the caches, against the oracle and against the same
tokens in portions that stay below that: rows of up to four and of up to eight groups of values per thread."""
import functools

import pytest
import torch

from tests import kagapel_models as M
from tests.test_gpu_kagapel import DTYPES, IDS, LIMIT, build

N = 4100


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("dim", [16, 100])
def test_large_projections(dim, dtype):
    heads, rot, vdim, rank = 64, 8, 250, 24
    cfg = M.model(48, 51, [M.gated(heads, dim, rot, vdim, rank, ff=24)], positions=N)
    values = heads * (dim + rot) + rank + rot
    assert (values > 4096) == (dim == 100) and values <= 8192 and N * (values + heads * vdim) * 4 >= 256 << 20 > 1025 * (values + heads * vdim) * 4
    w, toks = M.weights(cfg, 5), M.prompt(cfg, N, 6)
    whole = build(cfg, w, dtype, capacity=N, max_portion=N).forward(0, toks, 0, range(N))
    m = build(cfg, w, dtype, capacity=N, max_portion=1025)
    parts = torch.cat([m.forward(0, toks[i:i + 1025], i, range(1025)) for i in range(0, N, 1025)])
    assert M.error(whole, parts.double().cpu()) < LIMIT[dtype]


@functools.lru_cache(maxsize=None)
def many_heads(dim):
    heads, rot, vdim, rank, n = 128, 8, 250, 24, 1950
    cfg = M.model(48, 51, [M.gated(heads, dim, rot, vdim, rank, ff=24)], positions=n)
    values = heads * (dim + rot) + rank + rot
    assert (values > 4096) == (dim == 50) and values <= 8192 and n * (values + heads * vdim) * 4 >= 256 << 20
    w, toks = M.weights(cfg, 5), M.prompt(cfg, n, 6)
    return cfg, w, toks, M.oracle(cfg, w, toks)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("dim", [16, 50])
def test_large_projections_and_the_oracle(dim, dtype):
    cfg, w, toks, want = many_heads(dim)
    m = build(cfg, w, dtype, capacity=len(toks), max_portion=len(toks))
    assert M.error(m.forward(0, toks, 0, range(len(toks))), want) < LIMIT[dtype]
