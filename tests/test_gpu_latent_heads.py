"""One token's latent attention with many heads: on both sides of two workgroups of k_seq_latent_out per compute unit (512), heads of more outputs than a workgroup has."""
import pytest
import torch

from tests import kagapel_models as M
from tests.test_gpu_kagapel import DTYPES, IDS, LIMIT, build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", DTYPES, ids=IDS)
@pytest.mark.parametrize("heads,vdim", [(512, 16), (513, 16), (257, 17)], ids=str)
def test_steps_with_many_heads(heads, vdim, dtype):
    cfg = M.model(64, 51, [M.sunk(heads, 8, 8, vdim, 40)])
    w, toks = M.weights(cfg, 5), M.prompt(cfg, 70, 6)
    want = M.oracle(cfg, w, toks)
    m = build(cfg, w, dtype)
    m.forward(0, toks[:60], 0, [59])
    got = torch.cat([m.forward(0, [toks[i]], i, [0]) for i in range(60, 70)])
    assert M.error(got, want[60:]) < LIMIT[dtype]
