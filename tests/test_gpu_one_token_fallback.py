"""The exact chains of one uncertified token in the parallel-bounds router:
tiles of 32 experts over a block's four waves."""
import numpy as np
import pytest

import leafcutterllm_amd as L
from parity_util import run_and_check

pytestmark = pytest.mark.gpu


# E of one tile to eight (two rounds of the waves), whole and partial last
# tiles, with and without the four mul-then-add columns of E % 8 = 4; two
# experts tie in the lead, so no bound orders them
@pytest.mark.parametrize("E,d", [(32, 256), (36, 7168), (60, 2048), (64, 512), (100, 512),
                                 (128, 256), (132, 512), (248, 256), (256, 512)])
def test_one_token_exact_chains(E, d):
    cfg = L.configs.small_config("fb1", d, 256, E, 4, L.ROUTE_SOFTMAX_RENORM, L.TYPE_Q4_K,
                                 L.TYPE_Q4_K)
    layer = L.synth_layer(cfg, seed=E)
    x = L.synth_x(cfg, 1, seed=E, index=d)
    r = layer["router"].copy()
    # experts 1 and 2: one row, in the lead; the last two experts' logits are
    # selected next and lie apart, at the end of the last tile
    r[:, 1] = 4.0 * np.sign(x[0]) / np.sqrt(d)
    r[:, 2] = r[:, 1]
    r[:, E - 1] = 0.75 * r[:, 1]
    r[:, E - 2] = 0.5 * r[:, 1]
    layer["router"] = r
    with L.MoeFfn(cfg.desc(1), layer) as moe:
        res = run_and_check(cfg, layer, x, moe=moe)
        assert moe.route_fallbacks() == 1
    assert res["topk_idx"].reshape(-1).tolist() == [1, 2, E - 1, E - 2]
