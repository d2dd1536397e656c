"""Passes of at most 8 tokens with two f16 per activation: the hi and lo
halves packed into one matrix-core operand."""
import pytest

import leafcutterllm_amd as L
from parity_util import run_and_check

pytestmark = pytest.mark.gpu


# every token at the same expert: T tokens in one pass, both sides of 8; F
# whole super-blocks or the split layout; more experts than tokens take the
# row-per-lane kernels, hence E = 1
@pytest.mark.parametrize("F", [512, 384])
@pytest.mark.parametrize("T", [4, 7, 8, 9, 16, 17, 40])
def test_packed_pass_edges(T, F):
    cfg = L.configs.small_config("packed", 768, F, 1, 1, L.ROUTE_SOFTMAX_RENORM, L.TYPE_Q4_K,
                                 L.TYPE_Q4_K)
    layer = L.synth_layer(cfg, seed=T)
    x = L.synth_x(cfg, T, seed=T, index=F)
    with L.MoeFfn(cfg.desc(T), layer) as moe:
        moe.set_act_precision(L.ACT_F16X2)
        res = run_and_check(cfg, layer, x, moe=moe)
    # two f16 hold an activation to about 22 bits: 3e-6 at the largest shapes
    assert res["rel_l2"] < 1e-5
