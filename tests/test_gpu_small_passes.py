"""Passes of few tokens with two f16 per activation."""
import numpy as np
import pytest

import leafcutterllm_amd as L
from leafcutterllm_amd.configs import ModelConfig, small_config, synth_model
from parity_util import run_and_check

pytestmark = pytest.mark.gpu


# T tokens in one pass of the one expert, around the 8- and 16-token marks; F
# whole super-blocks or the split layout
@pytest.mark.parametrize("F", [512, 384])
@pytest.mark.parametrize("T", [4, 7, 8, 9, 16, 17, 40])
def test_two_f16_pass_edges(T, F):
    cfg = L.configs.small_config("small", 768, F, 1, 1, L.ROUTE_SOFTMAX_RENORM, L.TYPE_Q4_K,
                                 L.TYPE_Q4_K)
    layer = L.synth_layer(cfg, seed=T)
    x = L.synth_x(cfg, T, seed=T, index=F)
    with L.MoeFfn(cfg.desc(T), layer) as moe:
        moe.set_act_precision(L.ACT_F16X2)
        res = run_and_check(cfg, layer, x, moe=moe)
    # two f16 hold an activation to about 22 bits: 3e-6 at the largest shapes
    assert res["rel_l2"] < 1e-5


@pytest.mark.parametrize("F", [512, 384])
def test_token_is_independent_of_its_pass(F):
    """A token's output has the same bits however many tokens share its pass
    (2 to 16): every sum over its row runs in one order."""
    cfg = small_config("pass", 768, F, 1, 1, L.ROUTE_SOFTMAX_RENORM, L.TYPE_Q4_K, L.TYPE_Q4_K)
    layer = L.synth_layer(cfg, seed=F)
    x = L.synth_x(cfg, 16, seed=F, index=1)
    with L.MoeFfn(cfg.desc(16), layer) as moe:
        moe.set_act_precision(L.ACT_F16X2)
        full = moe.forward(x)[0]
        for T in range(2, 16):
            assert np.array_equal(moe.forward(x[:T])[0], full[:T]), T


def test_decoder_row_is_independent_of_the_batch():
    """The decoder's logits of a sequence have the same bits in a batch of 4 to
    12 (the K slices of its products depend on the shapes and, past 32 rows,
    on the rows; below 4 rows the experts take other kernels)."""
    mc = ModelConfig("rows", 2, 4, 2, 64, 256, 10000.0,
                     small_config("rows", 256, 512, 8, 2, L.ROUTE_SOFTMAX_RENORM, L.TYPE_Q4_K,
                                  L.TYPE_Q4_K))
    w = synth_model(mc, seed=21)
    tok = np.array([[(13 * i + 29 * b + 7) % mc.vocab for i in range(5)] for b in range(12)])

    def logits(m, B):
        m.reset()
        return np.stack([m.forward(tok[:B, i:i + 1]) for i in range(5)], axis=1)

    with L.Model(mc.desc(12, 8, 16, 1), w) as m:
        full = logits(m, 12)
        for B in (4, 5, 8, 9):
            assert np.array_equal(logits(m, B), full[:B]), B
