"""The prompt attention kernel (several tokens of one sequence, head_dim 32,
64 or 128) through the decoder model: against the oracle's engine, and bit
for bit against the kernel of single tokens."""
import numpy as np
import pytest

import lcengine as E
import leafcutterllm_amd as L
from leafcutterllm_amd.configs import ModelConfig, small_config, synth_model
from test_oracle_engine import rel, spec

pytestmark = pytest.mark.gpu

LOGIT_TOL = 1e-3


def _model_config(hd, H, KVH, qt):
    return ModelConfig("prompt", 2, H, KVH, hd, 64, 10000.0,
                       small_config("prompt", 256, 256, 8, 2, L.ROUTE_SOFTMAX_RENORM, L.TYPE_Q8_0,
                                    L.TYPE_Q8_0), attn_type=qt)


# T below the kernel's fewest tokens, above them, and past two 128-position
# chunks; then a second prompt on a filled cache
@pytest.mark.parametrize("T", [15, 16, 31, 32, 33, 65, 290])
@pytest.mark.parametrize("hd,H,KVH,qt", [(32, 4, 2, L.TYPE_Q8_0), (64, 4, 4, L.TYPE_Q4_K),
                                         (128, 2, 1, L.TYPE_Q4_K)])
def test_prompt_attention_matches_oracle(hd, H, KVH, qt, T):
    mc = _model_config(hd, H, KVH, qt)
    w = synth_model(mc, seed=hd + T)
    ref = E.RefEngine(spec(mc, E.ROPE_ABSOLUTE), w, threads=8)
    with L.Model(mc.desc(1, 320, 400, E.ROPE_ABSOLUTE), w) as m:
        for c in ([(7 * i + 3) % 64 for i in range(T)], [(5 * i + 1) % 64 for i in range(37)], [9]):
            g = m.forward(np.array([c]))[0]
            assert rel(g, ref.forward(c).astype(np.float64)) < LOGIT_TOL


# T and the cached tokens before it around the kernel's fewest tokens, its
# 4-query tiles and the 128-position chunks
@pytest.mark.parametrize("cached", [0, 100, 128])
@pytest.mark.parametrize("T", [39, 40, 42, 43, 129, 273])
@pytest.mark.parametrize("hd,H,KVH", [(32, 8, 2), (64, 4, 4), (128, 2, 1)])
def test_prompt_attention_is_the_one_token_kernel(hd, H, KVH, T, cached):
    """A prompt's logits have the bits of the same prompt with its last token
    in a call of its own: attention runs every sum in one order (the Q8_0
    products and experts of the decoder take each token alone anyway)."""
    mc = _model_config(hd, H, KVH, L.TYPE_Q8_0)
    w = synth_model(mc, seed=hd)
    tok = np.random.default_rng(T + cached).integers(0, 64, (1, cached + T)).astype(np.int32)
    with L.Model(mc.desc(1, 300, 420, E.ROPE_ABSOLUTE), w) as m:
        out = []
        for cut in (cached + T, cached + T - 1):
            m.reset()
            if cached:
                m.forward(tok[:, :cached])
            if cut > cached:
                out.append(m.forward(tok[:, cached:cut])[0])
            if cut < cached + T:
                out[-1] = m.forward(tok[:, cut:])[0]
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_infinite_value_stays_with_its_readers(sign):
    """A token whose V leaves f16's range reaches only the queries that see
    it: the routing of every earlier token, in every layer, is that of the
    prompt without it."""
    mc = _model_config(64, 4, 4, L.TYPE_F32)
    w = synth_model(mc, seed=3)
    d, A, j, T = 256, 63, 17, 40
    embd = w["token_embd"].view(np.float32).reshape(64, d)
    embd[A] = 0
    embd[A, j] = sign
    for lw in w["layers"]:
        lw["attn_norm"][j] = 100.0
        lw["attn_v"].view(np.float32).reshape(-1, d)[5, j] = 100.0  # 16 * 100 * 100 past 65504
    tok = [(7 * i + 3) % 61 for i in range(T - 1)]
    seen = []
    with L.Model(mc.desc(1, 64, 64, E.ROPE_ABSOLUTE), w) as m:
        for c in (tok, tok + [A]):
            m.reset()
            logits = m.forward(np.array([c]))[0]
            seen.append([m.layer_routing(l) for l in range(2)])
    assert not np.all(np.isfinite(logits))
    for a, b in zip(*seen):
        assert np.array_equal(a["topk_idx"], b["topk_idx"][:T - 1])
        np.testing.assert_allclose(b["topk_w"][:T - 1], a["topk_w"], rtol=1e-4)


@pytest.mark.parametrize("cut", [0, 128])
def test_nan_score_alone_in_its_chunk(cut):
    """A token whose own key scores NaN (K past f16's range with contributions
    of both signs) at position 128, the only one its query sees in that
    128-position chunk: its logits are not finite, in a prompt and in a call
    of one token."""
    mc = _model_config(64, 4, 4, L.TYPE_F32)
    w = synth_model(mc, seed=4)
    d, A, j, T = 256, 63, 17, 129
    embd = w["token_embd"].view(np.float32).reshape(64, d)
    embd[A] = 0
    embd[A, j] = 1.0
    for lw in w["layers"]:
        lw["attn_norm"][j] = 100.0
        lw["attn_k"].view(np.float32).reshape(-1, d)[:, j] = 100.0  # 16 * 100 * 100 past 65504
    tok = np.array([[(7 * i + 3) % 61 for i in range(T - 1)] + [A]])
    with L.Model(mc.desc(1, 160, 160, E.ROPE_ABSOLUTE), w) as m:
        if cut:
            assert np.all(np.isfinite(m.forward(tok[:, :cut])))
        assert not np.any(np.isfinite(m.forward(tok[:, cut:])))
