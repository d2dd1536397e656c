"""The certified softmax router with several blocks per token, its block-wide
fused norm, and the one-wave dispatch."""
import numpy as np
import pytest

import lcoracle as O
import leafcutterllm_amd as L
from parity_util import run_and_check

pytestmark = pytest.mark.gpu


def _cfg(d, E, K, kind=L.ROUTE_SOFTMAX):
    return L.configs.small_config("split", d, 256, E, K, kind, L.TYPE_Q4_K, L.TYPE_Q4_K)


# T around the splits (8, 4, 2, 1 blocks per token while they fit 256 CUs) and
# T * K around the one-wave dispatch's 256 assignments; E of whole and partial
# groups of 8; with two equal columns among the multiply-add chains (the first
# E // 8 * 8) tokens that rank both of them fall back to the exact chains
@pytest.mark.parametrize("T", [2, 31, 33, 63, 65, 127, 129])
@pytest.mark.parametrize("d,E,K", [(256, 33, 4), (512, 60, 2), (1024, 64, 8), (2048, 60, 4)])
def test_split_router_parity(d, E, K, T):
    cfg = _cfg(d, E, K)
    layer = L.synth_layer(cfg, seed=E + T)
    if T % 2 and T > 2:
        layer["router"][:, E // 8 * 8 - 1] = layer["router"][:, 0]
    run_and_check(cfg, layer, L.synth_x(cfg, T, seed=T, index=d))


# certified tokens and tokens that fall back side by side in one launch: experts
# 1 and 2 share a row, which leads for every odd token (no bound orders the
# pair) and comes last for the others.  One block per token and several.
@pytest.mark.parametrize("T", [2, 17, 100, 130, 257])
@pytest.mark.parametrize("d,E,K", [(256, 8, 2), (512, 16, 4), (1024, 60, 4), (2048, 64, 2)])
def test_certified_and_exact_tokens_together(d, E, K, T):
    cfg = _cfg(d, E, K)
    layer = L.synth_layer(cfg, seed=d + T)
    x = L.synth_x(cfg, T, seed=T, index=d)
    u = np.where(np.arange(d) % 2, 1.0, -1.0).astype(np.float32) / np.float32(np.sqrt(d))
    router = layer["router"].copy()
    router[:, 1] = router[:, 2] = u
    layer["router"] = router
    x -= np.outer(x @ u, u)
    x += np.outer(np.where(np.arange(T) % 2, 8.0, -8.0), u)
    idx = run_and_check(cfg, layer, x.astype(np.float32))["topk_idx"].reshape(T, K)
    assert np.all(idx[1::2, :2] == [1, 2])
    assert not np.any(np.isin(idx[::2], [1, 2]))


@pytest.mark.parametrize("d", [256, 512, 1024, 2048, 4096])
# blocks sharing a token; one per token with four fallback waves (E = 16, and
# E = 40 at T = 130), with one (E = 8, T = 257)
@pytest.mark.parametrize("E,T", [(8, 5), (40, 5), (40, 70), (16, 5), (40, 130), (16, 257)])
def test_fused_norm_router_is_the_separate_norm(d, E, T):
    cfg = _cfg(d, E, 2)
    layer = L.synth_layer(cfg, seed=d + E)
    rng = np.random.default_rng(d)
    hidden = rng.standard_normal((T, d)).astype(np.float32)
    hidden[T // 2] = 0
    hidden[1] *= np.float32(1e-20)
    w = (1 + 0.1 * rng.standard_normal(d)).astype(np.float32)
    with L.MoeFfn(cfg.desc(T), layer) as moe:
        moe.set_norm(w, 1e-5)
        out, idx, _ = moe.forward_norm_residual(hidden)
        y, idx2, _ = moe.forward(O.rms_norm(hidden, w, 1e-5))
    assert np.array_equal(idx, idx2)
    assert np.array_equal(out, hidden + y)


@pytest.mark.parametrize("T,K", [(63, 4), (64, 4), (65, 4), (255, 1), (257, 1), (32, 8)])
@pytest.mark.parametrize("E", [8, 72, 200])
def test_one_wave_dispatch_edges(E, T, K):
    cfg = _cfg(256, E, K, L.ROUTE_SOFTMAX_RENORM)
    run_and_check(cfg, L.synth_layer(cfg, seed=T), L.synth_x(cfg, T, seed=T, index=E))
