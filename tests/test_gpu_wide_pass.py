"""Matrix-core passes of 64 tokens (experts averaging more than 32 tokens, one
f16 per activation): accumulators in units of each super-block's scale, two
token tiles per decoded weight."""
import numpy as np
import pytest

import leafcutterllm_amd as L
from parity_util import run_and_check

pytestmark = pytest.mark.gpu


def _plant_scales(data, rng):
    """Q4_K blocks with d = 0 (dmin kept), runs of them, d < 0, and d far
    smaller than its neighbours': what the rescaling divides by."""
    b = data.reshape(-1, 144)
    d = b[:, :2].copy().view(np.float16).reshape(-1)
    kind = rng.integers(0, 8, d.size)
    d[kind == 0] = 0
    d[kind == 1] = -d[kind == 1]
    d[kind == 2] *= np.float16(2.0 ** -9)
    b[:, :2] = d.view(np.uint8).reshape(-1, 2)
    b[:3, :2] = 0  # the first row starts with zero scales
    return b.reshape(-1)


# tokens per expert around the tile and pass edges; d of an odd and an even
# number of super-blocks; F whole super-blocks or (384, 640) the split layout
@pytest.mark.parametrize("F", [256, 384, 512, 640])
@pytest.mark.parametrize("T", [33, 48, 64, 65, 96, 97, 129])
def test_wide_pass_edges(T, F):
    d = 768 if T % 2 else 512
    cfg = L.configs.small_config("wide", d, F, 1, 1, L.ROUTE_SOFTMAX_RENORM, L.TYPE_Q4_K,
                                 L.TYPE_Q4_K)
    layer = L.synth_layer(cfg, seed=T)
    rng = np.random.default_rng(F + T)
    for k in ("gate", "up", "down"):
        layer[k] = _plant_scales(layer[k], rng)
    run_and_check(cfg, layer, L.synth_x(cfg, T, seed=T, index=F))


@pytest.mark.parametrize("T", [120, 200])
@pytest.mark.parametrize("F,FS", [(512, 512), (384, 384), (512, 768)])
def test_wide_pass_skew_and_shared(T, F, FS):
    """Skewed routing (passes of 64 tokens beside nearly empty ones) with
    shared experts, fused (FS == F) and in launches of their own."""
    cfg = L.configs.small_config("wides", 512, F, 10, 4, L.ROUTE_SOFTMAX, L.TYPE_Q4_K,
                                 L.TYPE_Q4_K, n_shared=2, d_ff_shared=FS, bias="plus2_first8")
    layer = L.synth_layer(cfg, seed=5)
    run_and_check(cfg, layer, L.synth_x(cfg, T, seed=5, index=T))
