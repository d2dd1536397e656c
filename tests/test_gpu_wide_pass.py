"""Matrix-core passes of 64 tokens (experts averaging more than 32 tokens, one
f16 per activation): accumulators in units of each super-block's scale, two
token tiles per decoded weight."""
import numpy as np
import pytest

import leafcutterllm_amd as L
from kquant_pack import pack_q4_k
from leafcutterllm_amd.moe import dequantize
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


def _exact_h_layer(F, down, rng):
    """A layer and T = 256 tokens whose H is known exactly and exact in f16:
    unit vectors against gates of 32 (silu(32) = 32 in f32) and integer ups.
    Returns (cfg, layer, x, H [T, F] in float64)."""
    d = 256
    cfg = L.configs.small_config("exact", d, F, 1, 1, L.ROUTE_SOFTMAX_RENORM, L.TYPE_Q4_K,
                                 L.TYPE_Q4_K)
    layer = L.synth_layer(cfg, seed=F)

    def blocks(n, dd, dmin, sc, m, qs):
        b = np.empty((n, 144), np.uint8)
        b[:, :16] = np.frombuffer(pack_q4_k(dd, dmin, [sc] * 8, [m] * 8, np.zeros(256, int))[:16],
                                  np.uint8)
        b[:, 16:] = qs
        return b

    layer["gate"] = blocks(F, 1, 0, 32, 0, 0x11).reshape(-1)
    layer["up"] = blocks(F, 1, 1, 1, 8, rng.integers(0, 256, (F, 128))).reshape(-1)
    layer["down"] = down(layer, blocks).reshape(-1)
    up = dequantize(L.TYPE_Q4_K, layer["up"], F * d).astype(np.float64).reshape(F, d)
    return cfg, layer, np.eye(d, dtype=np.float32), 32.0 * up.T


def test_equal_scales_add_no_rounding():
    """Down weights of one scale d (between super-blocks of d = 0) and no mins:
    the accumulators hold integers below 2^24 in units of d, so the result is
    d times an integer, rounded once, in every bit."""
    F, dd = 1280, np.float16(0.0061)
    u = np.float32(dd) * np.float32(16384)
    assert np.float32(u * np.float32(np.float32(1) / u)) != 1  # the quotient d' / d would show
    rng = np.random.default_rng(1)

    def down(layer, blocks):
        b = blocks(F, dd, 0, 1, 0, rng.integers(0, 256, (F, 128)))
        b[rng.random(len(b)) < 0.25, :2] = 0
        return b

    cfg, layer, x, H = _exact_h_layer(F, down, rng)
    W = dequantize(L.TYPE_Q4_K, layer["down"], 256 * F).astype(np.float64).reshape(256, F)
    n = np.rint(H @ np.rint(W / float(dd)).T)
    with L.MoeFfn(cfg.desc(256), layer) as moe:
        y = moe.forward(x)[0]
    assert np.array_equal(y, (n * float(dd)).astype(np.float32))


@pytest.mark.parametrize("F", [512, 640, 2048])
@pytest.mark.parametrize("planted", [False, True])
def test_wide_pass_accumulates_in_f32(F, planted):
    """The down product alone against float64: 1.1e-6, four times the largest
    error measured (2.7e-7), where f16 activations leave 3.6e-4."""
    rng = np.random.default_rng(F)

    def down(layer, blocks):
        return _plant_scales(layer["down"].copy(), rng) if planted else layer["down"]

    cfg, layer, x, H = _exact_h_layer(F, down, rng)
    W = dequantize(L.TYPE_Q4_K, layer["down"], 256 * F)  # float32: right to 6e-8 per weight
    ref = H @ W.astype(np.float64).reshape(256, F).T
    with L.MoeFfn(cfg.desc(256), layer) as moe:
        y = moe.forward(x)[0]
    assert np.linalg.norm(y - ref) < 1.1e-6 * np.linalg.norm(ref)
