"""Causal rows whose weights are all alike -- the maximum score is infinite, or
every score is NaN -- against the oracle, bit for bit: the masked keys then weigh
what the visible ones do, in the sum and in the outputs. Rows for the vector
kernel (4 a block) and for the matrix cores (16-row tiles), f32 keys, and f16
caches whose keys are past binary16's range."""

import numpy as np
import pytest

from oracle import oracle as O
from trit_amd import hip, model, synth

pytestmark = pytest.mark.gpu


def same_or_both_nan(a, b):
    a, b = np.asarray(a, np.float32), np.asarray(b, np.float32)
    return np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)].view(np.uint32),
                                                                       b[~np.isnan(b)].view(np.uint32))


@pytest.mark.parametrize("rows", [6, 40])
@pytest.mark.parametrize("hd", [64, 128])
def test_f32_keys(gpu, rows, hd):
    print(f"case uniform rows f32 rows={rows} hd={hd}", flush=True)
    heads = 2
    q, k, v = (synth.normal(synth.seed_for(41, i), (rows, heads * hd)).astype(np.float32) for i in range(3))
    q[3, :hd] = 1e30   # with the large key: scores of +-inf
    k[2, :hd] = 1e30
    q[4, hd:] = np.nan  # every score NaN
    q[5, 1] = np.inf
    got = hip.attention(q, k, v, heads, heads, hd, True, hip.EXACT)
    want = O.attention(q, k, v, heads, heads, hd, causal=True)
    assert same_or_both_nan(got, want)
    assert not np.isnan(want[3]).any()


def scaled_layer(hd, first, last):
    """Two layers; the first one's qkv rows [first, last) 30000 times larger, so the
    caches hold them as +-inf."""
    cfg = dict(d=256, ffn=512, layers=2, heads=4, kv_heads=2, head_dim=hd, vocab=500, eps=1e-6, rope_base=1e6,
               qk_norm=0)
    w = synth.lm_weights(cfg, config=77 + hd, sigma=0.2, norm_jitter=0.2)
    blocks = w.layers[0].qkv.reshape(-1, cfg["d"] // 32, 34).copy()
    part = blocks[first:last]
    scales = part[..., :2].copy().view(np.float16)
    part[..., :2] = (scales.astype(np.float32) * 30000).astype(np.float16).view(np.uint8)
    w.layers[0].qkv[...] = blocks.reshape(w.layers[0].qkv.shape)
    return cfg, O.Lm(cfg, w, kv_f16=True), model.build_decoder(w)


@pytest.mark.parametrize("rows", [6, 40])
@pytest.mark.parametrize("hd", [64, 128])
def test_f16_keys_past_their_range(gpu, rows, hd):
    """One layer's keys of +-inf in the f16 caches; finite logits all the same."""
    print(f"case uniform rows f16 keys rows={rows} hd={hd}", flush=True)
    cfg, ref, lm = scaled_layer(hd, 4 * hd, 6 * hd)
    p = synth.prompt(78, rows, cfg["vocab"])
    s = lm.session(rows + 8)
    want = ref.forward(p)
    assert np.isfinite(want).all()
    assert same_or_both_nan(s.prefill(p), want)
    s.free()
    lm.free()


@pytest.mark.parametrize("rows", [6, 40])
def test_f16_values_past_their_range(gpu, rows):
    print(f"case f16 values rows={rows}", flush=True)
    cfg, ref, lm = scaled_layer(64, 6 * 64, 8 * 64)
    p = synth.prompt(78, rows, cfg["vocab"])
    s = lm.session(rows + 8)
    assert same_or_both_nan(s.prefill(p), ref.forward(p))
    s.free()
    lm.free()
