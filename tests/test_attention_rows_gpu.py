"""Trit's attention of many query rows on the f32 matrix cores against the
oracle, bit for bit: head_dim 64 and 128, the edges of the 16-row and 16-key
tiles, of the waves' chunks and of each register budget (128, 512, 1024, 1600
and 3200 keys), causal with keys before the rows, grouped heads, and more keys
than the kernel takes."""

import numpy as np
import pytest

from oracle import oracle as O
from trit_amd import hip, synth

pytestmark = pytest.mark.gpu


def bits_equal(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))


def inputs(seed, tq, tk, heads, kv_heads, hd):
    return [synth.normal(synth.seed_for(seed, i), (t, h * hd)).astype(np.float32)
            for i, (t, h) in enumerate([(tq, heads), (tk, kv_heads), (tk, kv_heads)], 1)]


@pytest.mark.parametrize("tq,tk,heads,kv_heads,hd,causal", [
    (9, 9, 2, 2, 64, False), (16, 17, 2, 1, 64, False), (17, 127, 3, 3, 128, False), (33, 129, 2, 2, 64, False),
    (15, 511, 2, 2, 128, False), (18, 513, 1, 1, 64, False), (16, 1025, 1, 1, 128, False),
    (20, 1600, 1, 1, 64, False), (20, 1601, 1, 1, 64, False), (12, 3200, 1, 1, 128, False),
    (12, 3201, 1, 1, 64, False), (64, 30, 2, 2, 64, False),
    (9, 9, 2, 2, 64, True), (50, 50, 4, 2, 128, True), (37, 300, 2, 1, 64, True), (40, 1605, 2, 2, 128, True),
])
def test_against_the_oracle(gpu, tq, tk, heads, kv_heads, hd, causal):
    print(f"case attention rows tq={tq} tk={tk} heads={heads}/{kv_heads} hd={hd} causal={causal}", flush=True)
    q, k, v = inputs(90 + tq + tk, tq, tk, heads, kv_heads, hd)
    got = hip.attention(q, k, v, heads, kv_heads, hd, causal, hip.EXACT)
    if causal:
        # The oracle's causal form masks from position tk - tq on.
        want = np.concatenate([O.attention(q[i:i + 1], k[:tk - tq + i + 1], v[:tk - tq + i + 1], heads, kv_heads, hd,
                                           causal=False) for i in range(tq)])
    else:
        want = O.attention(q, k, v, heads, kv_heads, hd, causal=False)
    assert bits_equal(got, want), float(np.max(np.abs(got - want)))


@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_non_finite(gpu, value):
    """A non-finite value reaches what it does in the oracle (masked keys' weights are not quite zero there)."""
    print(f"case attention rows {value}", flush=True)
    tq, heads, hd = 40, 2, 64
    q, k, v = inputs(95, tq, tq, heads, heads, hd)
    v[33, 5] = value
    got = hip.attention(q, k, v, heads, heads, hd, True, hip.EXACT)
    want = O.attention(q, k, v, heads, heads, hd, causal=True)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    keep = ~np.isnan(want)
    assert np.array_equal(got[keep].view(np.uint32), want[keep].view(np.uint32))
