"""attention_steps on both sides of its dispatch, against the oracle, bit for bit:
few keys by head size and by the number of blocks, the most keys the staged
kernel's shared memory holds (7928) and one more, head sizes that divide neither
a block nor a wave, and sequences of very different lengths in one call."""

import numpy as np
import pytest

from oracle import oracle as O
from tests.test_beam_gpu import bits_equal, caches
from trit_amd import hip, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,hd,tks", [
    (2, 2, 64, [7928]), (2, 1, 64, [7929]), (1, 1, 128, [7928, 3]), (1, 1, 128, [7929, 1]), (2, 2, 24, [7928]),
    (18, 18, 64, [64] * 32), (18, 6, 64, [64, 65] * 16), (16, 4, 64, [5] * 32), (20, 20, 32, [64] * 32),
    (20, 4, 32, [65] * 32), (4, 2, 8, [40, 1]), (4, 2, 8, [41, 8]), (3, 3, 24, [41, 40, 700]), (3, 1, 48, [40]),
    (2, 2, 40, [200, 64]), (3, 3, 96, [48, 49]), (3, 3, 96, [48, 47]), (2, 2, 120, [49, 2000]), (5, 5, 168, [300]),
    (2, 1, 200, [96, 97]), (2, 1, 200, [45]), (1, 1, 232, [9001]), (2, 2, 248, [500]), (4, 4, 256, [96] * 24),
    (4, 4, 256, [94] * 24), (17, 17, 256, [49] * 16)])
def test_against_the_oracle(gpu, heads, kv_heads, hd, tks):
    print(f"case attention_steps heads={heads}/{kv_heads} hd={hd} tk={tks[:4]} x{len(tks)}", flush=True)
    q = synth.activations(750 + hd, len(tks), heads * hd)
    cs = caches(760 + hd, tks, kv_heads * hd)
    assert bits_equal(hip.attention_steps(q, cs, heads, kv_heads), O.attention_steps(q, cs, heads, kv_heads))
