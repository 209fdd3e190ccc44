"""Q8_0 products large enough for 128 x 128 blocks whose k is not a multiple of
128, against the oracle, bit for bit: one to thirty-nine groups (odd counts, so
a row's scales start at either half of a dword), rows and columns past the last
whole block, bias and relu."""

import numpy as np
import pytest

from oracle import oracle as O
from trit_amd import hip, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,m", [(20480, 32, 9), (1312, 64, 1900), (96, 160, 20450), (1312, 416, 1921),
                                   (480, 1248, 5100)])
def test_wide(gpu, n, k, m):
    print(f"case q8_0 wide blocks n={n} k={k} m={m}", flush=True)
    codes, sbits = synth.q8_0_matrix(synth.seed_for(2, n + k), n, k)
    bias = synth.activations(91, 1, n)[0]
    x = synth.activations(92 + m, m, k)
    layer = hip.Dense.q8_0(n, k, synth.q8_0_blocks(codes, sbits), bias)
    got = layer.forward(x, relu=True)
    want = np.maximum(O.Int8(codes, sbits.view(np.float16).astype(np.float32), 32, True)(x) + bias, 0)
    assert np.array_equal(got.view(np.uint32), want.astype(np.float32).view(np.uint32))
    layer.free()


# As above, where the 128 x 128 blocks start: more than 256 of them, or 160 with
# long rows; and the last sizes before it.
@pytest.mark.parametrize("n,k,m", [(33024, 32, 9), (32768, 32, 9), (2656, 64, 1601), (96, 160, 32900), (2656, 416, 1665),
                                   (480, 2080, 5100), (480, 2016, 5100), (20480, 3104, 64), (20480, 3040, 17)])
def test_both_sides_of_the_rule(gpu, n, k, m):
    test_wide(gpu, n, k, m)
