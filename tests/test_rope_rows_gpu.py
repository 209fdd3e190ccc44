"""Prompts on both sides of the q/k norm and rotary dispatch (a block a head, or
32 heads a block from 13000 heads of rows, 7000 below head_dim 64), against the
oracle, bit for bit, with f16 and f32 caches."""

import numpy as np
import pytest

from oracle import oracle as O
from trit_amd import hip, model, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv_heads,hd,rows", [
    (16, 16, 64, 270), (16, 16, 64, 271), (16, 16, 128, 271), (32, 8, 96, 272), (16, 16, 32, 145), (16, 16, 32, 146),
    (32, 32, 8, 73)])
@pytest.mark.parametrize("flags", [0, hip.EXACT])
def test_prompt(gpu, heads, kv_heads, hd, rows, flags):
    print(f"case rope rows={rows} heads={heads}/{kv_heads} hd={hd} flags={flags}", flush=True)
    cfg = dict(d=64, ffn=64, layers=2, heads=heads, kv_heads=kv_heads, head_dim=hd, vocab=300, eps=1e-6, rope_base=1e6,
               qk_norm=1)
    w = synth.lm_weights(cfg, config=60 + hd, sigma=0.2, norm_jitter=0.2)
    lm = model.build_decoder(w)
    p = synth.prompt(61, rows, cfg["vocab"])
    s = lm.session(rows, flags)
    got, want = s.prefill(p), O.Lm(cfg, w, O.isa_best(), kv_f16=not flags).forward(p)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    s.free()
    lm.free()
