"""Prompts as products over the int8 cache: a chunk of n tokens at position
pos0 of a one-layer model whose earlier cache rows are given, against the
oracle's int8 model evaluating the same tokens one by one.

Shapes: each head dimension and query group, contexts around one 32-key
block, 64 keys and one step of four key groups, and a chunk with more row
tiles than compute units. The earlier rows' magnitudes span four decades, so
the V scales do too.

Bound: codes are equal unless a value lies within the products' rounding
(about 1e-6) of a rounding boundary; one code more or less moves one of ctx
positions by 1/127 of its scale, under 1/127 of the output. With the
products' own 1e-4 that stays under 1e-3 of the largest logit at contexts
above 40, and under 8e-3 below.
"""
import os

import numpy as np
import pytest

import oracle
from phonemap_amd import api
from tests.util import rel_err

pytestmark = pytest.mark.gpu
TMP = os.environ.get("SS_TEST_TMP", "/tmp")


@pytest.mark.parametrize("H,KVH,hd,cases", [
    (4, 4, 64, [(0, 1), (0, 33), (31, 33), (62, 3)]),
    (8, 1, 64, [(0, 9), (120, 8), (121, 8), (200, 40)]),
    (8, 2, 128, [(0, 8), (56, 8), (57, 8), (127, 2), (250, 30)]),
    (4, 2, 256, [(0, 2), (40, 25), (180, 9)]),
    (32, 32, 128, [(40, 260)]),
])
def test_chunk_over_int8_cache(H, KVH, hd, cases):
    path = os.path.join(TMP, "ss_test_int8_rows_%d_%d_%d.gguf" % (H, KVH, hd))
    if not os.path.exists(path):
        api.write_synthetic_gguf(path + ".part", api.SynthSpec(
            n_layers=1, hidden=H * hd, n_heads=H, n_kv_heads=KVH, head_dim=hd, ffn=512, vocab=512, context_length=320,
            seed=H + hd, scale_mode=1))
        os.replace(path + ".part", path)
    rng = np.random.default_rng(H + hd)
    for pos0, n in cases:
        print("int8 rows", H, KVH, hd, pos0, n, flush=True)
        om = oracle.Model(path, 320, "int8")
        with api.Model(path, max_context=320, kv="int8") as m:
            m.set_prompt_batch(1)
            if pos0:
                size = 10.0 ** rng.uniform(-3, 1, (2, pos0, 1))
                k, v = (size * rng.standard_normal((2, pos0, KVH * hd))).astype(np.float16)
                m.kv_write(0, 0, k.view(np.uint16), v.view(np.uint16))
                om.kv_write_rows(0, 0, k.view(np.uint16), v.view(np.uint16))
            tokens = rng.integers(3, 512, n).tolist()
            lg, am = m.eval_prompt(tokens, pos0)
            want = om.prefill(tokens, pos0)
            assert np.all(np.isfinite(lg))
            assert rel_err(lg, want) <= (1e-3 if pos0 + n > 40 else 8e-3)
            # the appended rows serve the next token
            lg, _ = m.eval_token(am, pos0 + n)
            assert rel_err(lg, om.forward(am, pos0 + n)) <= (1e-3 if pos0 + n > 40 else 8e-3)
        om.close()
