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
from tests.ref_model import RefModel
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


class _EdgeModel(RefModel):
    """The 64-bit model, which also keeps how near a K or V value came to the
    edge between two codes, in codes."""
    nearest = 1.0

    def kv_encode(self, x):
        t = np.abs(x) / (np.max(np.abs(x)) / 127.0)
        self.nearest = min(self.nearest, float(np.min(np.abs(t - np.floor(t) - 0.5))))
        return super().kv_encode(x)


@pytest.mark.parametrize("H,KVH,hd,n", [(4, 1, 64, 24), (8, 1, 64, 7), (8, 2, 128, 5), (4, 1, 256, 4)])
def test_prompt_whose_codes_are_certain(H, KVH, hd, n):
    """Where no value of the prompt lies within 1e-4 of an edge between two
    codes, the cache is the 64-bit model's own, and the logits are within the
    rounding of the products and the attention, 2e-6 (2-norm): as products and
    token by token alike. A value nearer to an edge may fall either way in any
    order of the sums, and moves the logits by 1e-4 to 1e-3: that is all that
    the two differ by."""
    path = os.path.join(TMP, "ss_test_int8_edge_%d_%d_%d.gguf" % (H, KVH, hd))
    if not os.path.exists(path):
        api.write_synthetic_gguf(path + ".part", api.SynthSpec(
            n_layers=1, hidden=H * hd, n_heads=H, n_kv_heads=KVH, head_dim=hd, ffn=512, vocab=512, context_length=64,
            seed=H + hd + n, scale_mode=1))
        os.replace(path + ".part", path)
    ref, found = _EdgeModel(path, 64, "int8"), 0
    with api.Model(path, max_context=64, kv="int8") as m:
        for seed in range(60):
            tokens = np.random.default_rng(seed).integers(3, 512, n).tolist()
            ref.reset()
            ref.nearest = 1.0
            want = ref.prefill(tokens, 0)
            if ref.nearest < 1e-4:
                continue
            found += 1
            for batch in (1, -1):
                m.reset()
                m.set_prompt_batch(batch)
                lg, _ = m.eval_prompt(tokens, 0)
                err = np.linalg.norm(lg - want) / np.linalg.norm(want)
                print("int8 prompt", H, KVH, hd, n, seed, batch, "%.2e" % err, flush=True)
                assert err <= 2e-6, (seed, batch, err)
            if found == 4:
                break
    assert found >= 2
