"""What a prompt as products allocates: room for 32 tokens for a prompt of up
to 32, for a chunk of 512 once one is longer, kept from then on; the results do
not depend on the room there is."""
import os

import numpy as np
import pytest

from phonemap_amd import api

pytestmark = pytest.mark.gpu
TMP = os.environ.get("SS_TEST_TMP", "/tmp")
D, QKV, FFN = 256, 256 + 2 * 128, 512


def _model(kv):
    path = os.path.join(TMP, "ss_test_prompt_buffers.gguf")
    if not os.path.exists(path):
        api.write_synthetic_gguf(path + ".part", api.SynthSpec(
            n_layers=2, hidden=D, n_heads=4, n_kv_heads=2, head_dim=64, ffn=FFN, vocab=512, context_length=1024,
            seed=9, scale_mode=1))
        os.replace(path + ".part", path)
    return api.Model(path, max_context=1024, kv=kv)


def _room(tokens):
    """fp32 rows of the hidden state, [q|k|v], attention and FFN, and x as two
    fp16 parts with its scales (at most 6 bytes a value); 8 KB of rounding."""
    return tokens * (4 * (D + QKV + D + FFN + 1) + 6 * FFN) + 8192


@pytest.mark.parametrize("kv", ["f16", "int8"])
def test_prompt_buffers_follow_the_prompt(kv):
    L = api._lib()
    rng = np.random.default_rng(3)
    prompts = [rng.integers(3, 512, n).tolist() for n in (4, 32, 33, 600, 5)]
    fresh = []
    for p in prompts:
        with _model(kv) as m:
            fresh.append(m.eval_prompt(p, 0)[0])
    with _model(kv) as m:
        used = lambda: L.ss_hip_model_bytes(L.ss_model_hip(m.h))
        base, got, grown = used(), [], []
        for p in prompts:
            print("prompt buffers", kv, len(p), flush=True)
            got.append(m.eval_prompt(p, 0)[0])
            grown.append(used() - base)
    few, chunk = _room(32) + 4 * 1024, _room(512) + 4 * 1024   # (and the positions)
    assert 0 < grown[0] <= few and grown[1] == grown[0]
    assert few < grown[2] <= chunk and grown[3] == grown[4] == grown[2]
    for a, b in zip(got, fresh):
        assert np.array_equal(a, b)
