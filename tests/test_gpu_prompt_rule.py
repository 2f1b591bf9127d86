"""Which prompts run as matrix products by default (ss_hip_eval_prompt)."""
import ctypes as C
import os

import pytest

from phonemap_amd import api

pytestmark = pytest.mark.gpu
TMP = os.environ.get("SS_TEST_TMP", "/tmp")


@pytest.mark.parametrize("kv", ["f16", "int8"])
@pytest.mark.parametrize("n,start,products", [
    (3, 0, False), (4, 0, True), (4, 4096, True), (4, 4097, False), (7, 10240, True), (7, 10241, False),
    (8, 12288, True), (8, 12289, None), (9, 14337, None),
])
def test_where_prompts_become_products(kv, n, start, products):
    """The default rule at its edges: 4 tokens, and 2048 positions of prefix
    per token above two; 8 tokens on an fp16 cache over any prefix (None:
    products with that cache only)."""
    _check(64, kv, n, start, products)


@pytest.mark.parametrize("kv", ["f16", "int8"])
@pytest.mark.parametrize("n,start,products", [
    (4, 0, True), (4, 2048, True), (4, 2049, False), (7, 5120, True), (7, 5121, False), (8, 6145, None), (14, 12288, True),
])
def test_where_prompts_become_products_head_dim_256(kv, n, start, products):
    """At head_dim 256 the prefix may grow by 1024 positions per token above two."""
    _check(256, kv, n, start, products)


def _check(hd, kv, n, start, products):
    path = os.path.join(TMP, "ss_test_rule_%d.gguf" % hd)
    if not os.path.exists(path):
        api.write_synthetic_gguf(path + ".part", api.SynthSpec(
            n_layers=1, hidden=hd, n_heads=1, n_kv_heads=1, head_dim=hd, ffn=64, vocab=64, context_length=16384,
            seed=5, scale_mode=1))
        os.replace(path + ".part", path)
    print("rule", hd, kv, n, start, flush=True)
    L = api._lib()

    def count():
        out = (C.c_int64 * 6)()
        assert L.ss_hip_gemm_launch_counts(out, 6) == 0
        return list(out)

    with api.Model(path, max_context=16384, kv=kv) as m:
        before = count()
        m.eval_prompt(list(range(3, 3 + n)), start, want_logits=False)
        used = count() != before
    assert used == (kv == "f16" if products is None else products)
