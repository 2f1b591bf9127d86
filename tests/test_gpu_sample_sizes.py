"""Device sampling at the sizes where its launches change: rows of one
workgroup (up to 1024 entries) and of many, at the edges of their 1024-entry
tiles; the top-k candidates just within and past their space (ties); no top-k
with a cutoff that keeps one value, most of the row, or everything; infinite
logits. Bars as in test_gpu_sample.py.
"""
import numpy as np
import pytest

import oracle
from tests.test_gpu_sample import _check_index, _device_sample

pytestmark = pytest.mark.gpu
PARAMS = [(0.8, 0.95, 40), (1.0, 0.9, 0), (1.2, 1.0, 0), (0.9, 1.0, 1024), (0.9, 0.7, 1025), (1.0, 1e-6, 0), (1.0, 0.9999, 0)]


@pytest.mark.parametrize("V", [1024, 1025, 4096, 5119, 5120, 5121, 70001])
@pytest.mark.parametrize("kind", ["normal", "flat", "steps", "inf"])
def test_sample_sizes(hip, V, kind):
    print("sample", V, kind, flush=True)
    rng = np.random.default_rng(V)
    for T, top_p, top_k in PARAMS:
        x = (2.5 * rng.standard_normal(V)).astype(np.float32)
        if kind == "flat":
            x[:] = 0.25
        elif kind == "steps":   # 2048 ties at the top: the candidates' space, and one more
            x[rng.permutation(V)[: 2048 + (top_k == 40)]] = 11.0
        elif kind == "inf":
            x[rng.integers(0, V, V // 2)] = -np.inf
        for _ in range(2):
            seed = int(rng.integers(1, 2 ** 63))
            want, want_st, p, r = oracle.sample(x, T, top_p, top_k, seed)
            got, got_st = _device_sample(hip, x, T, top_p, top_k, seed)
            assert got_st == want_st and 0 <= got < V
            _check_index(got, want, p, r)


@pytest.mark.parametrize("V", [1025, 3000, 70001])
@pytest.mark.parametrize("top_k", [1, 150, 288, 289, 513, 1000, 1024])
@pytest.mark.parametrize("kind", ["normal", "ties", "inf"])
def test_sample_few_and_many_candidates(hip, V, top_k, kind):
    """Candidates compared in pairs (up to 288 of them) and sorted, with what
    is kept after top-p on either side too, and ties across the k-th."""
    print("sample candidates", V, top_k, kind, flush=True)
    rng = np.random.default_rng(V + top_k)
    for T, top_p in [(0.7, 1.0), (1.5, 0.99), (0.8, 0.5)]:
        x = (2.5 * rng.standard_normal(V)).astype(np.float32)
        if kind == "ties":
            x = np.round(x * 4) / 4
        elif kind == "inf":
            x[rng.permutation(V)[: V - 400]] = -np.inf   # fewer terms than many a top_k
        for _ in range(3):
            seed = int(rng.integers(1, 2 ** 63))
            want, want_st, p, r = oracle.sample(x, T, top_p, top_k, seed)
            got, got_st = _device_sample(hip, x, T, top_p, top_k, seed)
            assert got_st == want_st and 0 <= got < V
            _check_index(got, want, p, r)
