"""Prompt rows over an fp16 cache in which the last position's V (or K) is not
finite (a value past 65504 is stored as inf): the rows before it do not see it
and keep their values, as they do when tokens are attended one by one; the row
that sees it is not finite.

Bound of the rows before: 2e-6 of a row, as without it (the sums of the kernel
and of its fp32 form add up to some 2^-22 per row).
"""
import numpy as np
import pytest

from tests.test_gpu_attention_rows_precision import _exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,KVH,hd,pos0,n", [
    (4, 4, 64, 0, 4), (32, 4, 64, 31, 34), (32, 8, 64, 200, 40), (8, 1, 64, 700, 5), (8, 2, 128, 57, 8),
    (32, 8, 128, 300, 40), (128, 32, 128, 3, 79), (2, 1, 256, 30, 33), (8, 1, 256, 126, 5), (8, 2, 256, 300, 40),
])
@pytest.mark.parametrize("what", ["v inf", "v nan", "k inf"])
def test_rows_before_a_position_do_not_see_it(hip, H, KVH, hd, pos0, n, what):
    print("rows, last position", what, H, KVH, hd, pos0, n, flush=True)
    rng = np.random.default_rng(H + hd + pos0 + n)
    ctx = pos0 + n
    q = rng.standard_normal((n, H, hd)).astype(np.float32)
    k, v = (rng.standard_normal((KVH, ctx, hd)).astype(np.float16) for _ in "kv")
    dim = int(rng.integers(hd))
    want = _exact(q[:-1], k[:, :-1].astype(np.float64), v[:, :-1].astype(np.float64), pos0)
    (k if what[0] == "k" else v)[:, -1, dim] = np.inf if what[2:] == "inf" else np.nan
    Q, K, V, O = hip.upload(q), hip.upload(k), hip.upload(v), hip.buf(4 * (q.size + 64))
    O.write(np.full(q.size + 64, 7.0, np.float32))
    assert hip.L.ss_hip_attention_rows(hip.ctx, O.ptr, Q.ptr, K.ptr, V.ptr, H, KVH, hd, ctx, pos0, n, None) == 0, hip.err()
    got = O.read(np.float32, q.size + 64)
    for b in (Q, K, V, O):
        b.free()
    assert np.all(got[q.size:] == 7.0)
    got = got[:q.size].reshape(n, H, hd)
    err = np.linalg.norm(got[:-1] - want, axis=2) / np.linalg.norm(want, axis=2)
    assert np.max(err) <= 2e-6
    last = np.isfinite(got[-1])
    if what[0] == "v":   # that dimension alone
        assert not last[:, dim].any() and np.delete(last, dim, 1).all()
    else:                # score +-inf: a NaN row, or a weight of 0
        s = q[-1, :, dim] > 0
        assert not last[s].any() and last[~s].all()
