"""Causal attention of prompt rows over the int8 cache
(ss_hip_attention_rows_int8) against 64 bits over the same codes and scales.

Error of a row: 2-norm of its difference over 2-norm of its exact output, per
query head. Bound: a weight's exponent, up to 2^5 here, is one fp32 rounding
(2^-20 of the weight, the same way for few keys only), q, the weights and the
sums add some 2^-22 each: 2e-6. One key of a row taken with 11 bits instead of
22 gives 1e-5 to 2e-4.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 2e-6


def _case(H, KVH, hd, pos0, n, seed):
    rng = np.random.default_rng(seed)
    max_seq = pos0 + n + 5
    q = rng.standard_normal((n, H, hd)).astype(np.float32)
    k, v = (rng.integers(-127, 128, (KVH, max_seq, hd)).astype(np.int8) for _ in "kv")
    ks, vs = (rng.uniform(0.01, 0.03, max_seq).astype(np.float32) for _ in "kv")
    ks[pos0 + n:] = np.nan   # what lies past the last row is not read
    vs[pos0 + n:] = np.nan
    return q, k, v, ks, vs


def _rows(hip, q, k, v, ks, vs, pos0):
    n, H, hd = q.shape
    bufs = [hip.upload(x) for x in (q, k, v, ks, vs)]
    out = hip.buf(4 * (q.size + 64))
    out.write(np.full(q.size + 64, 7.0, np.float32))
    rc = hip.L.ss_hip_attention_rows_int8(hip.ctx, out.ptr, *(b.ptr for b in bufs), H, k.shape[0], hd, k.shape[1], pos0,
                                          n, None)
    assert rc == 0, hip.err()
    got = out.read(np.float32, q.size + 64)
    for b in bufs + [out]:
        b.free()
    assert np.all(got[q.size:] == 7.0)   # nothing past the last row
    return got[:q.size].reshape(n, H, hd)


def _exact(q, k, v, ks, vs, pos0):
    n, H, hd = q.shape
    G, ctx = H // k.shape[0], pos0 + n
    kd = k[:, :ctx].astype(np.float64) * ks[:ctx].astype(np.float64)[None, :, None]
    vd = v[:, :ctx].astype(np.float64) * vs[:ctx].astype(np.float64)[None, :, None]
    out = np.zeros((n, H, hd))
    late = np.arange(ctx)[None, :] > pos0 + np.arange(n)[:, None]
    for h in range(H):
        s = q[:, h].astype(np.float64) @ kd[h // G].T / np.sqrt(hd)
        s[late] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = p @ vd[h // G] / p.sum(1, keepdims=True)
    return out


def _row_err(got, want):
    return np.linalg.norm(got - want, axis=2) / np.linalg.norm(want, axis=2)


SHAPES = [
    (4, 4, 64, 0, 33), (32, 4, 64, 31, 34), (32, 8, 64, 200, 40),              # two and four key groups
    (8, 2, 128, 57, 8), (32, 8, 128, 300, 40), (32, 32, 128, 0, 64),
    (128, 32, 128, 3, 79),                                                      # more row tiles than compute units
    (2, 1, 256, 30, 33), (8, 1, 256, 126, 9), (8, 2, 256, 300, 40),
]


@pytest.mark.parametrize("H,KVH,hd,pos0,n", SHAPES)
def test_rows_against_64_bits(hip, H, KVH, hd, pos0, n):
    print("int8 attention rows", H, KVH, hd, pos0, n, flush=True)
    c = _case(H, KVH, hd, pos0, n, H + hd + pos0 + n)
    err = _row_err(_rows(hip, *c, pos0), _exact(*c, pos0))
    print("worst row %.2e, all rows %.2e" % (err.max(), np.sqrt(np.mean(err ** 2))), flush=True)
    assert err.max() <= TOL


@pytest.mark.parametrize("H,KVH,hd,pos0,n", SHAPES)
@pytest.mark.parametrize("last", [1e6, np.inf])
def test_rows_do_not_depend_on_later_scales(hip, H, KVH, hd, pos0, n, last):
    """V scales spread over 8 decades, each position's above the next one's by
    chance only, and the last position's far above all (or infinite): the rows
    before it do not see it."""
    print("int8 attention rows, wide scales", H, KVH, hd, pos0, n, last, flush=True)
    q, k, v, ks, vs = _case(H, KVH, hd, pos0, n, 1000 + H + hd + pos0 + n)
    vs *= 10.0 ** np.random.default_rng(n).uniform(-8, 0, vs.size).astype(np.float32)
    vs[pos0 + n - 1] = last
    got = _rows(hip, q, k, v, ks, vs, pos0)
    if np.isinf(last):
        # weight * inf * code in every element (0 codes: NaN)
        assert not np.isfinite(got[-1]).any()
        got, q, vs = got[:-1], q[:-1], vs.copy()
    else:
        assert np.isfinite(got).all()
    err = _row_err(got, _exact(q, k, v, ks, vs, pos0))
    print("worst row %.2e" % err.max(), flush=True)
    assert err.max() <= TOL
