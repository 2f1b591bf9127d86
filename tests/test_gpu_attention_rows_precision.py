"""Attention of prompt rows against attention of the same tokens one by one
(ss_hip_attention_rows, ss_hip_attention_rows_int8 and ss_hip_attention on the
same queries and cache), both held to 64 bits.

The one-token kernels hold queries, scores and weights in fp32. The rows
kernel holds queries and weights as two fp16 parts each. Error of a launch:
root mean square over its rows and heads of |got - exact| / |exact|.

Bounds, on the geometric mean over the shapes of the rows' error over the
one-token error: 1.05 where a prompt would otherwise run token by token (the
int8 cache, and fp16 prompts of 4 to 7 tokens: no larger, and 5% for the
draw), and 1.6 for longer fp16 prompts, whose O is one chain of additions over
all blocks of keys (up to 1.8 at a context of 4000).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(32, 4, 64, 0, 4), (32, 4, 64, 60, 4), (32, 4, 64, 200, 7), (32, 8, 128, 0, 7), (32, 32, 128, 500, 6),
          (32, 8, 128, 2000, 5), (32, 8, 128, 4000, 7), (8, 4, 256, 100, 7), (16, 2, 256, 20, 5)]
LONGER = [(32, 4, 64, 0, 64), (32, 32, 128, 0, 32), (32, 8, 128, 1000, 32), (32, 8, 128, 4000, 8), (16, 8, 256, 0, 32)]


def _exact(q, k, v, pos0):
    n, H, hd = q.shape
    G, ctx = H // k.shape[0], pos0 + n
    out = np.zeros((n, H, hd))
    late = np.arange(ctx)[None, :] > pos0 + np.arange(n)[:, None]
    for h in range(H):
        s = q[:, h].astype(np.float64) @ k[h // G].T / np.sqrt(hd)
        s[late] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        out[:, h] = p @ v[h // G] / p.sum(1, keepdims=True)
    return out


def _ratio(hip, kv, size, H, KVH, hd, pos0, n):
    rng = np.random.default_rng(H + hd + pos0 + n)
    ctx = pos0 + n
    q = (size * rng.standard_normal((n, H, hd))).astype(np.float32)
    if kv:
        k, v = (np.clip(np.rint(32 * rng.standard_normal((KVH, ctx, hd))), -127, 127).astype(np.int8) for _ in "kv")
        ks, vs = ((0.03 * rng.uniform(0.5, 2, ctx)).astype(np.float32) for _ in "kv")
        kd, vd = (c.astype(np.float64) * s.astype(np.float64)[None, :, None] for c, s in ((k, ks), (v, vs)))
    else:
        k, v = (rng.standard_normal((KVH, ctx, hd)).astype(np.float16) for _ in "kv")
        ks = vs = np.ones(ctx, np.float32)
        kd, vd = k.astype(np.float64), v.astype(np.float64)
    want = _exact(q, kd, vd, pos0)
    Q, K, V, KS, VS = (hip.upload(x) for x in (q, k, v, ks, vs))
    O = hip.buf(4 * q.size)

    def err():
        got = O.read(np.float32, q.size).reshape(q.shape)
        return np.sqrt(np.mean((np.linalg.norm(got - want, axis=2) / np.linalg.norm(want, axis=2)) ** 2))

    if kv:
        rc = hip.L.ss_hip_attention_rows_int8(hip.ctx, O.ptr, Q.ptr, K.ptr, V.ptr, KS.ptr, VS.ptr, H, KVH, hd, ctx, pos0,
                                              n, None)
    else:
        rc = hip.L.ss_hip_attention_rows(hip.ctx, O.ptr, Q.ptr, K.ptr, V.ptr, H, KVH, hd, ctx, pos0, n, None)
    assert rc == 0, hip.err()
    rows = err()
    for z in range(n):
        rc = hip.L.ss_hip_attention(hip.ctx, O.ptr + 4 * z * H * hd, Q.ptr + 4 * z * H * hd, K.ptr, V.ptr,
                                    KS.ptr if kv else None, VS.ptr if kv else None, H, KVH, hd, ctx, pos0 + z + 1, kv, None)
        assert rc == 0, hip.err()
    hip.sync()
    single = err()
    for b in (Q, K, V, KS, VS, O):
        b.free()
    print("kv %d, queries x %g, %s: rows %.2e, one by one %.2e" % (kv, size, (H, KVH, hd, pos0, n), rows, single), flush=True)
    return rows / single


@pytest.mark.parametrize("kv,shapes,bound", [(0, SHAPES, 1.05), (1, SHAPES + LONGER, 1.05), (0, LONGER, 1.6)],
                         ids=["fp16-4-to-7", "int8", "fp16-longer"])
def test_rows_keep_the_precision_of_single_tokens(hip, kv, shapes, bound):
    r = [_ratio(hip, kv, size, *s) for s in shapes for size in (1.0, 4.0)]
    mean = np.exp(np.mean(np.log(r)))
    print("geometric mean %.3f, largest %.2f" % (mean, max(r)), flush=True)
    assert mean <= bound
