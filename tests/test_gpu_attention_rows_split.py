"""Causal attention of prompt rows where a workgroup's key groups and row
tiles end: contexts around one 32-key block, one step of two or four groups
and the two-group form's 64 keys; row counts around 32- and 64-row tiles; the
forms with one and with two row tiles, at each head dimension.

Against 64-bit attention over the same fp16 cache. Bound: q and P carry 22
bits through two fp16 parts, scores sum head_dim products in fp32 and the
output ctx of them: with |q . k| / sqrt(hd) below 8, an exponent's error is
below 8 * (2^-22 + 16 * 2^-24) and a sum's below sqrt(ctx) * 2^-24, together
under 2e-5 of the largest output.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 2e-5


def _ref(q, kc, vc, G, pos0):
    n, H, hd = q.shape
    out = np.zeros((n, H, hd))
    for t in range(n):
        ctx = pos0 + t + 1
        for h in range(H):
            s = kc[h // G, :ctx].astype(np.float64) @ q[t, h].astype(np.float64) / np.sqrt(hd)
            p = np.exp(s - s.max())
            out[t, h] = p @ vc[h // G, :ctx].astype(np.float64) / p.sum()
    return out


@pytest.mark.parametrize("H,KVH,hd,pos0,n", [
    (4, 4, 64, 0, 31), (4, 4, 64, 0, 32), (4, 4, 64, 0, 33),            # one tile, one block
    (8, 2, 64, 40, 24), (8, 2, 64, 40, 25),                             # 64 and 65 keys
    (8, 2, 128, 56, 8), (8, 2, 128, 57, 8),                             # the same at head_dim 128
    (8, 2, 128, 120, 8), (8, 2, 128, 121, 8), (8, 2, 128, 127, 2),      # one step of four groups, and one key more
    (4, 1, 128, 129, 7), (8, 1, 64, 255, 5),                            # a ragged tile over several steps
    (128, 32, 128, 3, 64), (128, 32, 128, 3, 65), (128, 32, 128, 0, 79),  # 256 tiles, and more: two tiles share
    (2, 1, 256, 30, 33), (2, 1, 256, 32, 33), (8, 1, 256, 126, 9),      # head_dim 256
])
def test_rows_at_tile_and_block_edges(hip, H, KVH, hd, pos0, n):
    print("attention rows", H, KVH, hd, pos0, n, flush=True)
    rng = np.random.default_rng(H + hd + pos0 + n)
    max_seq = pos0 + n + 5
    q = rng.standard_normal((n, H, hd)).astype(np.float32)
    kc = rng.standard_normal((KVH, max_seq, hd)).astype(np.float16)
    vc = rng.standard_normal((KVH, max_seq, hd)).astype(np.float16)
    kc[:, pos0 + n:] = np.nan
    vc[:, pos0 + n:] = np.nan
    Q, KC, VC, O = hip.upload(q), hip.upload(kc), hip.upload(vc), hip.buf(4 * (q.size + 64))
    O.write(np.full(q.size + 64, 7.0, np.float32))
    rc = hip.L.ss_hip_attention_rows(hip.ctx, O.ptr, Q.ptr, KC.ptr, VC.ptr, H, KVH, hd, max_seq, pos0, n, None)
    assert rc == 0, hip.err()
    got = O.read(np.float32, q.size + 64)
    for b in (Q, KC, VC, O):
        b.free()
    assert np.all(got[q.size:] == 7.0)   # nothing past the last row
    want = _ref(q, kc, vc, H // KVH, pos0)
    assert np.abs(got[:q.size].reshape(want.shape) - want).max() <= TOL * np.abs(want).max()
