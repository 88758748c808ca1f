"""GPU parity of the decode attention where its grid and its merge can go wrong:
grouped heads whose (kv head, split) pairs do and do not divide over the 8 dies,
positions on both sides of a split's edge, and every number of splits the merge
walks in batches, against float64 over the same fp16 rows.

Bar, per output: the weight p_j of position j is off by its score's error e_j, (hd + 8)
roundings of sum |q||k| / sqrt(hd) (RoPE included) and 4 of the score itself, in the sum
over values and in the sum they are divided by; both are `depth` additions deep, the
positions of a lane group, the groups and the splits:
|y - y64| <= sum_j p_j (1.1 e_j + depth 2^-24) (|v_j| + |y64|).
"""

import numpy as np
import pytest

from asmllm_amd.device import DeviceBuffer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_heads,n_kv,hd,max_ctx,pos", [
    (6, 3, 64, 384, 383), (6, 3, 64, 385, 384), (32, 8, 128, 3072, 3071), (32, 8, 128, 3073, 511),
    (14, 2, 64, 5000, 1536), (8, 1, 128, 5000, 1535), (4, 2, 48, 32768, 32767), (2, 2, 64, 17000, 16384),
    (3, 3, 128, 16384, 16383), (10, 5, 48, 1000, 0),
])
@pytest.mark.parametrize("rope", [False, True])
def test_attention_groups_and_splits(hip, n_heads, n_kv, hd, max_ctx, pos, rope):
    rng = np.random.default_rng(n_heads * 1000 + max_ctx + pos)
    qkv = rng.standard_normal((n_heads + 2 * n_kv) * hd).astype(np.float32)
    kc, vc = (rng.standard_normal((n_kv, max_ctx, hd)).astype(np.float16) for _ in range(2))
    dq, dk, dv = (DeviceBuffer.from_numpy(a) for a in (qkv, kc.view(np.uint16), vc.view(np.uint16)))
    dpos = DeviceBuffer.from_numpy(np.array([pos], np.int32))
    ws = DeviceBuffer(hip.asmhip_attention_decode_workspace(n_heads, hd, max_ctx) * 4)
    out = DeviceBuffer(4 * n_heads * hd)
    table = DeviceBuffer(4 * max_ctx * hd)
    assert hip.asmhip_rope_table(table.ptr, hd, max_ctx, 10000.0, None) == 0
    if rope:
        rc = hip.asmhip_attention_decode_rope_table(dq.ptr, dk.ptr, dv.ptr, ws.ptr, out.ptr, n_heads, n_kv, hd,
                                                    dpos.ptr, max_ctx, table.ptr, None)
    else:
        rc = hip.asmhip_attention_decode(dq.ptr, dk.ptr, dv.ptr, ws.ptr, out.ptr, n_heads, n_kv, hd, dpos.ptr,
                                         max_ctx, None)
    assert rc == 0, hip.asmhip_last_error()
    y = out.download(np.float32, (n_heads, hd)).astype(np.float64)
    k2, v2 = (b.download(np.uint16, (n_kv, max_ctx, hd)).view(np.float16) for b in (dk, dv))
    others = np.arange(max_ctx) != pos
    assert np.array_equal(k2[:, others], kc[:, others]) and np.array_equal(v2[:, others], vc[:, others])
    q = qkv[: n_heads * hd].reshape(n_heads, hd).astype(np.float64)
    if rope:  # the table's own angles: the rows it wrote are checked elsewhere
        cs = table.download(np.float32, (hd,), offset=4 * pos * hd).astype(np.float64).reshape(-1, 2)
        a, b = q[:, 0::2].copy(), q[:, 1::2].copy()
        q[:, 0::2], q[:, 1::2] = a * cs[:, 0] - b * cs[:, 1], a * cs[:, 1] + b * cs[:, 0]
    else:
        assert np.array_equal(k2, kc) and np.array_equal(v2, vc)
    for h in range(n_heads):
        k, v = (c[h // (n_heads // n_kv), : pos + 1].astype(np.float64) for c in (k2, v2))
        ref, bar, _ = _expected(q[h], k, v, max_ctx)
        assert np.all(np.abs(y[h] - ref) <= bar)


def _split_len(max_ctx):
    return 384 if max_ctx <= 3072 else 512


def _expected(q, k, v, max_ctx):
    """The output of one head, its bar, and the weights."""
    hd, sl = len(q), _split_len(max_ctx)
    s = k @ q / np.sqrt(hd)
    p = np.exp(s - s.max())
    p /= p.sum()
    groups = 256 // (16 if hd == 128 else 8)
    depth = sl // groups + groups + -(-max_ctx // sl) + 8
    e = 2.0 ** -24 * ((hd + 8) * (np.abs(k) @ np.abs(q)) / np.sqrt(hd) + 4 * np.abs(s))
    ref = p @ v
    w = p * (1.1 * e + depth * 2.0 ** -24)
    return ref, w @ np.abs(v) + w.sum() * np.abs(ref), p


@pytest.mark.parametrize("n_heads,n_kv,hd,max_ctx,pos", [
    (6, 3, 64, 385, 384), (4, 4, 128, 3072, 3071), (8, 2, 128, 5000, 4608), (4, 2, 48, 32768, 32767),
    (2, 2, 64, 17000, 16384), (3, 3, 128, 16384, 16383), (2, 1, 64, 32768, 32001),
])
@pytest.mark.parametrize("rope", [False, True])
def test_attention_every_split_counts(hip, n_heads, n_kv, hd, max_ctx, pos, rope):
    """One key in each split, and the row at pos, share nearly all of the weight, with values
    of their own: that the loss of any one of them, or another one's weight in its place,
    breaks the bar is itself checked."""
    rng = np.random.default_rng(max_ctx + pos + hd)
    sl = _split_len(max_ctx)
    heavy = np.array([min(s + int(rng.integers(sl)), pos) for s in range(0, pos + 1, sl)])
    heavy[-1] = pos
    qkv = rng.standard_normal((n_heads + 2 * n_kv) * hd).astype(np.float32)
    qkv[: n_heads * hd] = np.tile(qkv[:hd], n_heads)  # one query for all heads: heavy keys lie along it
    qkv[n_heads * hd : (n_heads + n_kv) * hd] = np.tile(qkv[:hd], n_kv)
    kc, vc = (rng.standard_normal((n_kv, max_ctx, hd)).astype(np.float16) for _ in range(2))
    table = DeviceBuffer(4 * max_ctx * hd)
    assert hip.asmhip_rope_table(table.ptr, hd, max_ctx, 10000.0, None) == 0
    q = qkv[:hd].astype(np.float64)
    if rope:
        cs = table.download(np.float32, (hd,), offset=4 * pos * hd).astype(np.float64).reshape(-1, 2)
        a, b = q[0::2].copy(), q[1::2].copy()
        q[0::2], q[1::2] = a * cs[:, 0] - b * cs[:, 1], a * cs[:, 1] + b * cs[:, 0]
    scale = 18 * np.sqrt(hd) / (q @ q)  # of a heavy key along q: a score of 18 against N(0, 1)
    kc[:, heavy] = (q * scale).astype(np.float16)
    if rope:  # the new key is the query's own, scaled alike
        qkv[n_heads * hd : (n_heads + n_kv) * hd] *= np.float32(scale)
    dq, dk, dv = (DeviceBuffer.from_numpy(t) for t in (qkv, kc.view(np.uint16), vc.view(np.uint16)))
    dpos = DeviceBuffer.from_numpy(np.array([pos], np.int32))
    ws = DeviceBuffer(hip.asmhip_attention_decode_workspace(n_heads, hd, max_ctx) * 4)
    out = DeviceBuffer(4 * n_heads * hd)
    args = (dq.ptr, dk.ptr, dv.ptr, ws.ptr, out.ptr, n_heads, n_kv, hd, dpos.ptr, max_ctx)
    rc = (hip.asmhip_attention_decode_rope_table(*args, table.ptr, None) if rope
          else hip.asmhip_attention_decode(*args, None))
    assert rc == 0, hip.asmhip_last_error()
    y = out.download(np.float32, (n_heads, hd)).astype(np.float64)
    k2, v2 = (t.download(np.uint16, (n_kv, max_ctx, hd)).view(np.float16).astype(np.float64) for t in (dk, dv))
    for h in range(n_heads):
        k, v = (c[h // (n_heads // n_kv), : pos + 1] for c in (k2, v2))
        ref, bar, p = _expected(q, k, v, max_ctx)
        assert p[heavy].min() > 0.5 / len(heavy)
        for j in heavy:  # the output without position j
            assert len(heavy) == 1 or np.any(np.abs((ref - p[j] * v[j]) / (1 - p[j]) - ref) > 4 * bar)
        assert np.all(np.abs(y[h] - ref) <= bar)


@pytest.mark.parametrize("n_heads,n_kv,hd,max_ctx,pos", [
    (4, 4, 64, 300, 100), (8, 2, 128, 300, 299), (6, 3, 48, 400, 0), (6, 6, 128, 5000, 4000),
])
@pytest.mark.parametrize("rope", [False, True])
def test_attention_new_row_past_fp16(hip, n_heads, n_kv, hd, max_ctx, pos, rope):
    """A v element at the current position that rounds to an fp16 infinity gives that
    infinity in its own dimension and leaves the others' bits alone."""
    rng = np.random.default_rng(hd + pos)
    qkv = rng.standard_normal((n_heads + 2 * n_kv) * hd).astype(np.float32)
    kc, vc = (rng.standard_normal((n_kv, max_ctx, hd)).astype(np.float16) for _ in range(2))
    dpos = DeviceBuffer.from_numpy(np.array([pos], np.int32))
    ws = DeviceBuffer(hip.asmhip_attention_decode_workspace(n_heads, hd, max_ctx) * 4)
    table = DeviceBuffer(4 * max_ctx * hd)
    assert hip.asmhip_rope_table(table.ptr, hd, max_ctx, 10000.0, None) == 0

    def run(a, b):
        new, cache = qkv.copy(), vc.copy()
        v = new[(n_heads + n_kv) * hd:].reshape(n_kv, hd)
        v[:, 3], v[:, hd - 1] = a, b
        with np.errstate(over="ignore"):
            cache[:, pos] = v.astype(np.float16)
        dq, dk, dv = (DeviceBuffer.from_numpy(t) for t in (new, kc.view(np.uint16), cache.view(np.uint16)))
        out = DeviceBuffer(4 * n_heads * hd)
        args = (dq.ptr, dk.ptr, dv.ptr, ws.ptr, out.ptr, n_heads, n_kv, hd, dpos.ptr, max_ctx)
        rc = (hip.asmhip_attention_decode_rope_table(*args, table.ptr, None) if rope
              else hip.asmhip_attention_decode(*args, None))
        assert rc == 0, hip.asmhip_last_error()
        return out.download(np.float32, (n_heads, hd))

    y, plain = run(1e5, -7e4), run(1.0, 1.0)
    assert np.all(y[:, 3] == np.inf) and np.all(y[:, hd - 1] == -np.inf)
    rest = np.setdiff1d(np.arange(hd), [3, hd - 1])
    assert np.array_equal(y[:, rest].view(np.uint32), plain[:, rest].view(np.uint32))
