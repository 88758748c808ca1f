"""GPU parity of the decode attention where its grid and its merge can go wrong:
grouped heads whose (kv head, split) pairs do and do not divide over the 8 dies,
positions on both sides of a split's edge, and every number of splits the merge
walks in batches, against float64 over the same fp16 rows.

Bar: scores within e = (hd + 4) roundings of sum |q||k| / sqrt(hd), so weights
within exp(2 e); the sums over positions and splits add pos + 80 roundings.
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
        s = k @ q[h] / np.sqrt(hd)
        p = np.exp(s - s.max())
        ref = p @ v / p.sum()
        e = (hd + 4) * 2.0 ** -24 * (np.abs(k) @ np.abs(q[h])).max() / np.sqrt(hd)
        assert np.all(np.abs(y[h] - ref) <= (2 * e + (pos + 80) * 2.0 ** -24) * np.abs(v).max())


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
