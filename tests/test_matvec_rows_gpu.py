"""GPU parity of the fp32 row kernels over the forms their dispatch divides: every
block type and layout, ragged K around each register pass and LDS unit, few and many
rows, the fused pre-ops, SwiGLU and the residual add, against float64 on the same
bytes.

Bar, per row: each product is exact; the sums are 8 roundings deep within an item of 8
columns, K / 2048 over a lane's blocks, 12 over items, lanes and waves, and a pre-op adds
8: well inside |y - y64| <= (48 + min(K / 32, 96) + K / 2048) 2^-24 sum |w| |x|, which the
pair kernels of the longest rows share.
"""

import numpy as np
import pytest

from asmllm_amd import gguf, native
from asmllm_amd.device import DeviceBuffer

pytestmark = pytest.mark.gpu


def _weights(rng, q, M, K):
    """GGUF blocks and the exact float64 matrix."""
    nb = K // 32
    d = (rng.standard_normal((M, nb)) * 0.01).astype(np.float16)
    if q == 8:
        n = rng.integers(-128, 128, (M, nb, 32)).astype(np.int8)
        b = np.concatenate([d[..., None].view(np.uint8), n.view(np.uint8)], -1)
        v = n.astype(np.float64)
    elif q == 4:
        qs = rng.integers(0, 256, (M, nb, 16)).astype(np.uint8)
        b = np.concatenate([d[..., None].view(np.uint8), qs], -1)
        v = np.concatenate([qs & 15, qs >> 4], -1).astype(np.float64) - 8
    else:
        ql = rng.integers(0, 256, (M, nb, 16)).astype(np.uint8)
        qh = rng.integers(0, 256, (M, nb, 4)).astype(np.uint8)
        b = gguf.pack_q5_0(ql, qh, d)
        return b, gguf.dequantize_q5_0(b).astype(np.float64)
    return np.ascontiguousarray(b), (v * d[..., None].astype(np.float64)).reshape(M, K)


def _long(rng, q, M, K):
    """M rows, the first 256 again and again, and their exact matrix."""
    b, w = _weights(rng, q, 256, K)
    return np.ascontiguousarray(np.concatenate([b] * (M // 256 + 1))[:M]), w, np.arange(M) % 256


def _bar(w, x, K):
    return (48 + min(K / 32, 96) + K / 2048) * 2.0 ** -24 * (np.abs(w) @ np.abs(x).astype(np.float64)) + 1e-30


def _call(hip, q, split, b, x, M, K):
    dx, dy = DeviceBuffer.from_numpy(x), DeviceBuffer.from_numpy(np.full(M, np.nan, np.float32))
    if split:
        parts = {4: gguf.split_q4_0, 5: gguf.split_q5_0, 8: gguf.split_q8_0}[q](b)
        bufs = [DeviceBuffer.from_numpy(np.ascontiguousarray(p).view(np.uint8)) for p in parts]
        fn = {4: hip.asmhip_matmul_q4_split, 5: hip.asmhip_matmul_q5_split, 8: hip.asmhip_matmul_q8_split}[q]
        rc = fn(*[t.ptr for t in bufs], dx.ptr, dy.ptr, M, K, None)
    else:
        bufs = [DeviceBuffer.from_numpy(b)]
        fn = {4: hip.asmhip_matmul_q4_0, 5: hip.asmhip_matmul_q5_0, 8: hip.asmhip_matmul_q8_0}[q]
        rc = fn(bufs[0].ptr, dx.ptr, dy.ptr, M, K, None)
    assert rc == 0, hip.asmhip_last_error()
    return dy.download(np.float32, (M,))


SHAPES = [(1, 32), (5, 64), (17, 96), (300, 288), (700, 512), (33, 544), (2100, 768), (63, 1024), (520, 1056),
          (70, 2080), (2100, 2080), (3, 4128), (600, 5504), (40, 8160), (24, 8224), (20, 16416), (9, 21024),
          (9000, 288), (17000, 544), (6145, 768)]


@pytest.mark.parametrize("q", [4, 5, 8])
@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("M,K", SHAPES)
def test_row_kernels_shapes(hip, q, split, M, K):
    rng = np.random.default_rng(M + K + q)
    b, w = _weights(rng, q, M, K)
    x = (rng.standard_normal(K) * np.exp(rng.standard_normal(K))).astype(np.float32)
    y = _call(hip, q, split, b, x, M, K)
    assert np.all(np.abs(y - w @ x.astype(np.float64)) <= _bar(w, x, K))
    for col in (0, K // 2 - 1, K - 1):  # one column, exactly: its bytes and no others
        one = np.zeros(K, np.float32)
        one[col] = 1.0
        assert np.array_equal(_call(hip, q, split, b, one, M, K).astype(np.float64), w[:, col])


@pytest.mark.parametrize("q", [4, 5, 8])
@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("M,K", [(1, 32), (300, 288), (9000, 512), (6144, 768), (2100, 1024)])
def test_row_kernels_sums_in_64_bits(hip, q, split, M, K):
    """Up to 1024 columns only fours of products round in 32 bits (four fused multiply-adds of
    at most u each), and the result.  The bound is far above what random signs give, so the
    error's norm is held too: with every sum in 32 bits it is 8.3e-8 to 9.2e-8 of the
    result's at these K (computed in the kernels' order), with 64-bit sums 4.4e-8 to 4.8e-8."""
    rng = np.random.default_rng(M + K + q)
    b, w = _weights(rng, q, M, K)
    x = rng.standard_normal(K).astype(np.float32)
    y, e, u = _call(hip, q, split, b, x, M, K), w @ x.astype(np.float64), 2.0 ** -24
    bar = 4.01 * u * (np.abs(w) @ np.abs(x).astype(np.float64)) + 1.01 * u * np.abs(e) + 1e-30
    assert (np.abs(y - e) <= bar).all()
    if M >= 300:
        assert np.linalg.norm(y - e) / np.linalg.norm(e) < 6e-8


ROWS_KS = [288, 544, 768, 1024, 1056, 1376, 2048 + 32, 3008, 4128, 5504, 6176, 8160, 8224]


def _rows_of_both_kernels(K):
    """Rows enough for every format that leaves matvec_wave at this K."""
    return 33008 if K <= 1376 else 16368


def _prefixes(M):
    return [m for m in (1, 5, 47, 300, 1000, 2049, 4000, 4097, 8100, 8193, 16400) if m < M]


@pytest.mark.parametrize("q", [4, 5, 8])
@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("K", ROWS_KS)
def test_rows_do_not_depend_on_the_number_of_rows(hip, q, split, K):
    """A row's bits are the same for every M, whichever kernel its size picks, and wherever
    the row stands: the leading m rows of a matrix give the first m outputs of the whole,
    whose 256 rows come again and again."""
    M = _rows_of_both_kernels(K) + 1
    rng = np.random.default_rng(K + q)
    b, _, row = _long(rng, q, M, K)
    x = (rng.standard_normal(K) * np.exp(rng.standard_normal(K))).astype(np.float32)
    parts = {4: gguf.split_q4_0, 5: gguf.split_q5_0, 8: gguf.split_q8_0}[q](b) if split else [b]
    bufs = [DeviceBuffer.from_numpy(np.ascontiguousarray(p).view(np.uint8)) for p in parts]
    name = f"asmhip_matmul_q{q}_split" if split else f"asmhip_matmul_q{q}_0"
    dx, dy = DeviceBuffer.from_numpy(x), DeviceBuffer(4 * M)

    def run(m):
        assert getattr(hip, name)(*[t.ptr for t in bufs], dx.ptr, dy.ptr, m, K, None) == 0, hip.asmhip_last_error()
        return dy.download(np.uint32, (m,))

    whole = run(M)
    assert np.array_equal(whole, whole[row])
    for m in _prefixes(M):
        assert np.array_equal(run(m), whole[:m]), m


@pytest.mark.parametrize("q", [4, 8])
@pytest.mark.parametrize("K", [576, 768, 1088, 3008, 4160, 6208, 8000])
@pytest.mark.parametrize("pre", ["rmsnorm", "swiglu"])
@pytest.mark.parametrize("form", ["accumulate", "pairs"])
def test_fused_rows_do_not_depend_on_the_number_of_rows(hip, q, K, pre, form):
    M = _rows_of_both_kernels(K)
    rng = np.random.default_rng(K + q)
    b = _long(rng, q, M, K)[0]
    x, arg, y0 = (rng.standard_normal(n).astype(np.float32) for n in (K, K, M))
    op = {"rmsnorm": native.PRE_RMSNORM, "swiglu": native.PRE_SWIGLU}[pre]
    qt = native.Q4_0 if q == 4 else native.Q8_0
    db, dx, da, work = DeviceBuffer.from_numpy(b), DeviceBuffer.from_numpy(x), DeviceBuffer.from_numpy(arg), DeviceBuffer(4 * M)

    def run(m):
        dy = DeviceBuffer.from_numpy(y0)
        if form == "pairs":
            rc = hip.asmhip_matmul_swiglu(qt, db.ptr, dx.ptr, dy.ptr, m // 2, K, op, da.ptr, 1e-5, work.ptr, None)
        else:
            rc = hip.asmhip_matmul_fused(qt, db.ptr, dx.ptr, dy.ptr, m, K, op, da.ptr, 1e-5, 1, None)
        assert rc == 0, hip.asmhip_last_error()
        return dy.download(np.uint32, (m // 2 if form == "pairs" else m,))

    whole = run(M)
    for m in (m // 16 * 16 + 16 for m in _prefixes(M - 16)):
        y = run(m)
        assert np.array_equal(y, whole[: len(y)]), m


@pytest.mark.parametrize("q", [4, 8])
@pytest.mark.parametrize("M,K", [(33000, 544), (26000, 1088), (13000, 2112), (9000, 3008), (4096, 5504), (17000, 4128)])
def test_row_kernels_error_of_the_norm(hip, q, M, K):
    """|y - y64| of a few thousand rows: 1.0e-7 of the norm with a lane's chains and a tree
    above them (4.8e-8 with 64-bit sums, K <= 1024); a row's block products added one after
    another in fp32 left 1.4e-7 to 2.0e-7 at these K from 1088 to 3008."""
    rng = np.random.default_rng(M + K + q)
    b, _ = _weights(rng, q, M, K)
    x = rng.standard_normal(K).astype(np.float32)
    y, n = _call(hip, q, False, b, x, M, K).astype(np.float64), 4000
    w = (gguf.dequantize_q4_0 if q == 4 else gguf.dequantize_q8_0)(b[:n]).astype(np.float64).reshape(n, K)
    e = w @ x.astype(np.float64)
    assert np.linalg.norm(y[:n] - e) / np.linalg.norm(e) < (6e-8 if K <= 1024 else 1.2e-7)


@pytest.mark.parametrize("q", [4, 5, 8])
@pytest.mark.parametrize("M,K", [(300, 288), (2000, 1024), (700, 1088), (33000, 1088), (600, 5504), (70, 8224), (16380, 3008)])
def test_row_kernels_x_off_16_bytes(hip, q, M, K):
    rng = np.random.default_rng(M + K)
    b, _ = _weights(rng, q, M, K)
    x = rng.standard_normal(K + 4).astype(np.float32)
    db, dx, dy = DeviceBuffer.from_numpy(b), DeviceBuffer.from_numpy(x), DeviceBuffer(4 * M)
    fn = {4: hip.asmhip_matmul_q4_0, 5: hip.asmhip_matmul_q5_0, 8: hip.asmhip_matmul_q8_0}[q]
    for off in (1, 2, 3):
        assert fn(db.ptr, dx.ptr + 4 * off, dy.ptr, M, K, None) == 0, hip.asmhip_last_error()
        assert np.array_equal(dy.download(np.float32, (M,)), _call(hip, q, False, b, x[off:off + K], M, K)), off


@pytest.mark.parametrize("M,K", [(4096, 5504), (16400, 2080), (5000, 8224), (16380, 2080), (8190, 5504)])
def test_row_kernels_many_units(hip, M, K):
    """Several units per wave, and rows cut into chunks (matvec_rows' stream)."""
    rng = np.random.default_rng(M)
    b, w = _weights(rng, 8, M, K)
    x = rng.standard_normal(K).astype(np.float32)
    y = _call(hip, 8, False, b, x, M, K)
    assert np.all(np.abs(y - w @ x.astype(np.float64)) <= _bar(w, x, K))


@pytest.mark.parametrize("q", [4, 8])
@pytest.mark.parametrize("M,K", [(16, 64), (304, 320), (1040, 768), (64, 1088), (160, 8256), (16400, 576)])
@pytest.mark.parametrize("pre", ["none", "rmsnorm", "swiglu"])
@pytest.mark.parametrize("form", ["plain", "accumulate", "pairs"])
def test_row_kernels_fused(hip, q, M, K, pre, form):
    rng = np.random.default_rng(M * 7 + K + q)
    b, w = _weights(rng, q, M, K)
    x, arg, y0 = (rng.standard_normal(n).astype(np.float32) for n in (K, K, M))
    x64, a64 = x.astype(np.float64), arg.astype(np.float64)
    xin = {"none": x64, "rmsnorm": x64 / np.sqrt((x64 ** 2).mean() + 1e-5) * a64,
           "swiglu": x64 / (1 + np.exp(-x64)) * a64}[pre]
    op = {"none": native.PRE_NONE, "rmsnorm": native.PRE_RMSNORM, "swiglu": native.PRE_SWIGLU}[pre]
    db, dx, da = DeviceBuffer.from_numpy(b), DeviceBuffer.from_numpy(x), DeviceBuffer.from_numpy(arg)
    dy = DeviceBuffer.from_numpy(y0)
    qt = native.Q4_0 if q == 4 else native.Q8_0
    ref, bar = w @ xin, _bar(w, xin, K)
    if form == "pairs":
        work = DeviceBuffer(4 * M)
        rc = hip.asmhip_matmul_swiglu(qt, db.ptr, dx.ptr, dy.ptr, M // 2, K, op, da.ptr, 1e-5, work.ptr, None)
        assert rc == 0, hip.asmhip_last_error()
        y = dy.download(np.float32, (M // 2,))
        g, u = (ref.reshape(-1, 2, 8)[:, i].reshape(-1) for i in (0, 1))
        bg, bu = (bar.reshape(-1, 2, 8)[:, i].reshape(-1) for i in (0, 1))
        sg = g / (1 + np.exp(-g))
        # |d silu| <= 1.1 |dg|; the division, exponential and product: 8 roundings
        assert np.all(np.abs(y - sg * u) <= 1.1 * bg * (np.abs(u) + bu) + np.abs(sg) * bu + 2.0 ** -21 * np.abs(sg * u) + 1e-30)
        return
    rc = hip.asmhip_matmul_fused(qt, db.ptr, dx.ptr, dy.ptr, M, K, op, da.ptr, 1e-5, int(form == "accumulate"), None)
    assert rc == 0, hip.asmhip_last_error()
    y = dy.download(np.float32, (M,))
    if form == "accumulate":
        ref, bar = ref + y0, bar + 2.0 ** -23 * (np.abs(y0) + np.abs(ref))
    assert np.all(np.abs(y - ref) <= bar)


@pytest.mark.parametrize("qt", [native.Q4_0, native.Q8_0])
@pytest.mark.parametrize("n_heads,hd,max_ctx,pos,M", [(6, 48, 256, 100, 288), (6, 48, 3072, 3000, 288), (2, 64, 900, 899, 70), (6, 128, 256, 100, 6144), (6, 128, 256, 100, 6145),
                                                       (8, 128, 770, 5, 1024), (16, 64, 3072, 1, 3000)])
def test_row_kernels_merge_attention(hip, qt, n_heads, hd, max_ctx, pos, M):
    """The split states merged by the o matvec give the bits of the merge launch and
    the matvec over its output."""
    rng = np.random.default_rng(pos + M)
    K = n_heads * hd
    b, _ = _weights(rng, 4 if qt == native.Q4_0 else 8, M, K)
    qkv = rng.standard_normal(3 * K).astype(np.float32)
    cache = [rng.standard_normal((n_heads, max_ctx, hd)).astype(np.float16).view(np.uint16) for _ in range(2)]
    db, dq, dk, dv = (DeviceBuffer.from_numpy(a) for a in (b, qkv, *cache))
    dpos = DeviceBuffer.from_numpy(np.array([pos], np.int32))
    ws = DeviceBuffer(4 * hip.asmhip_attention_decode_workspace(n_heads, hd, max_ctx))
    table, attn, work = DeviceBuffer(4 * max_ctx * hd), DeviceBuffer(4 * K), DeviceBuffer(4 * K)
    y0 = rng.standard_normal(M).astype(np.float32)
    d1, d2 = DeviceBuffer.from_numpy(y0), DeviceBuffer.from_numpy(y0)
    calls = [hip.asmhip_rope_table(table.ptr, hd, max_ctx, 10000.0, None),
             hip.asmhip_attention_decode_partials_rope_table(dq.ptr, dk.ptr, dv.ptr, ws.ptr, n_heads, n_heads, hd,
                                                             dpos.ptr, max_ctx, table.ptr, None),
             hip.asmhip_matmul_attn_output(qt, db.ptr, ws.ptr, work.ptr, d1.ptr, M, n_heads, hd, max_ctx, 1, None),
             hip.asmhip_attention_decode_rope_table(dq.ptr, dk.ptr, dv.ptr, ws.ptr, attn.ptr, n_heads, n_heads, hd,
                                                    dpos.ptr, max_ctx, table.ptr, None),
             hip.asmhip_matmul_fused(qt, db.ptr, attn.ptr, d2.ptr, M, K, native.PRE_NONE, None, 0.0, 1, None)]
    assert calls == [0] * 5, hip.asmhip_last_error()
    assert np.array_equal(d1.download(np.uint32, (M,)), d2.download(np.uint32, (M,)))


@pytest.mark.parametrize("q", [4, 8])
@pytest.mark.parametrize("M,K", [(16, 32), (864, 288), (2096, 544), (64, 1056), (176, 4128), (32, 8224), (16400, 1056)])
@pytest.mark.parametrize("swiglu", [0, 1])
def test_row_kernels_rmsnorm_any_width(hip, q, M, K, swiglu):
    rng = np.random.default_rng(M + K + q + 1)
    b, w = _weights(rng, q, M, K)
    x, g = (rng.standard_normal(K).astype(np.float32) for _ in range(2))
    x64 = x.astype(np.float64)
    xin = x64 / np.sqrt((x64 ** 2).mean() + 1e-5) * g.astype(np.float64)
    db, dx, dg, dy = (DeviceBuffer.from_numpy(a) for a in (b, x, g, np.full(M, np.nan, np.float32)))
    rc = hip.asmhip_matmul_rmsnorm(native.Q4_0 if q == 4 else native.Q8_0, db.ptr, dx.ptr, dg.ptr, 1e-5, dy.ptr, M, K,
                                   swiglu, None)
    assert rc == 0, hip.asmhip_last_error()
    y, ref, bar = dy.download(np.float32, (M,)), w @ xin, _bar(w, xin, K)
    if not swiglu:
        assert np.all(np.abs(y - ref) <= bar)
        return
    gate, up = (ref.reshape(-1, 2, 8)[:, i].reshape(-1) for i in (0, 1))
    bg, bu = (bar.reshape(-1, 2, 8)[:, i].reshape(-1) for i in (0, 1))
    sg = gate / (1 + np.exp(-gate))
    assert np.all(np.abs(y[: M // 2] - sg * up) <= 1.1 * bg * (np.abs(up) + bu) + np.abs(sg) * bu +
                  2.0 ** -21 * np.abs(sg * up) + 1e-30)
    assert np.all(np.isnan(y[M // 2:]))


@pytest.mark.parametrize("qt", [native.Q4_0, native.Q8_0])
@pytest.mark.parametrize("H,K", [(296, 320), (1024, 1088), (2048, 2048), (520, 4096)])
@pytest.mark.parametrize("pre,over", [("none", "x")] + [(p, o) for p in ("rmsnorm", "swiglu") for o in ("x", "arg", "arg's end")])
def test_swiglu_over_its_inputs(hip, qt, H, K, pre, over):
    """h over x or over the pre-op's argument: the pairs go through `work`, so that no
    workgroup writes what another still reads, with the bits of the call into a buffer
    of its own (which leaves `work` alone)."""
    rng = np.random.default_rng(H + K)
    b, _ = _weights(rng, 4 if qt == native.Q4_0 else 8, 2 * H, K)
    op = {"none": native.PRE_NONE, "rmsnorm": native.PRE_RMSNORM, "swiglu": native.PRE_SWIGLU}[pre]
    n = max(H, K) + K
    x, arg = (rng.standard_normal(n).astype(np.float32) for _ in range(2))
    db, dh = DeviceBuffer.from_numpy(b), DeviceBuffer(4 * H)

    def call(target):
        dx, da = DeviceBuffer.from_numpy(x), DeviceBuffer.from_numpy(arg)
        work = DeviceBuffer.from_numpy(np.full(2 * H, np.nan, np.float32))
        buf, offset = {"own": (dh, 0), "x": (dx, 0), "arg": (da, 0), "arg's end": (da, 4 * (K - 1))}[target]
        rc = hip.asmhip_matmul_swiglu(qt, db.ptr, dx.ptr, buf.ptr + offset, H, K, op, da.ptr if op else None, 1e-5,
                                      work.ptr, None)
        assert rc == 0, hip.asmhip_last_error()
        return buf.download(np.uint32, (H,), offset=offset), work.download(np.float32, (2 * H,))

    own, untouched = call("own")
    y, work = call(over)
    assert np.isnan(untouched).all() and not np.isnan(work).any()
    assert np.array_equal(y, own)


# Above about 25400 columns (Q8: 21700) x no longer fits LDS beside a unit of the row kernels:
# up to 38400 the pair kernels take K % 64 == 0, in forms of 1, 2, 4 and (Q4) 8 rows a wave.
LONG = [(40, 25600), (7, 38400), (4100, 25600), (8200, 32768), (16400, 25600)]


@pytest.mark.parametrize("q", [4, 5, 8])
@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("M,K", LONG)
def test_pair_kernels_long_rows(hip, q, split, M, K):
    rng = np.random.default_rng(M + K + q)
    b, w, row = _long(rng, q, M, K)
    x = rng.standard_normal(K).astype(np.float32)
    ref, bar = w @ x.astype(np.float64), _bar(w, x, K)
    assert np.all(np.abs(_call(hip, q, split, b, x, M, K) - ref[row]) <= bar[row])
    one = np.zeros(K, np.float32)
    one[K - 33] = 1.0
    assert np.array_equal(_call(hip, q, split, b, one, M, K).astype(np.float64), w[row, K - 33])


@pytest.mark.parametrize("q", [4, 8])
@pytest.mark.parametrize("M,K", [(48, 25600), (8208, 25600), (32, 38400)])
@pytest.mark.parametrize("pre", ["none", "rmsnorm", "swiglu"])
@pytest.mark.parametrize("form", ["accumulate", "pairs"])
def test_pair_kernels_fused(hip, q, M, K, pre, form):
    """The pre-ops, the residual add, and the two launches of SwiGLU through `work`."""
    rng = np.random.default_rng(M + K + q)
    b, w, row = _long(rng, q, M, K)
    x, arg, y0 = (rng.standard_normal(n).astype(np.float32) for n in (K, K, M))
    x64, a64 = x.astype(np.float64), arg.astype(np.float64)
    xin = {"none": x64, "rmsnorm": x64 / np.sqrt((x64 ** 2).mean() + 1e-5) * a64,
           "swiglu": x64 / (1 + np.exp(-x64)) * a64}[pre]
    op = {"none": native.PRE_NONE, "rmsnorm": native.PRE_RMSNORM, "swiglu": native.PRE_SWIGLU}[pre]
    db, dx, da, dy, work = (DeviceBuffer.from_numpy(a) for a in (b, x, arg, y0, np.full(M, np.nan, np.float32)))
    qt = native.Q4_0 if q == 4 else native.Q8_0
    ref, bar = (w @ xin)[row], _bar(w, xin, K)[row]
    if form == "accumulate":
        rc = hip.asmhip_matmul_fused(qt, db.ptr, dx.ptr, dy.ptr, M, K, op, da.ptr, 1e-5, 1, None)
        assert rc == 0, hip.asmhip_last_error()
        assert np.all(np.abs(dy.download(np.float32, (M,)) - (ref + y0)) <= bar + 2.0 ** -23 * (np.abs(y0) + np.abs(ref + y0)))
        return
    rc = hip.asmhip_matmul_swiglu(qt, db.ptr, dx.ptr, dy.ptr, M // 2, K, op, da.ptr, 1e-5, work.ptr, None)
    assert rc == 0, hip.asmhip_last_error()
    assert not np.isnan(work.download(np.float32, (M,))).any()
    g, u = (ref.reshape(-1, 2, 8)[:, i].reshape(-1) for i in (0, 1))
    bg, bu = (bar.reshape(-1, 2, 8)[:, i].reshape(-1) for i in (0, 1))
    sg = g / (1 + np.exp(-g))
    assert np.all(np.abs(dy.download(np.float32, (M // 2,)) - sg * u) <= 1.1 * bg * (np.abs(u) + bu) + np.abs(sg) * bu +
                  2.0 ** -21 * np.abs(sg * u) + 1e-30)


def test_row_kernels_rmsnorm_refusals(hip):
    d = DeviceBuffer(1 << 16)
    args = (d.ptr, d.ptr, d.ptr, 1e-5, d.ptr)
    assert hip.asmhip_matmul_rmsnorm(native.Q4_0, *args, 16, 40, 0, None) == native.ERR_INVALID_ARGUMENT
    assert hip.asmhip_matmul_rmsnorm(native.Q4_0, *args, 24, 32, 1, None) == native.ERR_INVALID_ARGUMENT
    assert hip.asmhip_matmul_rmsnorm(native.Q4_0, *args, 16, 64000, 0, None) == native.ERR_UNSUPPORTED
    assert hip.asmhip_matmul_rmsnorm(native.Q5_0, *args, 16, 32, 0, None) == native.ERR_INVALID_ARGUMENT
    # the fused entry points keep refusing the widths they refused
    assert hip.asmhip_matmul_fused(native.Q4_0, d.ptr, d.ptr, d.ptr, 16, 288, native.PRE_RMSNORM, d.ptr, 1e-5, 0,
                                   None) == native.ERR_UNSUPPORTED
