"""GPU parity of asmhip_attention over the forms its kernels divide: whole and
ragged key blocks and query tiles, head_dim below, at and above each padded
size, and the shapes and alignments only the row kernel takes.

Bar, per output row: with every score within e of its exact value (e = (hd + 2)
roundings of sum |q||k| scale), each weight is within a factor exp(2 e), and
the sums over keys add seq + 16 roundings: |y - y64| <= (2 e + (seq + 16)
2^-23) max |v|.
"""

import numpy as np
import pytest

from asmllm_amd.device import DeviceBuffer

pytestmark = pytest.mark.gpu


def _run(hip, q, k, v, scale, offset=0):
    seq, hd = q.shape
    bufs = []
    for a in (q, k, v, np.zeros_like(q)):
        b = DeviceBuffer(a.nbytes + 16)
        b.upload(np.ascontiguousarray(a), offset=offset)
        bufs.append(b)
    rc = hip.asmhip_attention(*[b.ptr + offset for b in bufs], seq, hd, scale, None)
    assert rc == 0, hip.asmhip_last_error()
    return bufs[3].download(np.float32, (seq, hd), offset=offset)


def _ref(q, k, v, scale):
    q, k, v = (a.astype(np.float64) for a in (q, k, v))
    s = q @ k.T * scale
    p = np.exp(s - s.max(-1, keepdims=True))
    return (p / p.sum(-1, keepdims=True)) @ v


def _bound(q, k, v, scale):
    seq, hd = q.shape
    e = (hd + 2) * 2.0 ** -24 * (np.abs(q).astype(np.float64) @ np.abs(k).astype(np.float64).T * scale).max(-1)
    return (2 * e + (seq + 16) * 2.0 ** -23)[:, None] * np.abs(v).max()


@pytest.mark.parametrize("seq,hd,offset", [
    (1, 64, 0), (5, 128, 0), (16, 64, 0), (17, 128, 0), (127, 64, 0), (129, 128, 0), (300, 48, 0), (300, 80, 0),
    (130, 4, 0), (70, 60, 0), (70, 68, 0), (70, 132, 0), (200, 256, 0),
    # 16-row tiles
    (1024, 64, 0), (1025, 128, 0), (2100, 64, 0), (1040, 48, 0), (1033, 80, 0), (1033, 20, 0), (1033, 100, 0),
    (33, 30, 0), (33, 260, 0), (65, 64, 4),  # row kernel: head_dim % 4, head_dim > 256, unaligned rows
])
def test_attention_shapes(hip, seq, hd, offset):
    rng = np.random.default_rng(seq * 1000 + hd)
    q, k, v = (rng.standard_normal((seq, hd)).astype(np.float32) for _ in range(3))
    for scale in (1.0 / np.sqrt(hd), 1.0):
        y = _run(hip, q, k, v, float(scale), offset)
        assert np.all(np.abs(y - _ref(q, k, v, scale)) <= _bound(q, k, v, scale))


@pytest.mark.parametrize("hd", [64, 128, 30])
def test_attention_infinite_scores(hip, hd):
    """A key at minus infinity weighs nothing, wherever its block stands; a row
    whose every score is minus infinity, or holds a NaN, is NaN."""
    rng = np.random.default_rng(hd)
    seq = 150
    q, k, v = (rng.standard_normal((seq, hd)).astype(np.float32) for _ in range(3))
    q[:, 0] = 1.0
    dead = np.r_[0:40, 149]
    k[dead, 0] = -np.inf
    y = _run(hip, q, k, v, 0.5)
    live = np.setdiff1d(np.arange(seq), dead)
    s = q.astype(np.float64) @ k[live].astype(np.float64).T * 0.5
    p = np.exp(s - s.max(-1, keepdims=True))
    ref = (p / p.sum(-1, keepdims=True)) @ v[live].astype(np.float64)
    assert np.all(np.abs(y - ref) <= _bound(q, np.where(np.isinf(k), 0, k), v, 0.5))
    k[:, 0] = -np.inf
    assert np.all(np.isnan(_run(hip, q, k, v, 0.5)))
    k[:, 0] = 1.0
    k[77, 3] = np.nan
    assert np.all(np.isnan(_run(hip, q, k, v, 0.5)))


@pytest.mark.parametrize("seq,hd", [(64, 64), (600, 128), (1100, 64), (1100, 48), (40, 30)])
def test_attention_values_near_the_largest_float(hip, seq, hd):
    """Weights stay at most 1 while later keys' scores rise above the first ones', so
    values whose sum over the keys is a third of the largest float come through."""
    rng = np.random.default_rng(seq + hd)
    q, k = np.zeros((seq, hd), np.float32), np.zeros((seq, hd), np.float32)
    q[:, 0] = 1.0
    k[:, 0] = np.linspace(0, 6.8, seq)  # 9.8 in powers of two
    v = (rng.uniform(0.5, 1.0, (seq, hd)) * 1e38 / seq).astype(np.float32)
    y = _run(hip, q, k, v, 1.0)
    assert np.isfinite(y).all()
    assert np.all(np.abs(y - _ref(q, k, v, 1.0)) <= _bound(q, k, v, 1.0))


@pytest.mark.parametrize("seq,hd", [(300, 128), (1100, 64)])
@pytest.mark.parametrize("scale", [-0.25, 0.0, 1e-30])
def test_attention_scale_of_any_sign(hip, seq, hd, scale):
    rng = np.random.default_rng(seq)
    q, k, v = (rng.standard_normal((seq, hd)).astype(np.float32) for _ in range(3))
    assert np.all(np.abs(_run(hip, q, k, v, scale) - _ref(q, k, v, scale)) <= _bound(q, k, v, abs(scale)))
