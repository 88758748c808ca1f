"""GPU parity of the GEMM's narrow tiles (few rows of A): every form of the operands
bitwise the oracle at one to four and more 16-row tiles, ragged M and every remainder
of a K step, on both sides of the choice of tiles, with scales of every size.
"""

import numpy as np
import pytest

from asmllm_amd import gguf
from asmllm_amd.device import DeviceBuffer, synchronize

pytestmark = pytest.mark.gpu


def _operands(seed, T, M, K):
    rng = np.random.default_rng(seed)
    out = []
    for rows in (M, T):
        n = rng.integers(-128, 128, (rows, K // 32, 32)).astype(np.int8)
        d = (rng.standard_normal((rows, K // 32)) * np.exp2(rng.integers(-16, 8, (rows, K // 32)))).astype(np.float16)
        d[rng.random(d.shape) < 0.05] = np.float16(2.0 ** -24)
        out.append(np.concatenate([d[..., None].view(np.uint8), n.view(np.uint8)], -1))
    return out


def _run(hip, form, w, a, T, M, K):
    dc = DeviceBuffer.from_numpy(np.full((T, M), np.nan, np.float32))
    if form == "split":
        bufs = [DeviceBuffer.from_numpy(np.ascontiguousarray(v)) for v in (*gguf.split_q8_0(w), *gguf.split_q8_0(a))]
        rc = hip.asmhip_gemm_q8_split(bufs[0].ptr, bufs[1].ptr, bufs[2].ptr, bufs[3].ptr, dc.ptr, T, M, K, None)
    else:
        dw, da = DeviceBuffer.from_numpy(w), DeviceBuffer.from_numpy(a)
        if form == "tiled":
            tw = DeviceBuffer(hip.asmhip_gemm_q8_0_tiled_weight_bytes(M, K))
            ta = DeviceBuffer.from_numpy(np.full(hip.asmhip_gemm_q8_0_tiled_activation_bytes(T, K), 0xFF, np.uint8))
            assert hip.asmhip_gemm_q8_0_tile_weights(dw.ptr, tw.ptr, M, K, None) == 0
            # the activation tiles' padding rows hold NaN scales: they must not reach C
            nb = K // 32
            host = ta.download(np.uint8, (ta.nbytes,))
            t, b = np.meshgrid(np.arange(T), np.arange(nb), indexing="ij")
            at = ((t // 64 * (nb // 2) + b // 2) * 64 + t % 64) * 68 + b % 2 * 34
            host[at[..., None] + np.arange(34)] = a
            ta.upload(host)
            rc = hip.asmhip_gemm_q8_0_tiled(tw.ptr, ta.ptr, dc.ptr, T, M, K, None)
        else:
            rc = hip.asmhip_gemm_q8_0(dw.ptr, da.ptr, dc.ptr, T, M, K, None)
    assert rc == 0, hip.asmhip_last_error()
    synchronize()
    return dc.download(np.float32, (T, M))


@pytest.mark.parametrize("form", ["blocks", "tiled", "split"])
@pytest.mark.parametrize("T,M,K", [
    (1, 1, 64), (5, 17, 192), (16, 100, 256), (17, 130, 320), (24, 15, 576), (32, 129, 64), (33, 16, 448), (48, 33, 1088),
    (49, 31, 128), (64, 130, 384), (65, 17, 704), (130, 250, 512), (200, 40, 1984), (3, 300, 4096), (40, 48, 2112),
    (50, 8300, 64), (130, 2800, 576), (64, 8225, 192),  # two columns of tiles a workgroup
    (1, 16384, 64), (1, 16385, 64), (70, 8200, 128),  # 1024 workgroups, and the larger tiles from there
    (17, 12288, 64), (17, 12289, 64), (17, 16384, 2048),  # 768 for 17 to 32 rows of a short K
    (65, 6144, 64), (65, 6145, 64),  # 768, the tile layout's
    (65, 4096, 64), (65, 4097, 64), (65, 8192, 2048), (65, 8193, 2048),  # 512 blocks, 1024 from K = 2048
    (40, 8192, 64), (40, 8193, 64), (40, 8300, 2048),  # three tiles of rows, and four with one idle
])
def test_narrow_gemm_is_the_oracle(hip, oracle, form, T, M, K):
    w, a = _operands(T * 31 + M + K, T, M, K)
    np.testing.assert_array_equal(_run(hip, form, w, a, T, M, K), oracle.gemm_q8_0(w, a, 8))


@pytest.mark.parametrize("T,M,K", [(5, 17, 32), (24, 40, 96), (50, 33, 544), (64, 20, 1120), (100, 4200, 96)])
def test_narrow_gemm_odd_block_counts(hip, oracle, T, M, K):
    """The split planes take the narrow tiles at any K % 32; blocks keep the general kernel."""
    w, a = _operands(T + M + K, T, M, K)
    ref = oracle.gemm_q8_0(w, a, 8)
    for form in ("split", "blocks"):
        np.testing.assert_array_equal(_run(hip, form, w, a, T, M, K), ref)
