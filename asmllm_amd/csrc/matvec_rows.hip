// Quantized matvec over whole rows in fp32 (VALU), for the shapes the int8-MFMA
// stream does not take: any K % 32 == 0, GGUF blocks or split planes, and the work
// the decode step fuses around its matvecs.
//
// y[m] = sum_b d[m,b] * sum_j (q[m,b,j] - z) * x[32b + j], the arithmetic of the
// reference's asm_matmul_q4 / _q5 / _q8 (src/kernels/x86_64/matmul_q4_avx2.asm:57-287,
// matmul_q5_avx2.asm:52-238, matmul_q8_avx2.asm:51-194).
//
// matvec_rows.  A unit is one wave's contiguous run of blocks: `rw` whole rows (small K: a row of 9
// blocks would leave most lanes idle), or a row's chunk of at most 64 NI blocks.  Its
// bytes are requested as consecutive 16-byte pieces (split planes: each lane its own
// block), parked in the wave's own piece of LDS, and read back one block a lane: a
// lane's block is 18, 22 or 34 bytes at a 2-byte address, and loads of those strides
// touch three lines per four lanes.  The next unit is requested as soon as the
// registers are parked, so a wave always has one unit in flight; waves wait for no
// one but at the start, for x.  x is staged once per workgroup (36 floats per block:
// the 16-byte reads of eight consecutive blocks fall on distinct banks), and a
// workgroup of 16 waves walks the tiles of 16 rw rows b, b + grid, ...
// Every weight becomes an exact float by one sign-extending byte conversion: a Q4
// nibble n as the byte 16 (n - 8), a Q5 value b as 8 (b - 16), with x staged as x / 16
// and x / 8 (exact).
//
// Bound by the read of the weights and, at the smallest shapes, by the chain x ->
// barrier -> dot -> reduction -> store of one workgroup.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace asmhip {

namespace {

constexpr int kWaves = 16;
constexpr int kThreads = kWaves * 64;
constexpr uint32_t kPastEnd = 0xFFFFFF00u;  // buffer offset that loads zeros
constexpr int kXPitch = 36;                 // floats of x per block in LDS
constexpr int kXEarly = 6;                  // x values a thread requests before the first weights

enum RowsFmt : int { kRows4 = 0, kRows5 = 1, kRows8 = 2 };

template <int QT, bool GGUF, int NI>
struct RowsUnit {
    static constexpr int kQs = QT == kRows8 ? 32 : 16;                         // qs bytes per block
    static constexpr int kBB = kQs + (QT == kRows5 ? 6 : 2);                   // GGUF block bytes
    static constexpr int kPieces = (64 * NI * kBB + 15 + 1023) / 1024;         // 16-byte loads a lane (GGUF)
    static constexpr int kSlot = GGUF ? kPieces * 1024 + 16 : 0;               // LDS of a wave's unit
    static constexpr float kXScale = QT == kRows4 ? 0.0625f : QT == kRows5 ? 0.125f : 1.0f;
    uint4 v[GGUF ? kPieces : NI * kQs / 16];
    uint32_t sc[GGUF ? 1 : NI], qh[!GGUF && QT == kRows5 ? NI : 1];
};

__device__ __forceinline__ uint32_t opaque(uint32_t v) {  // one byte conversion per weight, no bfe first
    asm("" : "+v"(v));
    return v;
}
__device__ __forceinline__ float sbyte(uint32_t v, int k) { return (float)(int)(int8_t)((v >> (8 * k)) & 0xFFu); }

// Bits [4g, 4g + 4) of h at bit 7 of bytes 0..3: with t = those bits at [7, 11),
// t * (1 + 2^7 + 2^14 + 2^21) puts bit j at 8j + 7 without carries.
__device__ __forceinline__ uint32_t spread_bits(uint32_t h, int g) {
    const int s = 4 * g - 7;
    return __umul24((s >= 0 ? h >> s : h << -s) & 0x780u, 0x204081u);
}

// sum_j q[j] xb[j] of one block, q its dwords (Q5: nh the inverted fifth bits)
template <int QT>
__device__ __forceinline__ float block_dot(const uint32_t* q, uint32_t nh, const float* xb) {
    float t0 = 0.f, t1 = 0.f;
    const float4* x4 = reinterpret_cast<const float4*>(xb);
    auto four = [&](uint32_t v, const float4& x, float t) {
        t = fmaf(sbyte(v, 0), x.x, t);
        t = fmaf(sbyte(v, 1), x.y, t);
        t = fmaf(sbyte(v, 2), x.z, t);
        return fmaf(sbyte(v, 3), x.w, t);
    };
    if constexpr (QT == kRows8) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            t0 = four(opaque(q[i]), x4[i], t0);
            t1 = four(opaque(q[4 + i]), x4[4 + i], t1);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t lo, hi;
            if constexpr (QT == kRows4) {
                lo = ((q[i] << 4) ^ 0x80808080u) & 0xF0F0F0F0u;
                hi = (q[i] ^ 0x80808080u) & 0xF0F0F0F0u;
            } else {
                lo = ((q[i] << 3) & 0x78787878u) | (spread_bits(nh, i) & 0x80808080u);
                hi = ((q[i] >> 1) & 0x78787878u) | (spread_bits(nh, 4 + i) & 0x80808080u);
            }
            t0 = four(opaque(lo), x4[i], t0);
            t1 = four(opaque(hi), x4[4 + i], t1);
        }
    }
    return t0 + t1;
}

struct RowsArgs {
    const uint8_t* w;    // GGUF blocks, or the qs plane
    const uint8_t* wh;   // split Q5: qh plane
    const float* wsc;    // split: scales
    const float* x;
    const float* pre_arg;
    float* y;
    int M, K, pre, accumulate, post, rw, chunk, nchunk, splits, hd;
    float eps;
};

template <int QT, bool GGUF, int NI>
__global__ __launch_bounds__(kThreads) void matvec_rows(const RowsArgs a) {
    using U = RowsUnit<QT, GGUF, NI>;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ float red[kWaves], ybuf[2][kWaves * 64];
    const int nb = a.K >> 5, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rw = a.rw, tile_rows = kWaves * rw, nchunk = a.nchunk, G = gridDim.x;
    const int n_tiles = (a.M + tile_rows - 1) / tile_rows;
    const int my_tiles = (n_tiles - (int)blockIdx.x + G - 1) / G, L = my_tiles * nchunk;
    const uint32_t nblocks = (uint32_t)a.M * (uint32_t)nb;
    // whole dwords: an odd number of GGUF blocks ends inside one (of the 4-byte aligned
    // buffer), and a dword that reaches past the descriptor would read as zero
    const auto wr = make_rsrc(a.w, (nblocks * (uint32_t)(GGUF ? U::kBB : U::kQs) + 3u) & ~3u);
    const auto hr = make_rsrc(a.wh, !GGUF && QT == kRows5 ? nblocks * 4u : 0u);
    const auto sr = make_rsrc(a.wsc, GGUF ? 0u : nblocks * 4u);
    float* xs = reinterpret_cast<float*>(lds);
    uint8_t* slot = lds + (size_t)nb * kXPitch * 4 + wave * U::kSlot;
    float* prod = reinterpret_cast<float*>(lds + (size_t)nb * kXPitch * 4 + kWaves * U::kSlot) + wave * 64 * NI;

    // unit s: tile i = s / nchunk, chunk s % nchunk; its first block and number of blocks
    auto unit = [&](int s, uint32_t* b0) {
        const int i = s / nchunk, c = s - i * nchunk;
        const int row0 = ((int)blockIdx.x + G * i) * tile_rows + wave * rw;
        *b0 = (uint32_t)row0 * (uint32_t)nb + (uint32_t)(c * a.chunk);
        const int n = rw > 1 ? min(rw, a.M - row0) * nb : min(a.chunk, nb - c * a.chunk);
        return s < L && row0 < a.M ? n : 0;
    };
    U u;
    auto load = [&](int s) {
        uint32_t b0;
        const int n = unit(s, &b0);
        if constexpr (GGUF) {
            const uint32_t begin = b0 * (uint32_t)U::kBB, end = begin + (uint32_t)(n * U::kBB);
            const uint32_t p0 = (begin & ~15u) + 16u * (uint32_t)lane;
#pragma unroll
            for (int k = 0; k < U::kPieces; ++k) {
                const uint32_t p = p0 + 1024u * k;
                u.v[k] = buf_load_b128(wr, n > 0 && p < end ? p : kPastEnd);
            }
        } else {
#pragma unroll
            for (int k = 0; k < NI; ++k) {
                const int b = lane + 64 * k;
                const uint32_t blk = b0 + (uint32_t)b;
#pragma unroll
                for (int h = 0; h < U::kQs / 16; ++h)
                    u.v[k * (U::kQs / 16) + h] = buf_load_b128(wr, b < n ? blk * (uint32_t)U::kQs + 16u * h : kPastEnd);
                if constexpr (QT == kRows5) u.qh[k] = buf_load_b32(hr, b < n ? blk * 4u : kPastEnd);
                u.sc[k] = buf_load_b32(sr, b < n ? blk * 4u : kPastEnd);
            }
        }
    };

    // 1) x and the pre-op's argument are requested before the weights, and staged once
    // the weights are under way
    const int pre = a.pre;
    float xv[kXEarly], gv[kXEarly];
#pragma unroll
    for (int i = 0; i < kXEarly; ++i) {
        const int e = (int)threadIdx.x + kThreads * i;
        xv[i] = e < a.K ? a.x[e] : 0.f;
        gv[i] = pre != kPreNone && e < a.K ? a.pre_arg[e] : 0.f;
    }
    __builtin_amdgcn_sched_barrier(0);
    load(0);
    __builtin_amdgcn_sched_barrier(0);
    float ss = 0.f;
    auto stage = [&](int e, float x, float g) {
        if (pre == kPreRmsNorm) {
            // y = W (inv (x g)) = inv (W (x g)): the row totals are scaled, so no
            // barrier comes before the staging
            ss = fmaf(x, x, ss);
            x = __fmul_rn(x, g);
        } else if (pre == kPreSwiGlu) {
            x = __fmul_rn(x / (1.0f + expf(-x)), g);
        }
        xs[(e >> 5) * kXPitch + (e & 31)] = x * U::kXScale;
    };
#pragma unroll
    for (int i = 0; i < kXEarly; ++i) {
        const int e = (int)threadIdx.x + kThreads * i;
        if (e < a.K) stage(e, xv[i], gv[i]);
    }
    for (int e = (int)threadIdx.x + kThreads * kXEarly; e < a.K; e += kThreads)
        stage(e, a.x[e], pre != kPreNone ? a.pre_arg[e] : 0.f);
    if (pre == kPreRmsNorm) {
        ss = wave_total_dpp(ss);
        if (lane == 0) red[wave] = ss;
    }
    // rw > 1: the column block of the lane's k-th block, the same in every unit
    int cb[NI];
#pragma unroll
    for (int k = 0; k < NI; ++k) cb[k] = rw > 1 ? (lane + 64 * k) % nb : lane + 64 * k;
    __syncthreads();
    float inv = 1.f;
    if (pre == kPreRmsNorm) {
        float tot = 0.f;
#pragma unroll
        for (int k = 0; k < kWaves; ++k) tot += red[k];
        inv = 1.0f / sqrtf(tot / (float)a.K + a.eps);
    }

    // 2) the stream
    float acc = 0.f;
    for (int s = 0; s < L; ++s) {
        uint32_t b0;
        const int n = unit(s, &b0);
        const int i = s / nchunk, c = s - i * nchunk;
        uint32_t shift = 0;
        U cur;
        if constexpr (GGUF) {
            shift = (b0 * (uint32_t)U::kBB) & 15u;
#pragma unroll
            for (int k = 0; k < U::kPieces; ++k) *reinterpret_cast<uint4*>(slot + 1024 * k + 16 * lane) = u.v[k];
            __builtin_amdgcn_wave_barrier();
        } else {
            cur = u;
        }
        load(s + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < NI; ++k) {
            if (64 * k >= n) break;  // wave-uniform
            const int b = min(lane + 64 * k, n - 1);
            uint32_t q[U::kQs / 4], nh = 0;
            float d;
            if constexpr (GGUF) {
                const uint32_t o = shift + (uint32_t)b * (uint32_t)U::kBB;  // even
                d = __half2float(__ushort_as_half(*reinterpret_cast<const uint16_t*>(slot + o)));
                const uint32_t* p = reinterpret_cast<const uint32_t*>(slot + ((o + 2u) & ~3u));
                const uint32_t sh = (o + 2u) & 3u;
                constexpr int kHead = QT == kRows5 ? 1 : 0;
                uint32_t r[U::kQs / 4 + kHead + 1];
#pragma unroll
                for (int t = 0; t < U::kQs / 4 + kHead + 1; ++t) r[t] = p[t];
                if constexpr (QT == kRows5) nh = ~__builtin_amdgcn_alignbyte(r[1], r[0], sh);
#pragma unroll
                for (int t = 0; t < U::kQs / 4; ++t) q[t] = __builtin_amdgcn_alignbyte(r[t + kHead + 1], r[t + kHead], sh);
            } else {
#pragma unroll
                for (int h = 0; h < U::kQs / 16; ++h) {
                    const uint4 v = cur.v[k * (U::kQs / 16) + h];
                    q[4 * h] = v.x, q[4 * h + 1] = v.y, q[4 * h + 2] = v.z, q[4 * h + 3] = v.w;
                }
                if constexpr (QT == kRows5) nh = ~cur.qh[k];
                d = __uint_as_float(cur.sc[k]);
            }
            const int col = rw > 1 ? cb[k] : c * a.chunk + b;
            const float t = block_dot<QT>(q, nh, xs + col * kXPitch);
            if (rw > 1)
                prod[lane + 64 * k] = d * t;
            else if (lane + 64 * k < n)
                acc = fmaf(d, t, acc);
        }
        if (c < nchunk - 1) continue;
        const int row0 = ((int)blockIdx.x + G * i) * tile_rows + wave * rw;
        float sum;  // rw > 1: lane r holds row r's total; else every lane the row's
        if (rw > 1) {
            __builtin_amdgcn_wave_barrier();
            sum = 0.f;
            if (lane * nb < n)
                for (int j = 0; j < nb; ++j) sum += prod[lane * nb + j];
            __builtin_amdgcn_wave_barrier();
        } else {
            sum = wave_total_dpp(acc);
            acc = 0.f;
        }
        sum = __fmul_rn(sum, inv);
        const int row = row0 + lane;
        if (a.post == kPostNone) {
            if (lane < rw && row < a.M) a.y[row] = a.accumulate ? a.y[row] + sum : sum;
        } else {
            // groups of 8 gate rows and their 8 up rows (tiles are whole groups): the
            // totals meet in LDS, two buffers so that one barrier a tile is enough
            float* yb = ybuf[i & 1];
            if (lane < rw) yb[wave * rw + lane] = sum;
            __syncthreads();
            for (int j = threadIdx.x; j < tile_rows / 2; j += kThreads) {
                const int r = 16 * (j >> 3) + (j & 7), g = ((int)blockIdx.x + G * i) * tile_rows + r;
                if (g < a.M) {
                    const float gs = yb[r], us = yb[r + 8];
                    a.y[8 * (g >> 4) + (j & 7)] = __fmul_rn(gs / (1.0f + expf(-gs)), us);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Small shapes: R whole rows per wave and nothing shared, so a launch is one memory
// round trip, the products and one reduction, without LDS or a barrier (the kernel
// above takes 4.4 us for any of them, an empty launch 1.6).  Four lanes to a block:
// lane item it = (block it / 4, g = it % 4) holds the 8 values of x at positions
// 4g.. and 16 + 4g.. (Q4, Q5: one dword of nibble pairs) or 8g.. (Q8: two dwords), in
// registers for all R rows; NP passes of 64 items cover K.  A wave holds all of x, so
// the RMSNorm's sum of squares is its own too.  kPostSwiGlu8: a wave's rows are gate /
// up pairs, 8 rows apart.
// ---------------------------------------------------------------------------
constexpr int kWaveThreads = 256;

template <typename T>
__device__ __forceinline__ T load_at(const uint8_t* p) {  // any 2-byte aligned address
    T v;
    __builtin_memcpy(&v, p, sizeof(T));
    return v;
}

template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, false);
    return v + __longlong_as_double((long long)hi << 32 | (uint32_t)lo);
}
__device__ __forceinline__ double lane_value(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double((long long)hi << 32 | (uint32_t)lo);
}
__device__ __forceinline__ double wave_total64(double v) {
    v = dpp_add<kDppQuadXor1>(v), v = dpp_add<kDppQuadXor2>(v);
    v = dpp_add<kDppRowHalfMirror>(v), v = dpp_add<kDppRowMirror>(v);
    return ((lane_value(v, 0) + lane_value(v, 16)) + lane_value(v, 32)) + lane_value(v, 48);
}

template <int QT, bool GGUF, int NP, int R, int W>
__global__ __launch_bounds__(kWaveThreads) void matvec_wave(const RowsArgs a) {
    static_assert(W == 1 || W == kWaveThreads / 64, "a wave or the workgroup per row");
    constexpr int kQs = QT == kRows8 ? 32 : 16, kBB = kQs + (QT == kRows5 ? 6 : 2);
    const int nb = a.K >> 5, items = 4 * nb, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int gw = W == 1 ? (int)blockIdx.x * (kWaveThreads / 64) + wave : (int)blockIdx.x;
    const int pre = a.pre;
    auto row_of = [&](int r) {
        if (a.post == kPostNone) return gw * R + r;
        const int j = gw * (R / 2) + (r >> 1);
        return 16 * (j >> 3) + (j & 7) + 8 * (r & 1);
    };
    if (row_of(0) >= a.M) return;
    // x first, then the weights of every row
    float x[NP][8], gn[NP][8];
    bool live[NP];
    int blk[NP], g[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const int it = lane + 64 * (W == 1 ? p : wave * NP + p);
        live[p] = it < items;
        const int ic = live[p] ? it : 0;
        blk[p] = ic >> 2, g[p] = ic & 3;
        const int e0 = 32 * blk[p] + (QT == kRows8 ? 8 : 4) * g[p], e1 = e0 + (QT == kRows8 ? 4 : 16);
        auto get8 = [&](const float* src, float* to) {
            const float4 u = *reinterpret_cast<const float4*>(src + e0), v = *reinterpret_cast<const float4*>(src + e1);
            to[0] = u.x, to[1] = u.y, to[2] = u.z, to[3] = u.w;
            to[4] = v.x, to[5] = v.y, to[6] = v.z, to[7] = v.w;
        };
        if (pre == kPreAttnMerge) {
            // the heads of the two quads (head_dim need not hold a whole block)
            const int stride = kAttnPartStride(a.hd);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int e = q ? e1 : e0, h = e / a.hd;
                const float* ph = a.pre_arg + (size_t)h * a.splits * stride;
                const float* pa = ph + 4 + e - h * a.hd;
                float M = -INFINITY, l = 0.f;
                float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
                for (int i = 0; i < a.splits; ++i) M = fmaxf(M, ph[i * stride]);
                if (M != -INFINITY)
                    for (int i = 0; i < a.splits; ++i) {
                        const float f = exp2_fast(ph[i * stride] - M);
                        const float4 v = *reinterpret_cast<const float4*>(pa + i * stride);
                        l = fmaf(ph[i * stride + 1], f, l);
                        s.x = fmaf(v.x, f, s.x), s.y = fmaf(v.y, f, s.y);
                        s.z = fmaf(v.z, f, s.z), s.w = fmaf(v.w, f, s.w);
                    }
                const bool none = M == -INFINITY;
                x[p][4 * q] = none ? 0.f : s.x / l;
                x[p][4 * q + 1] = none ? 0.f : s.y / l;
                x[p][4 * q + 2] = none ? 0.f : s.z / l;
                x[p][4 * q + 3] = none ? 0.f : s.w / l;
            }
        } else {
            get8(a.x, x[p]);
            if (pre != kPreNone) get8(a.pre_arg, gn[p]);
        }
    }
    uint32_t q[R][NP][kQs / 16], qh[R][QT == kRows5 ? NP : 1], sc[R][NP];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const size_t row = (size_t)min(row_of(r), a.M - 1) * nb;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const size_t b = row + blk[p];
            const uint8_t* qs = GGUF ? a.w + b * kBB + (kBB - kQs) : a.w + b * kQs;
            qs += kQs / 4 * g[p];
            if constexpr (QT == kRows8) {
                const uint2 v = load_at<uint2>(qs);
                q[r][p][0] = v.x, q[r][p][1] = v.y;
            } else {
                q[r][p][0] = load_at<uint32_t>(qs);
            }
            if constexpr (QT == kRows5) qh[r][p] = load_at<uint32_t>(GGUF ? a.w + b * kBB + 2 : a.wh + b * 4);
            if constexpr (GGUF)
                sc[r][p] = load_at<uint16_t>(a.w + b * kBB);
            else
                sc[r][p] = __float_as_uint(a.wsc[b]);
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            float v = x[p][t];
            if (pre == kPreRmsNorm) {  // y = W (inv (x g)) = inv (W (x g))
                ss = live[p] ? fmaf(v, v, ss) : ss;
                v = __fmul_rn(v, gn[p][t]);
            } else if (pre == kPreSwiGlu) {
                v = __fmul_rn(v / (1.0f + expf(-v)), gn[p][t]);
            }
            x[p][t] = v * RowsUnit<QT, GGUF, 1>::kXScale;
        }
    ss = wave_total_dpp(ss);
    float tot[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        // a wave per row (K <= 1024) adds its fours of products in 64 bits: in fp32 throughout
        // the error was 1.5 times the int8-MFMA stream's (15122 x 256 8.4e-8 against 5.6e-8
        // of the result's norm), so it is 4.7e-8, for 0.1 us at 288 x 288 and 0.7 at 32000 x 288
        std::conditional_t<W == 1, double, float> acc = 0;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            uint32_t lo, hi;
            if constexpr (QT == kRows8) {
                lo = q[r][p][0], hi = q[r][p][1];
            } else if constexpr (QT == kRows4) {
                lo = ((q[r][p][0] << 4) ^ 0x80808080u) & 0xF0F0F0F0u;
                hi = (q[r][p][0] ^ 0x80808080u) & 0xF0F0F0F0u;
            } else {
                const uint32_t nh = ~qh[r][p] >> (4 * g[p]);
                lo = ((q[r][p][0] << 3) & 0x78787878u) | (spread_bits(nh, 0) & 0x80808080u);
                hi = ((q[r][p][0] >> 1) & 0x78787878u) | (spread_bits(nh, 4) & 0x80808080u);
            }
            lo = opaque(lo), hi = opaque(hi);
            const float d = GGUF ? half_lo(sc[r][p]) : __uint_as_float(sc[r][p]);
            if constexpr (W == 1) {
                float t0 = 0.f, t1 = 0.f;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    t0 = fmaf(sbyte(lo, k), x[p][k], t0);
                    t1 = fmaf(sbyte(hi, k), x[p][4 + k], t1);
                }
                acc = live[p] ? fma((double)d, (double)t0 + (double)t1, acc) : acc;
            } else {
                float t = 0.f;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    t = fmaf(sbyte(lo, k), x[p][k], t);
                    t = fmaf(sbyte(hi, k), x[p][4 + k], t);
                }
                acc = live[p] ? fmaf(d, t, acc) : acc;
            }
        }
        if constexpr (W == 1)
            tot[r] = (float)wave_total64(acc);
        else
            tot[r] = wave_total_dpp(acc);
    }
    if constexpr (W > 1) {  // the waves' parts of K meet in LDS, added in order
        __shared__ float red[R + 1][W];
        if (lane == 0) {
            red[R][wave] = ss;
#pragma unroll
            for (int r = 0; r < R; ++r) red[r][wave] = tot[r];
        }
        __syncthreads();
        if (wave != 0) return;
        ss = 0.f;
#pragma unroll
        for (int k = 0; k < W; ++k) ss += red[R][k];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            tot[r] = 0.f;
#pragma unroll
            for (int k = 0; k < W; ++k) tot[r] += red[r][k];
        }
    }
    if (pre == kPreRmsNorm) {
        const float inv = 1.0f / sqrtf(ss / (float)a.K + a.eps);
#pragma unroll
        for (int r = 0; r < R; ++r) tot[r] = __fmul_rn(tot[r], inv);
    }
    if (lane == 0) {
        if (a.post == kPostNone) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int row = gw * R + r;
                if (row < a.M) a.y[row] = a.accumulate ? a.y[row] + tot[r] : tot[r];
            }
        } else {
#pragma unroll
            for (int r = 0; r + 1 < R; r += 2) {
                const int j = gw * (R / 2) + (r >> 1);
                if (2 * j < a.M) a.y[j] = __fmul_rn(tot[r] / (1.0f + expf(-tot[r])), tot[r + 1]);
            }
        }
    }
}

constexpr size_t kLdsBudget = 160 * 1024 - 12 * 1024;  // the static reduction buffers beside it

int row_units() {  // compute units of the current device
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
        (void)hipGetLastError();
        return 256;
    }
    return n;
}

template <int QT, bool GGUF, int NI>
size_t rows_lds(int nb, int rw) {
    return (size_t)nb * kXPitch * 4 + (size_t)kWaves * RowsUnit<QT, GGUF, NI>::kSlot +
           (rw > 1 ? (size_t)kWaves * 64 * NI * 4 : 0);
}

// Rows per wave: as many tiles as compute units while a unit holds the rows.
int rows_per_wave(int64_t M, int nb, int cus, int most) {
    const int64_t want = (M + (int64_t)kWaves * cus - 1) / ((int64_t)kWaves * cus);
    return (int)std::max<int64_t>(1, std::min<int64_t>({want, most / nb, 64}));
}

template <int QT, bool GGUF, int NI>
int rows_launch_ni(RowsArgs a, hipStream_t st) {
    const int nb = a.K / 32, cus = row_units();
    a.rw = rows_per_wave(a.M, nb, cus, 64 * NI);
    a.nchunk = a.rw > 1 ? 1 : (nb + 64 * NI - 1) / (64 * NI);
    a.chunk = (nb + a.nchunk - 1) / a.nchunk;
    const size_t lds = rows_lds<QT, GGUF, NI>(nb, a.rw);
    const int rc = dynamic_lds((const void*)matvec_rows<QT, GGUF, NI>, lds);
    if (rc) return rc;
    const int tiles = (int)(((int64_t)a.M + kWaves * a.rw - 1) / (kWaves * a.rw));
    hipLaunchKernelGGL((matvec_rows<QT, GGUF, NI>), dim3((unsigned)std::min(tiles, cus)), dim3(kThreads), lds, st, a);
    ASMHIP_TRY(hipGetLastError());
    return kOk;
}

// Three blocks a lane where the unit's LDS fits beside x, else one.
template <int QT, bool GGUF>
int rows_launch_fmt(const RowsArgs& a, hipStream_t st) {
    const int nb = a.K / 32;
    return rows_lds<QT, GGUF, 3>(nb, 2) <= kLdsBudget ? rows_launch_ni<QT, GGUF, 3>(a, st)
                                                      : rows_launch_ni<QT, GGUF, 1>(a, st);
}

template <int QT, bool GGUF, int NP, int R, int W>
int wave_launch(const RowsArgs& a, hipStream_t st) {
    const int64_t groups = ((int64_t)a.M + R - 1) / R, per = W == 1 ? kWaveThreads / 64 : 1;
    hipLaunchKernelGGL((matvec_wave<QT, GGUF, NP, R, W>), dim3((unsigned)((groups + per - 1) / per)),
                       dim3(kWaveThreads), 0, st, a);
    ASMHIP_TRY(hipGetLastError());
    return kOk;
}

template <int QT, bool GGUF, int NP, int W>
int wave_launch_r(const RowsArgs& a, int r, hipStream_t st) {
    if (r >= 4) return wave_launch<QT, GGUF, NP, 4, W>(a, st);
    if (r >= 2) return wave_launch<QT, GGUF, NP, 2, W>(a, st);
    return wave_launch<QT, GGUF, NP, 1, W>(a, st);
}

// Rows per wave (or per workgroup at W = 4): fewer while there are too few rows to
// fill the chip, more once x's registers and reduction are what a row costs (Q4_0,
// 1 / 2 / 4 rows: 864 x 288 2.0 / 2.1 / 2.5 us, 2000 x 4064 4.04 / 3.82 / 3.98, 4096 x
// 4064 6.6 / 5.8 / 5.5, 32000 x 288 6.6 / 4.9 / 4.4).
template <int QT, bool GGUF>
int wave_launch_fmt(const RowsArgs& a, hipStream_t st) {
    const int np = (a.K / 8 + 63) / 64;
    const int64_t weights = (int64_t)a.M * a.K;
    int r = a.M <= 512 || (a.M <= 2048 && a.K <= 1024) ? 1 : weights <= (int64_t)8 << 20 && a.M <= 8192 ? 2 : 4;
    if (a.post != kPostNone) r = std::max(r, 2);
    if (np <= 1) return wave_launch_r<QT, GGUF, 1, 1>(a, r, st);
    if (np <= 2) return wave_launch_r<QT, GGUF, 2, 1>(a, r, st);
    // four waves share a row's columns: a wave holds at most 4 passes of x
    if (np <= 4) return wave_launch_r<QT, GGUF, 1, 4>(a, r, st);
    if (np <= 8) return wave_launch_r<QT, GGUF, 2, 4>(a, r, st);
    if (np <= 12) return wave_launch_r<QT, GGUF, 3, 4>(a, r, st);
    return wave_launch_r<QT, GGUF, 4, 4>(a, r, st);
}

// matvec_wave up to 24 M weights (4096 x 5504 Q4_0 6.9 us against 7.7 of matvec_rows,
// 11008 x 2080 9.3 / 10.8, 1000 x 5504 Q8_0 3.8 / 6.7), where a row's columns fit its
// registers (K <= 8192); matvec_rows above (33000 x 4128 Q4_0 31 / 29 us, 4096 x 8032
// Q8_0 11.5 / 10.3), and for many short rows past 512 columns (33000 x 544 8.0 / 6.9;
// 32000 x 288 4.4 / 5.7).
template <int QT, bool GGUF>
int rows_or_wave(const RowsArgs& a, hipStream_t st) {
    const bool aligned = ((uintptr_t)a.x | (uintptr_t)(a.pre != kPreNone ? a.pre_arg : nullptr)) % 16 == 0;
    const int64_t weights = (int64_t)a.M * a.K;
    if (a.pre == kPreAttnMerge ||
        (aligned && a.K <= 8192 && (a.K <= 512 || (a.M <= 16384 && weights <= (int64_t)24 << 20))))
        return wave_launch_fmt<QT, GGUF>(a, st);
    return rows_launch_fmt<QT, GGUF>(a, st);
}

}  // namespace

bool matvec_rows_takes(int bits, bool gguf, const void* w, const void* qh, const float* scales, const float* x,
                       int64_t M, int64_t K, const MatvecOpts& o) {
    const int64_t nb = K / 32, bytes = M * nb * (bits == 8 ? 34 : bits == 5 ? 22 : 18);
    const int slot = bits == 8 ? RowsUnit<kRows8, true, 1>::kSlot
                               : bits == 5 ? RowsUnit<kRows5, true, 1>::kSlot : RowsUnit<kRows4, true, 1>::kSlot;
    const size_t lds = (size_t)nb * kXPitch * 4 + (size_t)kWaves * (slot + 64 * 4);
    // the merge runs in every wave that reads x: small K only, and the head_dims of the merge launch
    if (o.pre == kPreAttnMerge &&
        (!rows_before_stream(M, K) || o.attn_splits < 1 || o.attn_splits > kAttnMergeMaxSplits ||
         !attn_head_dim(o.attn_hd) || K % o.attn_hd || (uintptr_t)o.pre_arg % 16))
        return false;
    return K > 0 && K % 32 == 0 && M > 0 && M <= INT32_MAX - 4096 && bytes < (int64_t)kPastEnd && lds <= kLdsBudget &&
           (uintptr_t)w % 4 == 0 && (gguf || ((uintptr_t)scales % 4 == 0 && (uintptr_t)qh % 4 == 0)) &&
           (uintptr_t)x % 4 == 0 && (o.post == kPostNone || (M % 16 == 0 && !o.accumulate));
}

int matvec_rows_launch(int bits, bool gguf, const void* w, const uint8_t* qh, const float* scales, const float* x,
                       float* y, int64_t M, int64_t K, hipStream_t st, const MatvecOpts& o) {
    RowsArgs a{static_cast<const uint8_t*>(w), qh, scales, x, o.pre_arg, y, (int)M, (int)K, o.pre, (int)o.accumulate,
               o.post, 1, 0, 1, o.attn_splits, o.attn_hd, o.eps};
    switch (bits) {
        case 4: return gguf ? rows_or_wave<kRows4, true>(a, st) : rows_or_wave<kRows4, false>(a, st);
        case 5: return gguf ? rows_or_wave<kRows5, true>(a, st) : rows_or_wave<kRows5, false>(a, st);
        case 8: return gguf ? rows_or_wave<kRows8, true>(a, st) : rows_or_wave<kRows8, false>(a, st);
        default: return fail(kInvalidArgument, "matvec rows: %d-bit weights", bits);
    }
}

}  // namespace asmhip
