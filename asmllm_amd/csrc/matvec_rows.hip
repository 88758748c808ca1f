// Quantized matvec over whole rows in fp32 (VALU), for the shapes the int8-MFMA
// stream does not take: any K % 32 == 0, GGUF blocks or split planes, and the work
// the decode step fuses around its matvecs.
//
// y[m] = sum_b d[m,b] * sum_j (q[m,b,j] - z) * x[32b + j], the arithmetic of the
// reference's asm_matmul_q4 / _q5 / _q8 (src/kernels/x86_64/matmul_q4_avx2.asm:57-287,
// matmul_q5_avx2.asm:52-238, matmul_q8_avx2.asm:51-194).
//
// Two kernels, and one order of the sums, so that a row's bits do not depend on which of
// them a matrix's size picks (a weight cut by rows gives the rows of the whole).  An item
// is the 8 columns 4g..4g+3 and 16+4g..16+4g+3 of a block (Q8: 8g..8g+7), g = 0..3, and t
// its products with x added by fused multiply-adds:
//   K <= 1024  t in two halves, d (t0 + t1) in 64 bits; the four items of a block as
//              (v0 + v1) + (v2 + v3); blocks j and j + 16; the 16 j in fours as (e0 + e2) +
//              (e1 + e3); the fours as (h0 + h1) + (h2 + h3), all in 64 bits;
//   above      for each of 64 columns of blocks 64 p + l one chain of fused d t over p for
//              every item; the four items, then 16 l as above, in fp32, and the four
//              sixteens in order.
//
// matvec_rows.  A unit is one wave's contiguous run of blocks: `rw` whole rows, or a
// row's chunk of 64 NI blocks.  Its
// bytes are requested as consecutive 16-byte pieces (split planes: each lane its own
// block), parked in the wave's own piece of LDS, and read back one block a lane: a
// lane's block is 18, 22 or 34 bytes at a 2-byte address, and loads of those strides
// touch three lines per four lanes.  The next unit is requested as soon as the
// registers are parked, so a wave always has one unit in flight; waves wait for no
// one but at the start, for x.  x is staged once per workgroup (36 floats per block:
// the 16-byte reads of eight consecutive blocks fall on distinct banks), and the
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

constexpr uint32_t kPastEnd = 0xFFFFFF00u;  // buffer offset that loads zeros
constexpr int kXPitch = 36;                 // floats of x per block in LDS
constexpr int kXEarly = 6;                  // x values a thread requests before the first weights
constexpr int kWaves = 16;                  // of a matvec_rows workgroup
constexpr int kShortK = 1024, kWaveK = 8192;  // 64-bit sums up to, matvec_wave up to

enum RowsFmt : int { kRows4 = 0, kRows5 = 1, kRows8 = 2 };

// What a unit of matvec_rows holds: kPack64 (K <= 1024) and kPack32 (K <= 2048) the blocks
// of up to 16 rows, one after another on the lanes, so that no pass is half empty; 1 and 2
// so many blocks a lane of one row, a chunk of it.
enum RowsMode : int { kPack64 = 0, kPack32 = 3 };
template <int MODE>
struct RowsShape {
    static constexpr bool kPacked = MODE == kPack64 || MODE == kPack32;
    static constexpr int NI = kPacked ? 3 : MODE;
    static constexpr int kMaxRows = kPacked ? 16 : 1;
    // passes of RMSNorm's squares: as matvec_wave's, at most four (above kWaveK by threads)
    static constexpr int kSq = MODE == kPack64 ? 2 : MODE == kPack32 ? 1 : 4;
    using Sum = std::conditional_t<MODE == kPack64, double, float>;  // of a packed block's products
};

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

// An item's two groups of four weights as signed bytes, from its dwords of a block (Q4,
// Q5: one; Q8: two; nh: the inverted fifth bits, the item's from 4 g on)
template <int QT>
__device__ __forceinline__ void item_bytes(uint32_t q0, uint32_t q1, uint32_t nh, int g, uint32_t* lo, uint32_t* hi) {
    if constexpr (QT == kRows8) {
        *lo = q0, *hi = q1;
    } else if constexpr (QT == kRows4) {
        *lo = ((q0 << 4) ^ 0x80808080u) & 0xF0F0F0F0u;
        *hi = (q0 ^ 0x80808080u) & 0xF0F0F0F0u;
    } else {
        *lo = ((q0 << 3) & 0x78787878u) | (spread_bits(nh, g) & 0x80808080u);
        *hi = ((q0 >> 1) & 0x78787878u) | (spread_bits(nh, 4 + g) & 0x80808080u);
    }
    *lo = opaque(*lo), *hi = opaque(*hi);
}

// An item's sum of a short row: d (t0 + t1), rounded once to 64 bits
__device__ __forceinline__ double item_short(uint32_t lo, uint32_t hi, const float* xl, const float* xh, float d) {
#pragma clang fp contract(off)
    float t0 = 0.f, t1 = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        t0 = fmaf(sbyte(lo, k), xl[k], t0);
        t1 = fmaf(sbyte(hi, k), xh[k], t1);
    }
    return (double)d * ((double)t0 + (double)t1);
}
__device__ __forceinline__ float item_long(uint32_t lo, uint32_t hi, const float* xl, const float* xh) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        t = fmaf(sbyte(lo, k), xl[k], t);
        t = fmaf(sbyte(hi, k), xh[k], t);
    }
    return t;
}

// Item g of the block whose dwords are q
template <int QT>
__device__ __forceinline__ void item_of(const uint32_t* q, uint32_t nh, const float* xb, int g, uint32_t* lo,
                                        uint32_t* hi, const float** xl, const float** xh) {
    constexpr bool k8 = QT == kRows8;
    item_bytes<QT>(q[k8 ? 2 * g : g], k8 ? q[2 * g + 1] : 0u, nh, g, lo, hi);
    *xl = xb + (k8 ? 8 * g : 4 * g), *xh = xb + (k8 ? 8 * g + 4 : 16 + 4 * g);
}

// A row's total times RMSNorm's factor, rounded in both kernels: never part of an fma with y
__device__ __forceinline__ float scaled_total(float tot, float inv) {
#pragma clang fp contract(off)
    return tot * inv;
}

// Sum over the squares of x (RMSNorm) in the order of the items: one wave's NP passes from
// item `first` on
template <int QT, int NP>
__device__ __forceinline__ float item_squares(const float (*x)[8], const bool* live) {
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int t = 0; t < 8; ++t) ss = live[p] ? fmaf(x[p][t], x[p][t], ss) : ss;
    return wave_total_dpp(ss);
}

template <typename T>
__device__ __forceinline__ T load_at(const void* p) {  // any 2-byte aligned address
    T v;
    __builtin_memcpy(&v, p, sizeof(T));
    return v;
}

// The 8 values of item `it` (of a vector of K floats, 4-byte aligned)
template <int QT>
__device__ __forceinline__ void item_load(const float* src, int it, float* to) {
    const int b = it >> 2, g = it & 3;
    const int e0 = 32 * b + (QT == kRows8 ? 8 : 4) * g, e1 = e0 + (QT == kRows8 ? 4 : 16);
    const float4 u = load_at<float4>(src + e0), v = load_at<float4>(src + e1);
    to[0] = u.x, to[1] = u.y, to[2] = u.z, to[3] = u.w;
    to[4] = v.x, to[5] = v.y, to[6] = v.z, to[7] = v.w;
}

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, false);
    return __longlong_as_double((long long)hi << 32 | (uint32_t)lo);
}
constexpr int kDppRor4 = 0x124, kDppRor8 = 0x128;  // 16-lane rows rotated

// v of the even and of the odd 16-lane row of each half-wave, and of the halves
__device__ __forceinline__ void row_pair(float v, float* even, float* odd) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    *even = __uint_as_float(r[0]), *odd = __uint_as_float(r[1]);
}
__device__ __forceinline__ void half_pair(float v, float* low, float* high) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    *low = __uint_as_float(r[0]), *high = __uint_as_float(r[1]);
}
__device__ __forceinline__ void row_pair(double v, double* even, double* odd) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const auto l = __builtin_amdgcn_permlane16_swap((uint32_t)b, (uint32_t)b, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap((uint32_t)(b >> 32), (uint32_t)(b >> 32), false, false);
    *even = __longlong_as_double((long long)((uint64_t)h[0] << 32 | l[0]));
    *odd = __longlong_as_double((long long)((uint64_t)h[1] << 32 | l[1]));
}
__device__ __forceinline__ void half_pair(double v, double* low, double* high) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const auto l = __builtin_amdgcn_permlane32_swap((uint32_t)b, (uint32_t)b, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap((uint32_t)(b >> 32), (uint32_t)(b >> 32), false, false);
    *low = __longlong_as_double((long long)((uint64_t)h[0] << 32 | l[0]));
    *high = __longlong_as_double((long long)((uint64_t)h[1] << 32 | l[1]));
}

// The quads' sums (v0 + v1) + (v2 + v3) of R rows at once: lane l's result is row l % R's.
// The rows are dealt to the lanes as the sums halve, so that R of them take little more
// than one (one after another, with a readlane from each 16 lanes, the sums were a third of
// a short row's instructions).
template <int R, typename T>
__device__ __forceinline__ T quad_sums(const T (&v)[R], int lane) {
    T t[R > 1 ? R / 2 : 1];
    if constexpr (R == 1) {
        t[0] = v[0] + dpp<kDppQuadXor1>(v[0]);
    } else {
#pragma unroll
        for (int i = 0; i < R / 2; ++i) {
            const T keep = lane & 1 ? v[2 * i + 1] : v[2 * i], send = lane & 1 ? v[2 * i] : v[2 * i + 1];
            t[i] = keep + dpp<kDppQuadXor1>(send);
        }
    }
    if constexpr (R < 4) {
        return t[0] + dpp<kDppQuadXor2>(t[0]);
    } else {
        const T keep = lane & 2 ? t[1] : t[0], send = lane & 2 ? t[0] : t[1];
        return keep + dpp<kDppQuadXor2>(send);
    }
}
// The sum over the quads of a wave, lane by lane of a quad: of each 16 lanes as (q0 + q2) +
// (q1 + q3), of these as (h0 + h1) + (h2 + h3)
template <typename T>
__device__ __forceinline__ T over_quads(T q) {
    T a, b;
    q += dpp<kDppRor8>(q);
    q += dpp<kDppRor4>(q);
    row_pair(q, &a, &b);
    half_pair(a + b, &a, &b);
    return a + b;
}

struct RowsArgs {
    const uint8_t* w;    // GGUF blocks, or the qs plane
    const uint8_t* wh;   // split Q5: qh plane
    const float* wsc;    // split: scales
    const float* x;
    const float* pre_arg;
    float* y;
    int M, K, pre, accumulate, post, rw, nchunk, splits, hd;
    float eps;
};

template <int QT, bool GGUF, int MODE>
__global__ __launch_bounds__(kWaves * 64) void matvec_rows(const RowsArgs a) {
    using S = RowsShape<MODE>;
    constexpr int NI = S::NI, kThreads = kWaves * 64;
    using U = RowsUnit<QT, GGUF, NI>;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ float red[kWaves], ybuf[2][kWaves * S::kMaxRows];
    const int nb = a.K >> 5, lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rw = a.rw, tile_rows = kWaves * rw, nchunk = S::kPacked ? 1 : a.nchunk, G = gridDim.x;
    const uint32_t nblocks = (uint32_t)a.M * (uint32_t)nb;
    // whole dwords: an odd number of GGUF blocks ends inside one (of the 4-byte aligned
    // buffer), and a dword that reaches past the descriptor would read as zero
    const auto wr = make_rsrc(a.w, (nblocks * (uint32_t)(GGUF ? U::kBB : U::kQs) + 3u) & ~3u);
    const auto hr = make_rsrc(a.wh, !GGUF && QT == kRows5 ? nblocks * 4u : 0u);
    const auto sr = make_rsrc(a.wsc, GGUF ? 0u : nblocks * 4u);
    float* xs = reinterpret_cast<float*>(lds);
    uint8_t* slot = lds + (size_t)nb * kXPitch * 4 + wave * U::kSlot;
    typename S::Sum* prod = reinterpret_cast<typename S::Sum*>(lds + (size_t)nb * kXPitch * 4 + kWaves * U::kSlot) + wave * 64 * NI;

    // chunk c of a tile from row `row` on: this wave's first block and number of blocks
    auto unit = [&](int row, int c, uint32_t* b0) {
        const int row0 = row + wave * rw;
        *b0 = (uint32_t)row0 * (uint32_t)nb + (uint32_t)(c * 64 * NI);
        const int n = S::kPacked ? min(rw, a.M - row0) * nb : min(64 * NI, nb - c * 64 * NI);
        return row0 < a.M ? n : 0;
    };
    U u;
    auto load = [&](int row, int c) {
        uint32_t b0;
        const int n = unit(row, c, &b0);
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
    // RMSNorm's sum of squares as matvec_wave forms it, by as many waves as share a row there
    const bool by_items = a.K <= kWaveK;
    const int sq_waves = MODE == kPack64 ? 1 : 4;
    float xq[S::kSq][8];
    bool live[S::kSq];
    if (pre == kPreRmsNorm && by_items && wave < sq_waves) {
#pragma unroll
        for (int p = 0; p < S::kSq; ++p) {
            const int it = lane + 64 * (sq_waves * p + wave);
            live[p] = it < 4 * nb;
            item_load<QT>(a.x, live[p] ? it : 0, xq[p]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    load((int)blockIdx.x * tile_rows, 0);
    __builtin_amdgcn_sched_barrier(0);
    float ss = 0.f;
    auto stage = [&](int e, float x, float g) {
        if (pre == kPreRmsNorm) {
            // y = W (inv (x g)) = inv (W (x g)): the row totals are scaled, so no
            // barrier comes before the staging
            if (!by_items) ss = fmaf(x, x, ss);
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
        if (!by_items)
            ss = wave_total_dpp(ss);
        else if (wave < sq_waves)
            ss = item_squares<QT, S::kSq>(xq, live);
        if (lane == 0) red[wave] = ss;
    }
    // packed: the column block of the lane's k-th block, the same in every unit
    int cb[S::kPacked ? NI : 1];
    if constexpr (S::kPacked) {
#pragma unroll
        for (int k = 0; k < NI; ++k) cb[k] = (lane + 64 * k) % nb;
    }
    __syncthreads();
    float inv = 1.f;
    if (pre == kPreRmsNorm) {
        float tot = 0.f;
#pragma unroll
        for (int k = 0; k < kWaves; ++k)
            if (k < (by_items ? sq_waves : kWaves)) tot += red[k];
        inv = 1.0f / sqrtf(tot / (float)a.K + a.eps);
    }

    // 2) the stream
    float part[4] = {0.f, 0.f, 0.f, 0.f};  // the lane's chain of each item
    for (int tile_row = (int)blockIdx.x * tile_rows, c = 0, buf = 0; tile_row < a.M;) {
        uint32_t b0;
        const int n = unit(tile_row, c, &b0), next = tile_row + G * tile_rows;
        uint32_t shift = 0;
        U cur;
        if constexpr (GGUF) {
            shift = (b0 * (uint32_t)U::kBB) & 15u;
#pragma unroll
            for (int k = 0; k < U::kPieces; ++k) *reinterpret_cast<uint4*>(slot + 1024 * k + 16 * lane) = u.v[k];
            wave_lds_order();
        } else {
            cur = u;
        }
        if (c < nchunk - 1)
            load(tile_row, c + 1);
        else
            load(next, 0);
        __builtin_amdgcn_sched_barrier(0);
        // the block at place b of the unit, the lane's k-th
        auto block = [&](int k, int b, uint32_t* q, uint32_t* nh, float* d) {
            if constexpr (GGUF) {
                const uint32_t o = shift + (uint32_t)b * (uint32_t)U::kBB;  // even
                *d = __half2float(__ushort_as_half(*reinterpret_cast<const uint16_t*>(slot + o)));
                const uint32_t* p = reinterpret_cast<const uint32_t*>(slot + ((o + 2u) & ~3u));
                const uint32_t sh = (o + 2u) & 3u;
                constexpr int kHead = QT == kRows5 ? 1 : 0;
                uint32_t r[U::kQs / 4 + kHead + 1];
#pragma unroll
                for (int t = 0; t < U::kQs / 4 + kHead + 1; ++t) r[t] = p[t];
                if constexpr (QT == kRows5) *nh = ~__builtin_amdgcn_alignbyte(r[1], r[0], sh);
#pragma unroll
                for (int t = 0; t < U::kQs / 4; ++t) q[t] = __builtin_amdgcn_alignbyte(r[t + kHead + 1], r[t + kHead], sh);
            } else {
#pragma unroll
                for (int h = 0; h < U::kQs / 16; ++h) {
                    const uint4 v = cur.v[k * (U::kQs / 16) + h];
                    q[4 * h] = v.x, q[4 * h + 1] = v.y, q[4 * h + 2] = v.z, q[4 * h + 3] = v.w;
                }
                if constexpr (QT == kRows5) *nh = ~cur.qh[k];
                *d = __uint_as_float(cur.sc[k]);
            }
        };
        float sum = 0.f;  // the total of row row0 + r of lanes where `owner`
        int r = lane;
        bool owner = lane < rw;
        if constexpr (S::kPacked) {
#pragma clang fp contract(off)
#pragma unroll
            for (int k = 0; k < NI; ++k) {
                if (64 * k >= n) break;  // wave-uniform
                uint32_t q[U::kQs / 4], nh = 0, lo, hi;
                float d;
                block(k, min(lane + 64 * k, n - 1), q, &nh, &d);
                typename S::Sum v[4];
                const float *xl, *xh;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    item_of<QT>(q, nh, xs + cb[k] * kXPitch, g, &lo, &hi, &xl, &xh);
                    if constexpr (MODE == kPack64)
                        v[g] = item_short(lo, hi, xl, xh, d);
                    else
                        v[g] = fmaf(d, item_long(lo, hi, xl, xh), 0.f);
                }
                prod[lane + 64 * k] = (v[0] + v[1]) + (v[2] + v[3]);
            }
            wave_lds_order();
            // four lanes a row
            r = lane >> 2;
            const int part4 = lane & 3;
            owner = part4 == 0 && r < rw;
            const typename S::Sum* row = prod + r * nb;
            if constexpr (MODE == kPack64) {  // four j each
                const int j0 = 4 * part4;
                double e[4] = {};
                if (r * nb < n) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) e[j] = row[j0 + j] + (j0 + 16 + j < nb ? row[j0 + 16 + j] : 0.0);
                }
                double h = (e[0] + e[2]) + (e[1] + e[3]);
                h += dpp<kDppQuadXor1>(h);
                h += dpp<kDppQuadXor2>(h);
                sum = (float)h;
            } else {  // a sixteen each
                float h[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float e[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int l = 16 * part4 + 4 * i + j;
                        e[j] = r * nb < n && l < nb ? row[l] : 0.f;
                    }
                    h[i] = (e[0] + e[2]) + (e[1] + e[3]);
                }
                const float t = (h[0] + h[1]) + (h[2] + h[3]);
                sum = (((0.f + dpp<0x00>(t)) + dpp<0x55>(t)) + dpp<0xAA>(t)) + dpp<0xFF>(t);  // lanes 0..3 of the quad
            }
        } else {
#pragma unroll
            for (int k = 0; k < NI; ++k) {
                const int b = lane + 64 * k;
                if (b < n) {
                    uint32_t q[U::kQs / 4], nh = 0, lo, hi;
                    float d;
                    block(k, b, q, &nh, &d);
                    const float *xl, *xh;
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        item_of<QT>(q, nh, xs + (c * 64 * NI + b) * kXPitch, g, &lo, &hi, &xl, &xh);
                        part[g] = fmaf(d, item_long(lo, hi, xl, xh), part[g]);
                    }
                }
            }
            if (c == nchunk - 1) {
                float h = (part[0] + part[1]) + (part[2] + part[3]);
                h += dpp<kDppQuadXor2>(h);
                h += dpp<kDppQuadXor1>(h);
                h += dpp<kDppRowHalfMirror>(h);
                h += dpp<kDppRowMirror>(h);
                const int v = __float_as_int(h);
#pragma unroll
                for (int w = 0; w < 4; ++w) sum += __int_as_float(__builtin_amdgcn_readlane(v, 16 * w));
                part[0] = part[1] = part[2] = part[3] = 0.f;
            }
        }
        wave_lds_order();  // the next unit's bytes (and products) take the place of this one's
        if (c < nchunk - 1) {
            ++c;
            continue;
        }
        sum = scaled_total(sum, inv);
        const int row = tile_row + wave * rw + r;
        if (a.post == kPostNone) {
            if (owner && row < a.M) a.y[row] = a.accumulate ? a.y[row] + sum : sum;
        } else {
            // groups of 8 gate rows and their 8 up rows (tiles are whole groups): the
            // totals meet in LDS, two buffers so that one barrier a tile is enough
            float* yb = ybuf[buf];
            if (owner) yb[wave * rw + r] = sum;
            __syncthreads();
            for (int j = threadIdx.x; j < tile_rows / 2; j += kThreads) {
                const int r = 16 * (j >> 3) + (j & 7), g = tile_row + r;
                if (g < a.M) {
                    const float gs = yb[r], us = yb[r + 8];
                    a.y[8 * (g >> 4) + (j & 7)] = __fmul_rn(gs / (1.0f + expf(-gs)), us);
                }
            }
        }
        tile_row = next, c = 0, buf ^= 1;
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
        const int it = lane + 64 * (W * p + (W == 1 ? 0 : wave));
        live[p] = it < items;
        const int ic = live[p] ? it : 0;
        blk[p] = ic >> 2, g[p] = ic & 3;
        const int e0 = 32 * blk[p] + (QT == kRows8 ? 8 : 4) * g[p], e1 = e0 + (QT == kRows8 ? 4 : 16);
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
            item_load<QT>(a.x, ic, x[p]);
            if (pre != kPreNone) item_load<QT>(a.pre_arg, ic, gn[p]);
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
    // one branch for all of x: a pre-op looked at element by element was a branch for each
    float ss = 0.f;
    auto each = [&](auto f) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int t = 0; t < 8; ++t) x[p][t] = f(x[p][t], gn[p][t]);
    };
    if (pre == kPreRmsNorm) {  // y = W (inv (x g)) = inv (W (x g))
        ss = item_squares<QT, NP>(x, live);
        each([](float v, float g) { return __fmul_rn(v, g); });
    } else if (pre == kPreSwiGlu) {
        each([](float v, float g) { return __fmul_rn(v / (1.0f + expf(-v)), g); });
    }
    each([](float v, float) { return v * RowsUnit<QT, GGUF, 1>::kXScale; });
    // lane l: the total of row l % R.  A wave per row (K <= 1024) adds in 64 bits: in fp32
    // throughout the error was 1.5 times the int8-MFMA stream's (15122 x 256 8.4e-8 against
    // 5.6e-8 of the result's norm), so it is 4.7e-8
    float tot;
    auto bytes = [&](int r, int p, uint32_t* lo, uint32_t* hi) {
        item_bytes<QT>(q[r][p][0], q[r][p][kQs / 16 - 1], QT == kRows5 ? ~qh[r][QT == kRows5 ? p : 0] >> (4 * g[p]) : 0u, 0,
                       lo, hi);
        return GGUF ? half_lo(sc[r][p]) : __uint_as_float(sc[r][p]);
    };
    if constexpr (W == 1) {
        double sum = 0.0;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
#pragma clang fp contract(off)
            double v[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                uint32_t lo, hi;
                const float d = bytes(r, p, &lo, &hi);
                v[r] = item_short(lo, hi, x[p], x[p] + 4, d);
                v[r] = live[p] ? v[r] : 0.0;
            }
            const double s = quad_sums(v, lane);
            sum = p == 0 ? s : sum + s;
        }
        tot = (float)over_quads(sum);
    } else {
        __shared__ float red[R + 1][W];  // the waves' parts of K, added in order
        float acc[R] = {};
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            if (64 * (W * p + wave) >= items) break;  // wave-uniform
#pragma unroll
            for (int r = 0; r < R; ++r) {
                uint32_t lo, hi;
                const float d = bytes(r, p, &lo, &hi), v = fmaf(d, item_long(lo, hi, x[p], x[p] + 4), acc[r]);
                acc[r] = live[p] ? v : acc[r];
            }
        }
        tot = over_quads(quad_sums(acc, lane));
        if (lane < R) red[lane][wave] = tot;
        if (lane == 0) red[R][wave] = ss;
        __syncthreads();
        if (wave != 0) return;
        ss = 0.f, tot = 0.f;
#pragma unroll
        for (int k = 0; k < W; ++k) ss += red[R][k], tot += red[lane % R][k];
    }
    if (pre == kPreRmsNorm) tot = scaled_total(tot, 1.0f / sqrtf(ss / (float)a.K + a.eps));
    if (a.post == kPostNone) {
        const int row = gw * R + lane;
        if (lane < R && row < a.M) a.y[row] = a.accumulate ? a.y[row] + tot : tot;
    } else {
        const float up = dpp<kDppQuadXor1>(tot);  // lanes 0 and 2: a gate row's total, its up row's beside it
        const int j = gw * (R / 2) + (lane >> 1);
        if (lane < R && !(lane & 1) && 2 * j < a.M) a.y[j] = __fmul_rn(tot / (1.0f + expf(-tot)), up);
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

template <int QT, bool GGUF, int MODE>
size_t rows_lds(int nb) {
    constexpr int NI = RowsShape<MODE>::NI;
    return (size_t)nb * kXPitch * 4 + (size_t)kWaves * RowsUnit<QT, GGUF, NI>::kSlot +
           (RowsShape<MODE>::kPacked ? (size_t)kWaves * 64 * NI * sizeof(typename RowsShape<MODE>::Sum) : 0);
}

template <int QT, bool GGUF, int MODE>
int rows_launch_mode(RowsArgs a, hipStream_t st) {
    using S = RowsShape<MODE>;
    const int nb = a.K / 32, cus = row_units();
    // rows a wave: what gives the busiest compute unit's waves the fewest passes, with one
    // more for a unit's loads and sums (26000 x 1024 12.8 us with the fewest rows, one a unit)
    auto tiles = [&](int rw) { return ((int64_t)a.M + kWaves * rw - 1) / (kWaves * rw); };
    auto cost = [&](int rw) {
        return (tiles(rw) + cus - 1) / cus * ((rw * nb + 63) / 64 + 1);
    };
    a.rw = S::kPacked ? std::min(S::kMaxRows, 64 * S::NI / nb) : 1;
    for (int rw = a.rw - 1; rw >= 1; --rw)
        if (cost(rw) < cost(a.rw)) a.rw = rw;
    a.nchunk = (nb + 64 * S::NI - 1) / (64 * S::NI);
    const size_t lds = rows_lds<QT, GGUF, MODE>(nb);
    const int rc = dynamic_lds((const void*)matvec_rows<QT, GGUF, MODE>, lds);
    if (rc) return rc;
    hipLaunchKernelGGL((matvec_rows<QT, GGUF, MODE>), dim3((unsigned)std::min<int64_t>(tiles(a.rw), cus)),
                       dim3(kWaves * 64), lds, st, a);
    ASMHIP_TRY(hipGetLastError());
    return kOk;
}

// More than 512 columns (16 blocks).  Small units: a wave multiplies one while the next is
// under way, and starts sooner (8192 x 5504 Q8_0 one, two and three blocks a lane 11.0 / 12.3 /
// 12.9 us, Q4_0 9.1 / 9.6 / 10.3); two for Q4 and Q5 rows that are many, short or above 8192
// columns (33000 x 2080 Q5_0 24.2 / 23.4 / 24.7, 33000 x 8032 Q4_0 38.9 / 38.4 / 38.9).
template <int QT, bool GGUF>
int rows_launch_fmt(const RowsArgs& a, hipStream_t st) {
    if (a.K <= kShortK) return rows_launch_mode<QT, GGUF, kPack64>(a, st);
    if (a.K <= 2048) return rows_launch_mode<QT, GGUF, kPack32>(a, st);
    if constexpr (QT != kRows8)
        if ((a.K <= 4096 || a.K > kWaveK || a.M > 10000) && rows_lds<QT, GGUF, 2>(a.K / 32) <= kLdsBudget)
            return rows_launch_mode<QT, GGUF, 2>(a, st);
    return rows_launch_mode<QT, GGUF, 1>(a, st);
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
// 1 / 2 / 4 rows: 300 x 768 2.03 / 2.15 / 2.67 us, 2048 x 768 2.57 / 2.47 / 2.92, 8192 x 768
// 3.99 / 3.59 / 3.69, 32000 x 288 7.3 / 5.5 / 4.5; 2 / 4 rows: 1000 x 2080 2.81 / 2.94, 4096 x
// 2080 4.41 / 4.06).
template <int QT, bool GGUF>
int wave_launch_fmt(const RowsArgs& a, hipStream_t st) {
    int r = a.K <= kShortK ? (a.M <= 1024 ? 1 : a.M <= 10000 ? 2 : 4) : (a.M <= 512 ? 1 : a.M <= 3000 ? 2 : 4);
    // every wave forms the SwiGLU of x anew, eight exponentials and divisions a pass and lane,
    // for R rows (Q4_0, 2 / 4 rows: 2048 x 576 3.25 / 3.62 us, 4096 x 576 4.21 / 3.69; 512 x 2112
    // 3.36 / 3.60, 1024 x 2112 4.28 / 3.67)
    if (a.pre == kPreSwiGlu) r = a.K <= kShortK ? (a.M <= 1024 ? 1 : a.M <= 3000 ? 2 : 4) : a.M <= 700 ? 2 : 4;
    if (a.post != kPostNone) r = std::max(r, 2);
    const int np = (a.K / 8 + 63) / 64;  // passes of 64 items
    if (a.K <= kShortK) return np <= 1 ? wave_launch_r<QT, GGUF, 1, 1>(a, r, st) : wave_launch_r<QT, GGUF, 2, 1>(a, r, st);
    // four waves share a row's columns: a wave holds at most 4 passes of x
    switch ((np + 3) / 4) {
        case 1: return wave_launch_r<QT, GGUF, 1, 4>(a, r, st);
        case 2: return wave_launch_r<QT, GGUF, 2, 4>(a, r, st);
        case 3: return wave_launch_r<QT, GGUF, 3, 4>(a, r, st);
        default: return wave_launch_r<QT, GGUF, 4, 4>(a, r, st);
    }
}

// Whether matvec_rows is faster than matvec_wave, which takes up to kWaveK columns: wide
// loads and x shared by 16 waves, against no barrier before the weights.  Wave / rows, us,
// with weights from memory, then with weights that stay in the caches:
//   many short rows, several of them a pass: 33000 x 544 Q4_0 8.3 / 6.7, 7.3 / 5.8, 24000 x 544
//     6.2 / 5.1, 5.7 / 5.0, 33000 x 1376 (four rows a unit no more) 11.2 / 12.3, 8.8 / 11.5;
//     from memory 24000 x 1216 9.0 / 8.1; Q5_0, whose wave is the slowest, 12000 x 1216 7.8 /
//     6.4; Q8_0 24000 x 1216 11.8 / 10.1, 33000 x 544 8.7 / 8.3, 6.7 / 6.3 (split 7.8 / 8.3,
//     6.5 / 5.6), but 32000 x 768 8.8 / 9.2;
//   longer rows, a wave each and nearly all waves of the device the same number of them: Q8_0
//     8192 x 4128 11.9 / 9.9, 8.4 / 8.7, but 5000 x 4128 8.4 / 9.5, 5.9 / 8.4, and 4096 x 4128
//     7.4 / 6.7, 5.1 / 5.7, 4096 x 6208 10.1 / 8.9, 6.8 / 7.1; Q5_0 4096 x 4128 8.0 / 6.6, 6.1 /
//     6.2; Q4_0 8192 x 4128 9.2 / 8.5, 7.4 / 8.0, 16384 x 4128 16.0 / 14.4, 12.7 / 13.3, 8192 x
//     8032 13.3 / 11.4, 10.4 / 10.4; split Q4 16384 x 4128 13.6 / 13.5, 11.2 / 12.4, 8192 x 8032
//     12.3 / 11.2, 9.9 / 9.5; split Q8 16384 x 4128 18.9 / 17.2, 13.5 / 13.7.
// matvec_rows also forms the SwiGLU of x once for 16 waves and all their rows (Q4_0 8192 x 576
// 5.0 / 4.3, 4096 x 576 3.7 / 4.3; 4096 x 2112 6.4 / 4.8, 2048 x 2112 4.6 / 4.7; Q8_0 alike).
template <int QT, bool GGUF>
bool rows_faster(const RowsArgs& a) {
    constexpr bool k5 = QT == kRows5 && GGUF;
    if (a.K > kWaveK) return true;
    if (a.K <= 512) return false;
    if (a.pre == kPreSwiGlu) return a.M > (a.K <= 1344 ? 6000 : 2500);
    if (a.K <= kShortK && QT == kRows8) return a.K <= 640 && a.M > 28000;
    if (a.K <= kShortK) return a.M > (k5 ? 14000 : a.K <= 768 ? 20000 : 24000);
    if (a.K <= 1344) return a.M > (k5 ? 10000 : GGUF ? 16000 : 20000);
    if (a.K <= 2048) return k5 && a.M > 11000;
    const int64_t round = (int64_t)kWaves * row_units(), rounds = (a.M + round - 1) / round;
    if (20 * (int64_t)a.M < 17 * rounds * round) return false;  // the last round too empty
    if (GGUF && a.K > (QT == kRows5 ? 4096 : 6144)) return a.M > 3400;
    if (QT != kRows8 && !GGUF) return a.K > 6144 && a.M > 8000;
    return a.M > (GGUF && QT != kRows4 ? 8000 : 11000);
}

template <int QT, bool GGUF>
int rows_or_wave(const RowsArgs& a, hipStream_t st) {
    return a.pre != kPreAttnMerge && rows_faster<QT, GGUF>(a) ? rows_launch_fmt<QT, GGUF>(a, st)
                                                              : wave_launch_fmt<QT, GGUF>(a, st);
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
        (!rows_before_stream(K) || o.attn_splits < 1 || o.attn_splits > kAttnMergeMaxSplits ||
         !attn_head_dim(o.attn_hd) || K % o.attn_hd || (uintptr_t)o.pre_arg % 16))
        return false;
    return K > 0 && K % 32 == 0 && M > 0 && M <= INT32_MAX - 4096 && bytes < (int64_t)kPastEnd && lds <= kLdsBudget &&
           (uintptr_t)w % 4 == 0 && (gguf || ((uintptr_t)scales % 4 == 0 && (uintptr_t)qh % 4 == 0)) &&
           (uintptr_t)x % 4 == 0 && (o.post == kPostNone || (M % 16 == 0 && !o.accumulate));
}

int matvec_rows_launch(int bits, bool gguf, const void* w, const uint8_t* qh, const float* scales, const float* x,
                       float* y, int64_t M, int64_t K, hipStream_t st, const MatvecOpts& o) {
    RowsArgs a{static_cast<const uint8_t*>(w), qh, scales, x, o.pre_arg, y, (int)M, (int)K, o.pre, (int)o.accumulate,
               o.post, 1, 1, o.attn_splits, o.attn_hd, o.eps};
    switch (bits) {
        case 4: return gguf ? rows_or_wave<kRows4, true>(a, st) : rows_or_wave<kRows4, false>(a, st);
        case 5: return gguf ? rows_or_wave<kRows5, true>(a, st) : rows_or_wave<kRows5, false>(a, st);
        case 8: return gguf ? rows_or_wave<kRows8, true>(a, st) : rows_or_wave<kRows8, false>(a, st);
        default: return fail(kInvalidArgument, "matvec rows: %d-bit weights", bits);
    }
}

}  // namespace asmhip
