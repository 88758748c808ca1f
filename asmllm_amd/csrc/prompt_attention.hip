// Attention over a prompt in fp32 for gfx950: y = softmax(q k^T * scale) v over
// [seq][head_dim] rows, all of them (non-causal), the reference's asm_attention
// (attention_avx2.asm:59-218).
#include <math.h>

#include "common.hpp"
#include "kernels.hpp"

namespace asmhip {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr uint32_t kRowPastEnd = 0x80000000u;  // buffer offset that loads zeros, with room for a block's rows above it

__device__ __forceinline__ v4f load4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    const uint4 u = buf_load_b128(r, off);
    return v4f{__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w)};
}

// Rows 16 b.. of a [seq][hd] matrix: offsets into the descriptor are the same for
// every block, and rows past the last one still fall beyond it.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_at(const float* x, int b, int seq, int hd) {
    return make_rsrc(x + (size_t)b * 16 * hd, (uint32_t)(seq - 16 * b) * (uint32_t)hd * 4u);
}

// The online softmax of one query, in powers of two: p = 2^-kSlack 2^(s scale - base),
// base = m scale, for scores s = q.k and scale > 0 (log2(e) included; q takes its sign).
// m follows the maximum of s only when that has grown by more than kSlack / scale (the
// rescaling of the sums is left out for all but a wave's first block as a rule), so that
// a weight is at most 1 and the sums reach no further than the values do; the power of
// two costs no precision.  base is 0 while every score so far is -inf: such scores then
// weigh 0, and a NaN stays one.
constexpr float kSlack = 10.f, kUnit = 0x1p-10f;
__device__ __forceinline__ float base_of(float m) { return m == -INFINITY ? 0.f : m; }
__device__ __forceinline__ float scaled(float m, float scale) {  // one rounding wherever it is used: never part of an fma
#pragma clang fp contract(off)
    return m * scale;
}

// The merge of NW softmax states of one row, a quad of dimensions: state w is
// acc[w * stride], m[w * n] (times scale), l[w * n].
template <int NW>
__device__ __forceinline__ v4f merge_states(const float* acc, const float* m, const float* l, int stride, int n) {
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, m[w * n]);
    const float base = base_of(M);
    float L = 0.f;
    v4f a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const float f = exp2_fast(m[w * n] - base);
        L = fmaf(l[w * n], f, L);
        a += *reinterpret_cast<const v4f*>(acc + w * stride) * f;
    }
    return a / L;
}

// A wave's 16 keys of NJ 16-dimension groups in LDS: loaded with four consecutive
// lanes on 64 bytes of a row (lane l: key l / 4, quads 4 j + l % 4), written and read
// back by the same wave (LDS operations of a wave complete in order, so no barrier).
// Quad p of key r stands at p ^ fold(r), where fold spreads eight consecutive lanes
// over the banks on both sides: consecutive keys differ in bit 2 (the write: two keys
// of four quads), and the read's eight keys in all three bits (SPREAD 8: lanes on keys
// 0-7 or 8-15 of one quad) or four keys in bits 1 and 2 (SPREAD 4: lanes on four
// keys, two quads).
template <int NJ, int SPREAD>
struct KTile {
    static constexpr int kRow = 64 * (NJ + (NJ & 1));  // an even number of groups: fold's bit 2 swaps two
    static constexpr int kBytes = 16 * kRow;
    static __device__ __forceinline__ int fold(int r) {
        return ((r & 1) << 2) | (SPREAD == 8 ? (r >> 1) & 3 : r & 2);
    }
    // The compiler sees one lane: a reader hides its offsets from it, so that it never
    // finds them apart from the lane's own writes and reorders the two (a fence between
    // them also held V's loads back, 1024 x 128 15.6 -> 16.0 us).
    __device__ __forceinline__ void hide() { asm("" : "+v"(even), "+v"(odd)); }
    // byte offset of quad 4 j + s of key r, as two bases (even and odd j) and 64 j
    int even, odd;
    __device__ __forceinline__ KTile(int r, int s) {
        const int f = fold(r), low = r * kRow + 16 * (s ^ (f & 3)), swap = f & 4 ? 64 : 0;
        even = low + swap;
        odd = low - swap;
    }
    __device__ __forceinline__ int at(int j) const { return (j & 1 ? odd : even) + 64 * j; }
};

// One workgroup of NW waves per 16 query rows; wave w walks key blocks
// w, w + NW, ... of 16 keys with its own online softmax state, and the
// states merge once through LDS.  Both products run on v_mfma_f32_16x16x4_f32
// (fp32 in, fp32 sums: the rate of this path's floor) with the operands in the
// layout they leave memory and the first product in:
//   S^T = K Q^T: lane l takes key l % 16 and the four dimensions 16 j + 4 (l / 16)..
//     of one 16-byte LDS read, one dimension a step (Q is loaded the same way, so
//     the order of the contraction is the same on both sides);
//   S^T lands with query l % 16 and keys 4 (l / 16) + i in register i, which is
//     the B operand of Y^T = V^T P^T at step i once it has been exponentiated: k
//     index l / 16 of step i stands for key 4 (l / 16) + i;
//   V: lane l loads dimensions 64 u + 4 (l % 16).. of keys 4 (l / 16) + i: tile t
//     of group u holds dimension 64 u + 4 r + t in its row r.
// K passes through the wave's own piece of LDS (KTile): a load with the keys on
// consecutive lanes, as the operand wants them, touches four cache lines per four
// lanes.  The next block's K is in flight while a block is multiplied.  Bound by the
// fp32 matrix rate of the compute units a prompt's tiles reach (2048 x 128: 128 of
// 256, 37.3 us for 2.1 GFLOP) and the vector work beside it: 46 us with a rescaling
// and expf in every block.
// NJ: 16-dimension groups; FULL: head_dim = 16 NJ, else the dimensions past it load
// zeros.
template <int NJ, bool FULL, int NW>
__global__ __launch_bounds__(NW * 64) void attention_mfma16(const float* __restrict__ q,
                                                            const float* __restrict__ k,
                                                            const float* __restrict__ v, int seq, int hd_,
                                                            float scale, float sign, float slack, float* y) {
    constexpr int NU = (NJ + 3) / 4;  // 64-dimension groups of the second product
    constexpr int HDP = 64 * NU;
    const int hd = FULL ? 16 * NJ : hd_;
    extern __shared__ __attribute__((aligned(16))) float smem[];
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = (int)blockIdx.x * 16;
    const uint32_t row_bytes = (uint32_t)hd * 4u;
    using KT = KTile<NJ, 8>;
    uint8_t* tile = reinterpret_cast<uint8_t*>(smem) + wave * KT::kBytes;
    const KT put(lane >> 2, lane & 3);
    KT get(c, g);
    get.hide();
    // offsets within a block's rows; dimensions past head_dim are sent past the end
    auto off = [&](int row, int d) { return FULL || d < hd ? (uint32_t)row * row_bytes + 4u * (uint32_t)d : kRowPastEnd; };
    uint32_t koff[NJ], voff[NU][4];
#pragma unroll
    for (int j = 0; j < NJ; ++j) koff[j] = off(lane >> 2, 16 * j + 4 * (lane & 3));
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = 64 * u + 4 * c;
            voff[u][i] = d < hd ? (uint32_t)(4 * g + i) * row_bytes + 4u * (uint32_t)d : kRowPastEnd;
        }

    v4f qv[NJ], kv[NJ];
    const int nblk = (seq + 15) >> 4;
    auto load_k = [&](int b) {
        const auto kr = rows_at(k, b, seq, hd);
#pragma unroll
        for (int j = 0; j < NJ; ++j) kv[j] = load4(kr, koff[j]);
    };
    if (wave < nblk) load_k(wave);
    {
        const auto qr = rows_at(q, (int)blockIdx.x, seq, hd);
#pragma unroll
        for (int j = 0; j < NJ; ++j) qv[j] = load4(qr, off(c, 16 * j + 4 * g));
    }
    v4f acc[NU][4];
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[u][t] = v4f{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, ms = m, l = 0.f;  // ms: m scale
    if (sign != 1.f) {  // not otherwise: no wait for q before the first keys are requested
#pragma unroll
        for (int j = 0; j < NJ; ++j) qv[j] *= sign;
    }

    for (int b = wave; b < nblk; b += NW) {
        const auto vr = rows_at(v, b, seq, hd);
        v4f vv[NU][4];
#pragma unroll
        for (int j = 0; j < NJ; ++j) *reinterpret_cast<v4f*>(tile + put.at(j)) = kv[j];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int u = 0; u < NU; ++u) vv[u][i] = load4(vr, voff[u][i]);
        if (b + NW < nblk) load_k(b + NW);
        v4f s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;  // two chains: consecutive steps do not wait for each other
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const v4f kk = *reinterpret_cast<const v4f*>(tile + get.at(j));
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[0], qv[j][0], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[1], qv[j][1], s1, 0, 0, 0);
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[2], qv[j][2], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[3], qv[j][3], s1, 0, 0, 0);
        }
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = s0[i] + s1[i];
        if (16 * b + 16 > seq) {  // the last block: keys past the end weigh nothing
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] = 16 * b + 4 * g + i < seq ? p[i] : -INFINITY;
        }
        float mb = fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3]));
        if (__any(mb > m + slack || m == -INFINITY)) {
            mb = fmaxf(mb, __shfl_xor(mb, 16, kWave));
            mb = fmaxf(mb, __shfl_xor(mb, 32, kWave));
            const float mn = fmaxf(m, mb), msn = scaled(mn, scale), f = exp2_fast(ms - base_of(msn));
            m = mn, ms = msn;
            l *= f;
#pragma unroll
            for (int u = 0; u < NU; ++u)
#pragma unroll
                for (int t = 0; t < 4; ++t) acc[u][t] *= f;
        }
        const float base = base_of(ms);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            p[i] = exp2_fast(fmaf(p[i], scale, -base)) * kUnit;
            l += p[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int u = 0; u < NU; ++u)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[u][i][t], p[i], acc[u][t], 0, 0, 0);
    }
    // wave w's state for query c: acc at [w][c][dimension] (over the K tiles), m and l behind all of them
    __syncthreads();
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);
    constexpr int kPitch = HDP + 4;  // the 16 queries of a store land 4 floats apart modulo the banks
    float* sm_m = smem + NW * 16 * kPitch;
    float* sm_l = sm_m + NW * 16;
    float* mine = smem + (wave * 16 + c) * kPitch;
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i)  // row r = 4 g + i of the tiles: dimensions 64 u + 4 r + t
            *reinterpret_cast<v4f*>(mine + 64 * u + 16 * g + 4 * i) =
                v4f{acc[u][0][i], acc[u][1][i], acc[u][2][i], acc[u][3][i]};
    if (g == 0) sm_m[wave * 16 + c] = ms, sm_l[wave * 16 + c] = l;
    __syncthreads();
    constexpr int kQuads = 16 * HDP / 4;  // output quads, in row order
    for (int e = threadIdx.x; e < kQuads; e += NW * 64) {
        const int r = e / (HDP / 4), d = 4 * (e - r * (HDP / 4));
        const v4f o = merge_states<NW>(smem + r * kPitch + d, sm_m + r, sm_l + r, 16 * kPitch, 16);
        if (row0 + r < seq && d < hd) *reinterpret_cast<v4f*>(y + (size_t)(row0 + r) * hd + d) = o;
    }
}

// The same over 4 query rows a workgroup, for prompts whose 16-row tiles leave
// most of the chip idle: v_mfma_f32_4x4x1_16b_f32 multiplies 16 pairs of 4 x 1
// and 1 x 4 operands, so 4 queries fill it.  Wave w walks blocks w, w + NW, ...
// of 16 keys.  Bound by each workgroup's reading of all of k and v from its L2
// (1 MB at 1024 x 128, 7 us at 64 bytes a clock); keys on consecutive lanes in the
// loads instead of KTile: 28.7 us against 15.9.
//   S^T: the 16 pairs are 4 key sets x 4 slices of the contraction: lane l takes
//     dimensions 16 j + 4 ((l / 4) % 4).. of key 4 (l / 16) + l % 4 (and of query
//     l % 4); the slices are added within the 16-lane row, after which register i
//     holds key 4 (l / 16) + i, query l % 4 in all four of them.
//   Y^T: the 16 pairs are sets of 4 dimension quads; a 16-byte load holds quad
//     l % (HDP / 4) of key set l / (HDP / 4), so at HDP = 64 a row multiplies the
//     keys its own registers hold, and at 128 each half-wave needs the keys of its
//     two rows (one v_permlane16_swap per register).  Tile t, register i, lane l:
//     dimension 4 (4 (l / 4) + i) + t modulo HDP; the halves or rows of a wave that
//     share dimensions add up at the end.
__device__ __forceinline__ float add_row_slices(float v) {  // lanes l, l ^ 4, l ^ 8, l ^ 12: row_ror 8, then 4
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, false));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, false));
    return v;
}

// rows 0 and 1 (2 and 3) of the wave exchanged: lo = the even row's value in both, hi = the odd row's
__device__ __forceinline__ void row_pair(float v, float* lo, float* hi) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    *lo = __uint_as_float(r[0]), *hi = __uint_as_float(r[1]);
}
__device__ __forceinline__ void half_pair(float v, float* lo, float* hi) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    *lo = __uint_as_float(r[0]), *hi = __uint_as_float(r[1]);
}

template <int NJ, bool FULL, int NW>
__global__ __launch_bounds__(NW * 64) void attention_mfma4(const float* __restrict__ q, const float* __restrict__ k,
                                                           const float* __restrict__ v, int seq, int hd_, float scale,
                                                           float sign, float slack, float* y) {
    constexpr int HDP = NJ <= 4 ? 64 : 128;
    constexpr int NV = HDP / 16;  // 16-byte-a-lane loads of V per block
    const int hd = FULL ? 16 * NJ : hd_;
    extern __shared__ __attribute__((aligned(16))) float smem[];
    const int lane = threadIdx.x & 63, qi = lane & 3, row = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = (int)blockIdx.x * 4;
    const uint32_t row_bytes = (uint32_t)hd * 4u;
    using KT = KTile<NJ, 4>;
    uint8_t* tile = reinterpret_cast<uint8_t*>(smem) + wave * KT::kBytes;
    const KT put(lane >> 2, lane & 3);
    KT get(4 * row + qi, (lane >> 2) & 3);
    get.hide();
    auto off = [&](int r, int d) { return FULL || d < hd ? (uint32_t)r * row_bytes + 4u * (uint32_t)d : kRowPastEnd; };
    uint32_t koff[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) koff[j] = off(lane >> 2, 16 * j + 4 * (lane & 3));
    // load n of V: at HDP = 64 key 4 (l / 16) + n, at 128 key 8 (l / 32) + n
    const int vkey = HDP == 64 ? 4 * row : 8 * (lane >> 5), vdim = 4 * (lane % (HDP / 4));
    const uint32_t voff0 = vdim < hd ? (uint32_t)vkey * row_bytes + 4u * (uint32_t)vdim : kRowPastEnd;
    v4f qv[NJ];
    const int nblk = (seq + 15) >> 4;
    // the idle waves of a short prompt leave q alone, whose requests would hold up the others'
    // (64 x 128 6.3 us with them, 4.3 without)
    if (wave < nblk) {
        const auto qr = make_rsrc(q + (size_t)row0 * hd, (uint32_t)(seq - row0) * row_bytes);
#pragma unroll
        for (int j = 0; j < NJ; ++j) qv[j] = load4(qr, off(qi, 16 * j + (lane & 12)));
        if (sign != 1.f) {  // not otherwise: no wait for q before the first keys are requested
#pragma unroll
            for (int j = 0; j < NJ; ++j) qv[j] *= sign;
        }
    }
    v4f acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, ms = m, l = 0.f, lo, hi;  // ms: m scale

    for (int b = wave; b < nblk; b += NW) {
        const auto kr = rows_at(k, b, seq, hd), vr = rows_at(v, b, seq, hd);
        v4f kv[NJ], vv[NV];
        // the rows' offsets formed anew in every block where head_dim is no constant: eight
        // of them kept in registers went to scratch memory (head_dim 116, 1000 rows 14.4 us, 13.6 so)
        uint32_t voff = voff0;
        if (!FULL) asm("" : "+v"(voff));
#pragma unroll
        for (int j = 0; j < NJ; ++j) kv[j] = load4(kr, koff[j]);
#pragma unroll
        for (int n = 0; n < NV; ++n) vv[n] = load4(vr, voff + (uint32_t)n * row_bytes);
#pragma unroll
        for (int j = 0; j < NJ; ++j) *reinterpret_cast<v4f*>(tile + put.at(j)) = kv[j];
        v4f s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const v4f kk = *reinterpret_cast<const v4f*>(tile + get.at(j));
            s0 = __builtin_amdgcn_mfma_f32_4x4x1f32(kk[0], qv[j][0], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_4x4x1f32(kk[1], qv[j][1], s1, 0, 0, 0);
            s0 = __builtin_amdgcn_mfma_f32_4x4x1f32(kk[2], qv[j][2], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_4x4x1f32(kk[3], qv[j][3], s1, 0, 0, 0);
        }
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = add_row_slices(s0[i] + s1[i]);
        if (16 * b + 16 > seq) {
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] = 16 * b + 4 * row + i < seq ? p[i] : -INFINITY;
        }
        float mb = fmaxf(fmaxf(p[0], p[1]), fmaxf(p[2], p[3]));
        if (__any(mb > m + slack || m == -INFINITY)) {
            row_pair(mb, &lo, &hi);
            mb = fmaxf(lo, hi);
            half_pair(mb, &lo, &hi);
            const float mn = fmaxf(m, fmaxf(lo, hi)), msn = scaled(mn, scale), f = exp2_fast(ms - base_of(msn));
            m = mn, ms = msn;
            l *= f;
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t] *= f;
        }
        const float base = base_of(ms);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            p[i] = exp2_fast(fmaf(p[i], scale, -base)) * kUnit;
            l += p[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (HDP == 64) {
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_4x4x1f32(vv[i][t], p[i], acc[t], 0, 0, 0);
            } else {
                row_pair(p[i], &lo, &hi);  // keys 8 (l / 32) + i and + 4 + i
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    acc[t] = __builtin_amdgcn_mfma_f32_4x4x1f32(vv[i][t], lo, acc[t], 0, 0, 0);
                    acc[t] = __builtin_amdgcn_mfma_f32_4x4x1f32(vv[4 + i][t], hi, acc[t], 0, 0, 0);
                }
            }
        }
    }
    // the wave's state: sums over its rows (and halves), then [wave][query][dimension] in LDS
    row_pair(l, &lo, &hi);
    l = lo + hi;
    half_pair(l, &lo, &hi);
    l = lo + hi;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float a = acc[t][i];
            if constexpr (HDP == 64) {
                row_pair(a, &lo, &hi);
                a = lo + hi;
            }
            half_pair(a, &lo, &hi);
            acc[t][i] = lo + hi;
        }
    constexpr int kPitch = HDP + 4;
    __syncthreads();  // the K tiles are read
    float* sm_m = smem + NW * 4 * kPitch;
    float* sm_l = sm_m + NW * 4;
    if (lane < HDP / 4) {  // lane: query qi, quads 4 (l / 4) + i of tile order t
        float* mine = smem + (wave * 4 + qi) * kPitch + 16 * (lane >> 2);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<v4f*>(mine + 4 * i) = v4f{acc[0][i], acc[1][i], acc[2][i], acc[3][i]};
    }
    if (lane < 4) sm_m[wave * 4 + lane] = ms, sm_l[wave * 4 + lane] = l;
    __syncthreads();
    if (threadIdx.x < HDP) {  // 4 rows x HDP / 4 quads
        const int r = threadIdx.x / (HDP / 4), d = 4 * (threadIdx.x % (HDP / 4));
        const v4f o = merge_states<NW>(smem + r * kPitch + d, sm_m + r, sm_l + r, 4 * kPitch, 4);
        if (row0 + r < seq && d < hd) *reinterpret_cast<v4f*>(y + (size_t)(row0 + r) * hd + d) = o;
    }
}

// Any head_dim and alignment: one workgroup per query row, scores in LDS.
constexpr int kRowThreads = 256;

template <bool kMax>
__device__ __forceinline__ float row_reduce(float v, float* red) {
    v = kMax ? wave_max(v) : wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = red[0];
#pragma unroll
    for (int i = 1; i < kRowThreads / kWave; ++i) t = kMax ? fmaxf(t, red[i]) : t + red[i];
    return t;
}

__global__ __launch_bounds__(kRowThreads) void attention_rows(const float* __restrict__ q, const float* __restrict__ k,
                                                              const float* __restrict__ v, float* __restrict__ y,
                                                              int seq, int hd, float scale) {
    extern __shared__ float sc[];  // seq scores
    __shared__ float red[kRowThreads / kWave];
    const int row = blockIdx.x;
    const float* qi = q + (size_t)row * hd;
    for (int j = threadIdx.x; j < seq; j += kRowThreads) {
        const float* kj = k + (size_t)j * hd;
        float d = 0.f;
        for (int t = 0; t < hd; ++t) d = fmaf(qi[t], kj[t], d);
        sc[j] = d * scale;
    }
    __syncthreads();
    float m = -INFINITY;
    for (int j = threadIdx.x; j < seq; j += kRowThreads) m = fmaxf(m, sc[j]);
    m = row_reduce<true>(m, red);
    float s = 0.f;
    for (int j = threadIdx.x; j < seq; j += kRowThreads) {
        const float e = expf(sc[j] - m);
        sc[j] = e;
        s += e;
    }
    s = row_reduce<false>(s, red);
    __syncthreads();
    for (int t = threadIdx.x; t < hd; t += kRowThreads) {
        float a = 0.f;
        for (int j = 0; j < seq; ++j) a = fmaf(sc[j], v[(size_t)j * hd + t], a);
        y[(size_t)row * hd + t] = a / s;
    }
}

// Up to 1024 rows the 4-row tiles are at most one workgroup per compute unit (256):
// head_dim 128, 1024 rows 15.9 us against 22.3 with 16-row tiles on 64 units (one
// workgroup per row and scalar dots before: 274), 64 x 128 4.3 against 4.5, head_dim
// 64, 1024 rows 10.1 against 12.8.  Past that they take a second round and read k and
// v four times as often: 1100 rows 29.2 against 22.7, 2048 rows 49.2 against 37.3.
constexpr int kFourRowSeq = 1024;

template <int NJ, bool FULL>
int launch_mfma(const float* q, const float* k, const float* v, float* y, int seq, int hd, float factor,
                hipStream_t st) {
    // the score's scale as the kernels take it: > 0 with log2(e); its slack; q's factor 1, -1 or
    // 0.  The first ten dwords of the arguments are in registers when a wave starts; a factor
    // that came by a load, before the first keys were requested, cost 64 x 128 2 us of 4.3.
    const float scale = factor == 0.f ? 1.f : fabsf(factor) * 1.44269504088896340736f, slack = kSlack / scale;
    const float sign = factor < 0.f ? -1.f : factor == 0.f ? 0.f : 1.f;
    if constexpr (NJ <= 8) {
        if (seq <= kFourRowSeq) {
            constexpr int NW = 16, HDP = NJ <= 4 ? 64 : 128;
            const size_t lds = (size_t)max(NW * KTile<NJ, 4>::kBytes, NW * 4 * (HDP + 6) * (int)sizeof(float));
            const int rc = dynamic_lds((const void*)attention_mfma4<NJ, FULL, NW>, lds);
            if (rc) return rc;
            hipLaunchKernelGGL((attention_mfma4<NJ, FULL, NW>), dim3((unsigned)((seq + 3) / 4)), dim3(NW * 64), lds, st,
                               q, k, v, seq, hd, scale, sign, slack, y);
            return kOk;
        }
    }
    constexpr int NW = NJ <= 8 ? 8 : 4, HDP = (NJ + 3) / 4 * 64;
    const size_t lds = (size_t)max(NW * KTile<NJ, 8>::kBytes, NW * 16 * (HDP + 6) * (int)sizeof(float));
    const int rc = dynamic_lds((const void*)attention_mfma16<NJ, FULL, NW>, lds);
    if (rc) return rc;
    hipLaunchKernelGGL((attention_mfma16<NJ, FULL, NW>), dim3((unsigned)((seq + 15) / 16)), dim3(NW * 64), lds, st, q,
                       k, v, seq, hd, scale, sign, slack, y);
    return kOk;
}

template <int NJ>
int launch_groups(const float* q, const float* k, const float* v, float* y, int seq, int hd, float scale,
                  hipStream_t st) {
    return hd == 16 * NJ ? launch_mfma<NJ, true>(q, k, v, y, seq, hd, scale, st)
                         : launch_mfma<NJ, false>(q, k, v, y, seq, hd, scale, st);
}

}  // namespace

int attention_launch(const float* q, const float* k, const float* v, float* y, int64_t seq, int64_t hd, float scale,
                     hipStream_t st) {
    if (seq <= 0 || hd <= 0) return fail(kInvalidArgument, "attention: need seq > 0 and head_dim > 0");
    if (hd > kMaxStridedLen) return fail(kInvalidArgument, "attention: head_dim %lld", (long long)hd);
    if (seq > 40000) return fail(kUnsupported, "attention: seq_len %lld exceeds the LDS score buffer", (long long)seq);
    // 16-byte loads and stores of whole quads of dimensions, at most 256 of them;
    // 32-bit byte offsets hold: 40000 rows x 1 KB
    const bool quads = hd % 4 == 0 && hd <= 256 &&
                       ((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)y) % 16 == 0;
    const int n = (int)seq, d = (int)hd;
    int rc = kOk;
    if (!quads) {
        rc = dynamic_lds((const void*)attention_rows, (size_t)seq * sizeof(float));
        if (rc) return rc;
        hipLaunchKernelGGL(attention_rows, dim3((unsigned)seq), dim3(kRowThreads), (size_t)seq * sizeof(float), st, q,
                           k, v, y, n, d, scale);
    } else if (hd <= 48) {
        rc = launch_groups<3>(q, k, v, y, n, d, scale, st);
    } else if (hd <= 64) {
        rc = launch_groups<4>(q, k, v, y, n, d, scale, st);
    } else if (hd <= 80) {
        rc = launch_groups<5>(q, k, v, y, n, d, scale, st);
    } else if (hd <= 128) {
        rc = launch_groups<8>(q, k, v, y, n, d, scale, st);
    } else {
        rc = launch_groups<16>(q, k, v, y, n, d, scale, st);
    }
    if (rc) return rc;
    ASMHIP_TRY(hipGetLastError());
    return kOk;
}

}  // namespace asmhip
