// Factor-streaming forward kernel for base-4 schedules -- any number of blocks -- over rows of up to
// 4096 elements, in ONE launch: each row is read once and written once.
//
// A workgroup of W wavefronts takes a tile of 1024 * W * RB values: 4 * RB << (NBITS - log_n) rows,
// NBITS = 8 + log2(W).  Within the tile a value is addressed by an index of NBITS bits (the element
// in the low log_n bits, row bits above), two row bits that always sit on the lane bits 0 and 1, and
// RB planes.  A thread holds 16 values of a plane: four consecutive index bits ("the register bits")
// run over its registers, four over lane bits 2..5, the rest over the wavefronts.
//
// The schedule is cut into PHASES, each a run of stages on the four bits that sit in registers; between
// phases the tile passes through LDS, which changes what the register bits are.  Within a phase every
// stage (a "level") is one v_mfma_f32_4x4x1_16b per column of its 4x4 factors: operand A is the factor
// (lane = 4 * block + output), B the rows (lane = 4 * block + row), and the result comes back in the
// layout of B, so levels chain without moving data.  The closing 2x2 stage of an odd number of bits
// runs pair by pair on the vector units: as a 4x4 matrix with zeros for the other bit of its register
// pair, an infinity would reach the other pair's outputs as 0 * Inf.
//
// The factors are not kept from tile to tile: they stream from L2 while the previous level computes,
// 4 * RB << (NBITS - log_n) rows sharing each read.  Register-resident factors (fast4g.hpp) reach 1024
// elements; beyond that they need a chunk pass and one pass over memory per remaining stage.
// Measured against those (float): 1500 rows of 2048, two blocks: 23.5 against 43 us; 16384 rows of 2048,
// two blocks: 121 against 208 us; 8192 rows of 4096, one block: 99 against 123 us, two blocks 139 against 213;
// 16384 rows of 4096, one block, which those leave to the LDS fallback: 209 against 658 us.  What bounds
// it: one workgroup a compute unit at 4096 elements (128 KiB of LDS), whose loads, levels and stores
// follow one another.
#pragma once

#include <type_traits>

#include "fast.hpp"

namespace bf {

constexpr int kStreamMaxLevels = 64;
constexpr int kStreamMaxPhases = 40;
constexpr int kStreamMaxSaves = 7;

// The tables travel as kernel arguments, packed into whole words: the kernel indexes them with loop
// counters, and scalar loads come in words.
struct StreamLevel {
    unsigned off;           // bytes from the start of the stack's factors to the stage's
    unsigned bits;

    // p: lowest element bit of the stage; radix4: it pairs p and p + 1 (tw4), otherwise p alone (tw2)
    // pair: it takes the register bits (2, 3) instead of (0, 1); upper: its single bit is the upper one
    // save: 1 + plane that receives the tile behind this level, 0: none
    // ends: 1 + number of the phase that follows, 0: the phase goes on
    static __host__ __device__ unsigned pack(int p, int radix4, int pair, int upper, int save, int ends)
    {
        return (unsigned)(p | radix4 << 4 | pair << 5 | upper << 6 | save << 7 | ends << 16);
    }
    __host__ __device__ int p() const { return bits & 15; }
    __host__ __device__ int radix4() const { return (bits >> 4) & 1; }
    __host__ __device__ int pair() const { return (bits >> 5) & 1; }
    __host__ __device__ int upper() const { return (bits >> 6) & 1; }
    __host__ __device__ int save() const { return (bits >> 7) & 7; }
    __host__ __device__ int ends() const { return (bits >> 16) & 255; }
};

struct StreamPhase {
    unsigned places;   // index bits on lane bits 2..5 and on the wavefront number's bits, four bits each
    unsigned reg;      // first of the four register bits
    __host__ __device__ int lane(int k) const { return (places >> (4 * k)) & 15; }
    __host__ __device__ int wave(int k) const { return (places >> (16 + 4 * k)) & 15; }
};

struct StreamArgs {
    const void *tw4, *tw2;
    int64_t tw4_stack_stride, tw2_stack_stride;   // scalars
    const void *in;
    View in_view;
    void *out;
    StackView out_view;
    const void *bias;         // NULL, or the columns of all stacks side by side
    void *save[kStreamMaxSaves];   // dense (B, S, n) planes
    int64_t batch;
    int log_n;
    int nlevels;
    int in_vec, out_vec;      // rows can be read / written four scalars (complex64: two) at a time
    StreamPhase phase[kStreamMaxPhases];
    StreamLevel level[kStreamMaxLevels];
};

typedef float StreamV4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ StreamV4 stream_mfma(float a, float b, StreamV4 c)
{
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
}

// The 4x4 matrices of one level: a row of each of the four blocks that the register bits outside
// the level's pair run over.
template <typename T> struct StreamRows;
template <> struct StreamRows<float> { float a[4][4]; };
template <> struct StreamRows<float2> { float re[4][4], im[4][4]; };

// y = M x for the four settings q of a plane; value k of setting q is v[q * QS + k * KS].  The four
// chains of dependent MFMAs are interleaved.
template <int QS, int KS>
__device__ __forceinline__ void stream_apply(const StreamRows<float> &m, float (&v)[16])
{
    StreamV4 d[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) d[q] = stream_mfma(m.a[q][0], v[q * QS], StreamV4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int k = 1; k < 4; ++k)
#pragma unroll
        for (int q = 0; q < 4; ++q) d[q] = stream_mfma(m.a[q][k], v[q * QS + k * KS], d[q]);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        v[q * QS] = d[q].x; v[q * QS + KS] = d[q].y;
        v[q * QS + 2 * KS] = d[q].z; v[q * QS + 3 * KS] = d[q].w;
    }
}
template <int QS, int KS>
__device__ __forceinline__ void stream_apply(const StreamRows<float2> &m, float2 (&v)[16])
{
#pragma unroll
    for (int h = 0; h < 4; h += 2) {   // two settings at a time: four chains
        StreamV4 re[2], im[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) re[q] = im[q] = StreamV4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                re[q] = stream_mfma(m.re[h + q][k], v[(h + q) * QS + k * KS].x, re[q]);
                im[q] = stream_mfma(m.im[h + q][k], v[(h + q) * QS + k * KS].x, im[q]);
            }
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                re[q] = stream_mfma(m.im[h + q][k], -v[(h + q) * QS + k * KS].y, re[q]);
                im[q] = stream_mfma(m.re[h + q][k], v[(h + q) * QS + k * KS].y, im[q]);
            }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            v[(h + q) * QS] = make_float2(re[q].x, im[q].x);
            v[(h + q) * QS + KS] = make_float2(re[q].y, im[q].y);
            v[(h + q) * QS + 2 * KS] = make_float2(re[q].z, im[q].z);
            v[(h + q) * QS + 3 * KS] = make_float2(re[q].w, im[q].w);
        }
    }
}

// The same for a 2x2 stage.  OWN, OTHER: register steps of the stage's bit and of the other bit of
// the pair.  Lane i of a block holds the factor's row of output i & 1 at the value i >> 1 of the other
// bit; the block's four lanes read them from each other as DPP operands, two instructions an output
// (16384 rows of 2048, one block: 76.9 us against 82.2 for a 4x4 matrix on the matrix units).
template <int QS, int OTHER, int OWN>
__device__ __forceinline__ void stream_apply2(const StreamRows<float> &m, float (&v)[16])
{
    auto pair = [&](int q, auto other) {
        constexpr int o = decltype(other)::value;
        float &x0 = v[q * QS + o * OTHER], &x1 = v[q * QS + o * OTHER + OWN];
        float y0 = mul(dpp_move<(2 * o) * 0x55>(m.a[q][0]), x0), y1 = mul(dpp_move<(2 * o + 1) * 0x55>(m.a[q][0]), x0);
        y0 = mac(y0, dpp_move<(2 * o) * 0x55>(m.a[q][1]), x1);
        y1 = mac(y1, dpp_move<(2 * o + 1) * 0x55>(m.a[q][1]), x1);
        x0 = y0;
        x1 = y1;
    };
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        pair(q, std::integral_constant<int, 0>());
        pair(q, std::integral_constant<int, 1>());
    }
}
template <int QS, int OTHER, int OWN>
__device__ __forceinline__ void stream_apply2(const StreamRows<float2> &m, float2 (&v)[16])
{
    auto pair = [&](int q, auto other) {
        constexpr int o = decltype(other)::value;
        float2 &x0 = v[q * QS + o * OTHER], &x1 = v[q * QS + o * OTHER + OWN];
        auto row = [&](int k, auto own) {
            constexpr int ctrl = (2 * o + decltype(own)::value) * 0x55;
            return make_float2(dpp_move<ctrl>(m.re[q][k]), dpp_move<ctrl>(m.im[q][k]));
        };
        constexpr std::integral_constant<int, 0> first = {};
        constexpr std::integral_constant<int, 1> second = {};
        const float2 zero = zero_of(float2());
        const float2 y0 = mac(mac(zero, row(0, first), x0), row(1, first), x1);
        const float2 y1 = mac(mac(zero, row(0, second), x0), row(1, second), x1);
        x0 = y0;
        x1 = y1;
    };
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        pair(q, std::integral_constant<int, 0>());
        pair(q, std::integral_constant<int, 1>());
    }
}

// Two scalars that are next to each other in memory: the row of a 2x2 factor.
template <typename T> struct StreamPair { T x, y; };

__device__ __forceinline__ StreamPair<float> stream_load2(__amdgpu_buffer_rsrc_t r, int voff, int soff, float)
{
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    const v2u raw = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
    const unsigned x = raw.x, y = raw.y;
    return {__uint_as_float(x), __uint_as_float(y)};
}
__device__ __forceinline__ StreamPair<float2> stream_load2(__amdgpu_buffer_rsrc_t r, int voff, int soff, float2)
{
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    const v4u raw = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
    const unsigned x = raw.x, y = raw.y, z = raw.z, w = raw.w;
    return {make_float2(__uint_as_float(x), __uint_as_float(y)), make_float2(__uint_as_float(z), __uint_as_float(w))};
}

__device__ __forceinline__ void stream_load4(__amdgpu_buffer_rsrc_t r, int voff, float (&v)[4])
{
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    const v4u raw = __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0);
    const unsigned x = raw.x, y = raw.y, z = raw.z, w = raw.w;
    v[0] = __uint_as_float(x); v[1] = __uint_as_float(y); v[2] = __uint_as_float(z); v[3] = __uint_as_float(w);
}
__device__ __forceinline__ void stream_load4(__amdgpu_buffer_rsrc_t r, int voff, float2 (&v)[4])
{
    const StreamPair<float2> lo = stream_load2(r, voff, 0, float2()), hi = stream_load2(r, voff, 16, float2());
    v[0] = lo.x; v[1] = lo.y; v[2] = hi.x; v[3] = hi.y;
}
__device__ __forceinline__ void stream_store4(__amdgpu_buffer_rsrc_t r, int voff, float v0, float v1, float v2, float v3)
{
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    v4u raw;
    raw.x = __float_as_uint(v0); raw.y = __float_as_uint(v1); raw.z = __float_as_uint(v2); raw.w = __float_as_uint(v3);
    __builtin_amdgcn_raw_buffer_store_b128(raw, r, voff, 0, 0);
}
__device__ __forceinline__ void stream_store4(__amdgpu_buffer_rsrc_t r, int voff, float2 v0, float2 v1, float2 v2, float2 v3)
{
    stream_store4(r, voff, v0.x, v0.y, v1.x, v1.y);
    stream_store4(r, voff + 16, v2.x, v2.y, v3.x, v3.y);
}

// The lane's row of the level's factors, as loaded: a row of the 4x4 factor, or (s1 alone) of the
// 2x2 factor at a value of the other bit (stream_apply2).  One for each setting q of the register
// bits outside the level's pair.
template <typename T>
struct StreamRaw { StreamPair<T> s1[4], s2[4]; };

__host__ __device__ constexpr int stream_fold(int idx) { return idx ^ ((idx >> 4) & 15) ^ ((idx >> 8) & 15); }

__device__ __forceinline__ int stream_pair(int e, int p) { return ((e >> (p + 1)) << p) | (e & ((1 << p) - 1)); }
__device__ __forceinline__ int stream_quad(int e, int p) { return ((e >> (p + 2)) << p) | (e & ((1 << p) - 1)); }

__device__ __forceinline__ void stream_put(StreamRows<float> &m, int q, int k, float v) { m.a[q][k] = v; }
__device__ __forceinline__ void stream_put(StreamRows<float2> &m, int q, int k, float2 v) { m.re[q][k] = v.x; m.im[q][k] = v.y; }

// The lane's row as loaded: of four entries, or (a 2x2 stage) of two.
template <typename T, bool RADIX4>
__device__ __forceinline__ void stream_rows(StreamRows<T> &m, const StreamRaw<T> &raw)
{
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        stream_put(m, q, 0, raw.s1[q].x);
        stream_put(m, q, 1, raw.s1[q].y);
        if constexpr (RADIX4) {
            stream_put(m, q, 2, raw.s2[q].x);
            stream_put(m, q, 3, raw.s2[q].y);
        }
    }
}

template <typename T, int W, int RB>
__global__ __launch_bounds__(W * 64, W == 16 ? 4 : 2) void stream_fw_kernel(StreamArgs a)
{
    constexpr int LOGW = W == 16 ? 4 : W == 8 ? 3 : 2;
    constexpr int NBITS = 8 + LOGW;
    constexpr int PLANE = 4 << NBITS;   // values of a plane
    constexpr int EB = (int)sizeof(T);
    __shared__ __align__(16) T lds[RB * PLANE];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int row4 = lane & 3;
    const int stack = blockIdx.y;
    const int L = a.log_n, n = 1 << L, emask = n - 1;
    const int hi_rows = 1 << (NBITS - L);              // row groups (of four) in a plane
    const int64_t row0 = (int64_t)blockIdx.x * (4 * RB * hi_rows);
    const int rows_valid = (int)(a.batch - row0 < 4 * RB * hi_rows ? a.batch - row0 : 4 * RB * hi_rows);
    const View in_view = a.in_view, out_view = stack_view(a.out_view, stack);
    const T *in = reinterpret_cast<const T *>(a.in) + row0 * in_view.sb + stack * in_view.ss;
    T *out = reinterpret_cast<T *>(a.out) + row0 * out_view.sb + stack * out_view.ss;
    const __amdgpu_buffer_rsrc_t in_rs = make_rsrc(in), out_rs = make_rsrc(out);
    const __amdgpu_buffer_rsrc_t tw4_rs = make_rsrc(reinterpret_cast<const T *>(a.tw4) + stack * a.tw4_stack_stride);
    const __amdgpu_buffer_rsrc_t tw2_rs = make_rsrc(reinterpret_cast<const T *>(a.tw2) + stack * a.tw2_stack_stride);

    // ---- factors of a level, in the phase they are used in
    int idx_base = 0, reg_lo = 0;   // index of the thread's value 0; first register bit
    auto enter = [&](int ph) {
        const StreamPhase p = a.phase[ph];
        reg_lo = (int)p.reg;
        int v = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) v |= ((lane >> (2 + b)) & 1) << p.lane(b);
#pragma unroll
        for (int b = 0; b < LOGW; ++b) v |= ((wave >> b) & 1) << p.wave(b);
        idx_base = v;
    };
    StreamRaw<T> raw;
    auto load_level = [&](int lv) {
        const StreamLevel l = a.level[lv];
        const int e = idx_base & emask;
        const int i = lane & 3;
        const int p = l.p();
        const int other = l.pair() ? reg_lo : reg_lo + 2;   // index bits of the settings q
        if (l.radix4()) {
            const int voff = (stream_quad(e, p) * 16 + i * 4) * EB;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int soff = (int)l.off + stream_quad((q << other) & emask, p) * 16 * EB;
                raw.s1[q] = stream_load2(tw4_rs, voff, soff, T());
                raw.s2[q] = stream_load2(tw4_rs, voff + 2 * EB, soff, T());
            }
        } else {
            const int rest = (i >> 1) << (l.upper() ? p - 1 : p + 1);
            const int voff = (stream_pair((e | rest) & emask, p) * 4 + (i & 1) * 2) * EB;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                raw.s1[q] = stream_load2(tw2_rs, voff, (int)l.off + stream_pair((q << other) & emask, p) * 4 * EB, T());
        }
    };
    enter(0);
    load_level(0);

    // ---- rows into LDS.  A unit is a run of 16 bytes' worth of four scalars (complex64: the same four
    // elements in two halves); lanes take four rows of sixteen consecutive units.
    auto unit = [&](int c, int &idx, int &row, int &word) {
        const int u = c * (W * 64) + t;
        const int chunk = u >> 2;
        const int rb = chunk >> (NBITS - 2);
        idx = (chunk & ((1 << (NBITS - 2)) - 1)) << 2;
        row = (u & 3) + 4 * ((idx >> L) + rb * hi_rows);
        word = rb * PLANE + (stream_fold(idx) << 2 | (u & 3));
    };
    const int in_row = (int)(in_view.sb * EB), out_row = (int)(out_view.sb * EB);
    if (a.in_vec) {
#pragma unroll
        for (int c = 0; c < 4 * RB; ++c) {
            int idx, row, word;
            unit(c, idx, row, word);
            const int e = idx & emask;
            const int voff = row < rows_valid && e < in_view.width ? row * in_row + e * EB : kOob;
            T x[4];
            stream_load4(in_rs, voff, x);
#pragma unroll
            for (int j = 0; j < 4; ++j) lds[word ^ (j << 2)] = x[j];
        }
    } else {
#pragma unroll
        for (int c = 0; c < 4 * RB; ++c) {
            int idx, row, word;
            unit(c, idx, row, word);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = (idx + j) & emask;
                const int r = row + 4 * (((idx + j) >> L) - (idx >> L));
                const int voff = r < rows_valid && e < in_view.width ? r * in_row + (int)(e * in_view.se * EB) : kOob;
                lds[word ^ (j << 2)] = buf_load<T>(in_rs, voff, 0);
            }
        }
    }

    // ---- the thread's 16 values of every plane through LDS, in the current phase's layout
    int word_base = 0, word_reg[16];
    auto words = [&] {
        word_base = stream_fold(idx_base) << 2 | row4;
#pragma unroll
        for (int r = 0; r < 16; ++r) word_reg[r] = stream_fold(r << reg_lo) << 2;
    };
    T v[RB][16];
    words();
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) v[rb][r] = lds[rb * PLANE + (word_base ^ word_reg[r])];

    for (int lv = 0; lv < a.nlevels; ++lv) {
        const StreamLevel l = a.level[lv];
        StreamRows<T> m;
        if (l.radix4()) stream_rows<T, true>(m, raw);
        else stream_rows<T, false>(m, raw);
        const int cur_base = idx_base, cur_lo = reg_lo;
        if (l.ends()) enter(l.ends() - 1);
        if (lv + 1 < a.nlevels) load_level(lv + 1);
        if (l.radix4()) {
            if (l.pair()) {
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) stream_apply<1, 4>(m, v[rb]);
            } else {
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) stream_apply<4, 1>(m, v[rb]);
            }
        } else if (l.pair()) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                if (l.upper()) stream_apply2<1, 4, 8>(m, v[rb]);
                else stream_apply2<1, 8, 4>(m, v[rb]);
            }
        } else {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                if (l.upper()) stream_apply2<4, 1, 2>(m, v[rb]);
                else stream_apply2<4, 2, 1>(m, v[rb]);
            }
        }
        if (l.save()) {
            // straight out of the registers: the plan saves where the lanes or the registers run over
            // the low bits, so that runs of at least 64 bytes leave together
            T *plane = reinterpret_cast<T *>(a.save[l.save() - 1]) + (row0 * gridDim.y + stack) * n;
            const __amdgpu_buffer_rsrc_t rs = make_rsrc(plane);
            const int pitch = (int)gridDim.y * n;
            if (cur_lo == 0 && L >= 4) {
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const int row = row4 + 4 * ((cur_base >> L) + rb * hi_rows);
                    const int voff = row < rows_valid ? (row * pitch + (cur_base & emask)) * EB : kOob;
#pragma unroll
                    for (int r = 0; r < 16; r += 4)
                        stream_store4(rs, voff + r * EB, v[rb][r], v[rb][r + 1], v[rb][r + 2], v[rb][r + 3]);
                }
            } else {
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int idx = cur_base | (r << cur_lo);
                        const int row = row4 + 4 * ((idx >> L) + rb * hi_rows);
                        buf_store(rs, row < rows_valid ? (row * pitch + (idx & emask)) * EB : kOob, 0, v[rb][r]);
                    }
            }
        }
        if (l.ends()) {
            __syncthreads();   // everybody has read the tile
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int r = 0; r < 16; ++r) lds[rb * PLANE + (word_base ^ word_reg[r])] = v[rb][r];
            words();
            __syncthreads();
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int r = 0; r < 16; ++r) v[rb][r] = lds[rb * PLANE + (word_base ^ word_reg[r])];
        }
    }

    // ---- rows out
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 16; ++r) lds[rb * PLANE + (word_base ^ word_reg[r])] = v[rb][r];
    __syncthreads();
    const T *bias = reinterpret_cast<const T *>(a.bias);
#pragma unroll
    for (int c = 0; c < 4 * RB; ++c) {
        int idx, row, word;
        unit(c, idx, row, word);
        T y[4] = {lds[word], lds[word ^ 4], lds[word ^ 8], lds[word ^ 12]};
        if (a.out_vec) {
            const int e = idx & emask;
            const bool ok = row < rows_valid && e < out_view.width;
            if (bias && e < out_view.width) {
#pragma unroll
                for (int j = 0; j < 4; ++j) y[j] = add(y[j], bias[stack * a.out_view.width + e + j]);
            }
            const int voff = ok ? row * out_row + e * EB : kOob;
            stream_store4(out_rs, voff, y[0], y[1], y[2], y[3]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = (idx + j) & emask;
                const int r = row + 4 * (((idx + j) >> L) - (idx >> L));
                const bool ok = r < rows_valid && e < out_view.width;
                if (bias && e < out_view.width) y[j] = add(y[j], bias[stack * a.out_view.width + e]);
                buf_store(out_rs, ok ? r * out_row + (int)(e * out_view.se * EB) : kOob, 0, y[j]);
            }
        }
    }
}

}  // namespace bf
