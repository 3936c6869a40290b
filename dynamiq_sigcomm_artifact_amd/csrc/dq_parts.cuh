// A part of a chunk per lane: eight or four elements instead of the sixteen of dq_tile16.cuh, for vectors too short to fill the GPU
// with a chunk per lane (dq_scaling_hier16_short.hip, dq_single_pass.hip).
#pragma once

#include "dq_tile16.cuh"

namespace dq {

// With sixteen elements per lane a wave works through four superchunks, and a short vector has fewer such waves than the GPU
// has SIMDs: what counts then is the length of a wave's instruction stream.  A lane with four elements makes it a third as
// long and the waves four times as many: a chunk is a quad of lanes, a superchunk a wave.  In between, eight: a chunk is a pair
// of lanes, a superchunk half a wave.
template <int DT, int N> struct RawPart;

template <int N> struct RawPart<DQ_BF16, N> {
    static constexpr int kCount = N, kWords = N / 2;
    uint32_t w[kWords];
    __device__ __forceinline__ void zero()
    {
#pragma unroll
        for (int k = 0; k < kWords; k++) w[k] = 0u;
    }
    // see Raw16
    __device__ __forceinline__ void halves()
    {
#pragma unroll
        for (int k = 0; k < kWords; k++) w[k] = 0x3f003f00u;
    }
    __device__ __forceinline__ uint32_t absmax_bits() const
    {
        uint32_t m = w[0] & 0x7fff7fffu;
#pragma unroll
        for (int k = 1; k < kWords; k++) m = pk_max_u16(m, w[k] & 0x7fff7fffu);
        return max(m << 16, m & 0xffff0000u);
    }
    // vec: p is 16-byte aligned (and e a multiple of N)
    __device__ __forceinline__ void load(const void *p, int64_t e, bool vec)
    {
        typedef uint32_t words __attribute__((ext_vector_type(kWords)));
        const volatile uint16_t *h = static_cast<const volatile uint16_t *>(p) + e;
        if (vec) {
            const words q = *reinterpret_cast<const words *>(static_cast<const uint16_t *>(p) + e);
#pragma unroll
            for (int k = 0; k < kWords; k++) w[k] = q[k];
        } else {
#pragma unroll
            for (int k = 0; k < kWords; k++) w[k] = (uint32_t)h[2 * k] | ((uint32_t)h[2 * k + 1] << 16);
        }
    }
    __device__ __forceinline__ void store(void *p, int64_t e, bool vec) const
    {
        typedef uint32_t words __attribute__((ext_vector_type(kWords)));
        volatile uint16_t *h = static_cast<volatile uint16_t *>(p) + e;
        if (vec) {
            words q;
#pragma unroll
            for (int k = 0; k < kWords; k++) q[k] = w[k];
            *reinterpret_cast<words *>(static_cast<uint16_t *>(p) + e) = q;
        } else {
#pragma unroll
            for (int k = 0; k < kWords; k++) { h[2 * k] = (uint16_t)w[k]; h[2 * k + 1] = (uint16_t)(w[k] >> 16); }
        }
    }
    // the N elements from e on, wherever that is
    __device__ __forceinline__ void load_anywhere(const void *p, int64_t e)
    {
        typedef uint32_t words __attribute__((ext_vector_type(kWords), aligned(2)));
        const words q = *reinterpret_cast<const words *>(static_cast<const uint16_t *>(p) + e);
#pragma unroll
        for (int k = 0; k < kWords; k++) w[k] = q[k];
    }
    // the first `by` (0 .. N) elements dropped, zeros behind the others
    __device__ __forceinline__ void drop(int by)
    {
        drop_words(w, by >> 1);
#pragma unroll
        for (int k = 0; k < kWords; k++) w[k] = (by & 1) ? (w[k] >> 16) | (k + 1 < kWords ? w[k + 1] << 16 : 0u) : w[k];
    }
    __device__ __forceinline__ float get(int i) const
    {
        return (i & 1) ? __uint_as_float(w[i >> 1] & 0xffff0000u) : __uint_as_float(w[i >> 1] << 16);
    }
    __device__ __forceinline__ void set(const float (&t)[N])
    {
#pragma unroll
        for (int k = 0; k < kWords; k++) w[k] = f32x2_to_bf16x2(t[2 * k], t[2 * k + 1]);
    }
    __device__ __forceinline__ bool unit_interval() const
    {
        uint32_t m = w[0];
#pragma unroll
        for (int k = 1; k < kWords; k++) m = pk_max_u16(m, w[k]);
        return max(m & 0xffffu, m >> 16) <= 0x3f80u;
    }
    template <int W> __device__ __forceinline__ static void drop_words(uint32_t (&w)[W], int by) // by <= W
    {
#pragma unroll
        for (int step = 1; step <= W; step *= 2) {
#pragma unroll
            for (int k = 0; k < W; k++) w[k] = (by & step) ? (k + step < W ? w[k + step] : 0u) : w[k];
        }
    }
};

template <int N> struct RawPart<DQ_F32, N> {
    static constexpr int kCount = N, kWords = N;
    uint32_t w[N];
    __device__ __forceinline__ void zero()
    {
#pragma unroll
        for (int k = 0; k < N; k++) w[k] = 0u;
    }
    __device__ __forceinline__ void halves()
    {
#pragma unroll
        for (int k = 0; k < N; k++) w[k] = 0x3f000000u;
    }
    __device__ __forceinline__ uint32_t absmax_bits() const
    {
        uint32_t m = w[0] & 0x7fffffffu;
#pragma unroll
        for (int k = 1; k < N; k++) m = max(m, w[k] & 0x7fffffffu);
        return m;
    }
    __device__ __forceinline__ void load(const void *p, int64_t e, bool vec)
    {
        const volatile uint32_t *f = static_cast<const volatile uint32_t *>(p) + e;
        if (vec) {
            const uint4 *q = reinterpret_cast<const uint4 *>(static_cast<const uint32_t *>(p) + e);
#pragma unroll
            for (int k = 0; k < N / 4; k++) {
                const uint4 t = q[k];
                w[4 * k] = t.x; w[4 * k + 1] = t.y; w[4 * k + 2] = t.z; w[4 * k + 3] = t.w;
            }
        } else {
#pragma unroll
            for (int k = 0; k < N; k++) w[k] = f[k];
        }
    }
    __device__ __forceinline__ void store(void *p, int64_t e, bool vec) const
    {
        volatile uint32_t *f = static_cast<volatile uint32_t *>(p) + e;
        if (vec) {
            uint4 *q = reinterpret_cast<uint4 *>(static_cast<uint32_t *>(p) + e);
#pragma unroll
            for (int k = 0; k < N / 4; k++) q[k] = make_uint4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
        } else {
#pragma unroll
            for (int k = 0; k < N; k++) f[k] = w[k];
        }
    }
    __device__ __forceinline__ void load_anywhere(const void *p, int64_t e)
    {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4), aligned(4)));
        const u32x4 *q = reinterpret_cast<const u32x4 *>(static_cast<const uint32_t *>(p) + e);
#pragma unroll
        for (int k = 0; k < N / 4; k++) {
            const u32x4 t = q[k];
            w[4 * k] = t.x; w[4 * k + 1] = t.y; w[4 * k + 2] = t.z; w[4 * k + 3] = t.w;
        }
    }
    __device__ __forceinline__ void drop(int by) { RawPart<DQ_BF16, 4>::drop_words(w, by); }
    __device__ __forceinline__ float get(int i) const { return __uint_as_float(w[i]); }
    __device__ __forceinline__ void set(const float (&t)[N])
    {
#pragma unroll
        for (int k = 0; k < N; k++) w[k] = __float_as_uint(t[k]);
    }
    __device__ __forceinline__ bool unit_interval() const
    {
        uint32_t m = w[0];
#pragma unroll
        for (int k = 1; k < N; k++) m = max(m, w[k]);
        return m <= 0x3f800000u;
    }
};

// the lane's words of the chunk's block of the rounding stream
template <int N> struct RawPart<DQ_PHILOX, N> {
    static constexpr int kCount = N, kWords = N / 4;
    uint32_t w[kWords]; // with the lowest bit of every byte set
    __device__ __forceinline__ void zero()
    {
#pragma unroll
        for (int k = 0; k < kWords; k++) w[k] = 0x01010101u;
    }
    __device__ __forceinline__ void halves() { zero(); }
    // part `at` of the chunk's block, which every lane of the chunk makes
    __device__ __forceinline__ void generate(const RandKey &key, int64_t chunk, int at)
    {
        uint32_t all[4];
        chunk_uniform_words(key, chunk, all);
#pragma unroll
        for (int k = 0; k < kWords; k++) {
            uint32_t word = all[k];
#pragma unroll
            for (int p = 1; p < 16 / N; p++) word = at == p ? all[p * kWords + k] : word;
            w[k] = word | 0x01010101u;
            asm("" : "+v"(w[k]));
        }
    }
    __device__ __forceinline__ float odd_byte(int i) const { return (float)((w[i >> 2] >> (8 * (i & 3))) & 0xffu); }
    __device__ __forceinline__ float get(int i) const { return odd_byte(i) * 0.00390625f; }
    __device__ __forceinline__ bool unit_interval() const { return true; }
};
template <int N> struct DrawnBytes<RawPart<DQ_PHILOX, N>> { static constexpr bool value = true; };

// The words that the lanes of a chunk need for as many draws as they are, of which lane q makes the q-th, so that a draw costs a lane
// its share of a block: words N / 4 d and following of w for draw d.  Quads: word q of all four (a 4 x 4 transpose in two
// exchanges); pairs: words 2 q and 2 q + 1 of both.
template <int N> __device__ __forceinline__ void part_words(const RandKey &key, int64_t chunk, int lane, uint32_t (&w)[4])
{
    chunk_uniform_words(key, chunk, w);
#pragma unroll
    for (int k = 0; k < 4; k++) w[k] |= 0x01010101u;
    const bool odd = (lane & 1) != 0, high = (lane & 2) != 0;
    if constexpr (N == 8) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const uint32_t got = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(odd ? w[k] : w[k + 2]), 0xB1, 0xf, 0xf, true);
            w[k] = odd ? got : w[k];
            w[k + 2] = odd ? w[k + 2] : got;
        }
    } else {
#pragma unroll
        for (int k = 0; k < 4; k += 2) {
            const uint32_t got = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(odd ? w[k] : w[k + 1]), 0xB1, 0xf, 0xf, true);
            w[k] = odd ? got : w[k];
            w[k + 1] = odd ? w[k + 1] : got;
        }
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const uint32_t got = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(high ? w[k] : w[k + 2]), 0x4E, 0xf, 0xf, true);
            w[k] = high ? got : w[k];
            w[k + 2] = high ? w[k + 2] : got;
        }
    }
}

// maximum over the lanes of a chunk (N elements per lane), and over those of a superchunk of values that are alike within
// a chunk; the integer forms for patterns of positive finite floats
template <int N> __device__ __forceinline__ uint32_t chunk_max(uint32_t u)
{
    if (N <= 8) u = max(u, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)u, 0xB1, 0xf, 0xf, true)); // quad_perm [1,0,3,2]
    if (N == 4) u = max(u, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)u, 0x4E, 0xf, 0xf, true)); // quad_perm [2,3,0,1]
    return u;
}

template <int N> __device__ __forceinline__ float chunk_max(float v)
{
    if (N <= 8) v = __builtin_fmaxf(v, dpp_f32<0xB1>(v));
    if (N == 4) v = __builtin_fmaxf(v, dpp_f32<0x4E>(v));
    return v;
}

// the other row of a pair (lane bit 4) and, with FOUR, of the other half (lane bit 5): two rows that change places with themselves
// leave one of them in either register
template <bool FOUR, class F> __device__ __forceinline__ uint32_t across_rows(uint32_t u, F combine)
{
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(u, u, false, false));
    u = combine(a[0], a[1]);
    if (!FOUR) return u;
    const u32x2 b = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(u, u, false, false));
    return combine(b[0], b[1]);
}

template <int N> __device__ __forceinline__ float superchunk_max_pos(float v)
{
    if (N == 16) return row16_max_pos(v);
    uint32_t u = __float_as_uint(v);
    if (N == 8) u = max(u, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)u, 0x4E, 0xf, 0xf, true)); // quad_perm [2,3,0,1]
    u = max(u, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)u, 0x141, 0xf, 0xf, true)); // row_half_mirror
    u = max(u, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)u, 0x140, 0xf, 0xf, true)); // row_mirror
    return __uint_as_float(across_rows<N == 4>(u, [](uint32_t p, uint32_t q) { return max(p, q); }));
}

template <int N> __device__ __forceinline__ float superchunk_max(float v)
{
    if (N == 16) return row16_max(v);
    if (N == 8) v = __builtin_fmaxf(v, dpp_f32<0x4E>(v));
    v = __builtin_fmaxf(v, dpp_f32<0x141>(v));
    v = __builtin_fmaxf(v, dpp_f32<0x140>(v));
    return __uint_as_float(across_rows<N == 4>(__float_as_uint(v), [](uint32_t p, uint32_t q) {
        return __float_as_uint(__builtin_fmaxf(__uint_as_float(p), __uint_as_float(q)));
    }));
}

} // namespace dq
