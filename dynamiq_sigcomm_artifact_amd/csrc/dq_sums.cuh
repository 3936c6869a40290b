// Sums of doubles over registers and lanes in a fixed order, and the order of EDEN's sums of squares.
#pragma once

#include <type_traits>

#include "dq_device.cuh"

namespace dq {

// EDEN's sum of the squares of n = 2^k >= 2^14 elements (other n: dq_eden.hip).  Element e has the row t = e / (n / 16), 0 .. 15,
// and lies at column l = e % 32 of piece p = e / 32 % (n / 512).  The squares of a piece are halved over its rows (t += t + 8,
// t + 4, t + 2, t + 1), then its columns are added, neighbours first (l += l + 1, l + 2, .. l + 16), and the n / 512 sums of the
// pieces are halved to one (p += p + n / 1024, .. p + 1).  A pass over the vector by rows far apart can add in this order, whatever
// number of rows from 16 on its tiles have, as well as one over consecutive elements: the bits are those of the vector alone.
constexpr int64_t kRowSumsFrom = (int64_t)1 << 14;
__host__ __device__ inline bool sums_by_rows(int64_t n) { return n >= kRowSumsFrom && (n & (n - 1)) == 0; }

// x of lane l + SHIFT of the row (0 beyond it)
template <int SHIFT> __device__ __forceinline__ double row_shift_f64(double x)
{
    const uint64_t b = (uint64_t)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, 0x100 + SHIFT, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), 0x100 + SHIFT, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// sum[l] += sum[l + 32], then sum[l + 16] (LANES), of the lanes below that
template <int LANES> __device__ __forceinline__ double add_across_f64(double x)
{
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    const uint64_t b = (uint64_t)__double_as_longlong(x);
    const auto both = [](uint32_t w) { // what the lower lanes hold, and what the upper ones hold, in both
        return LANES == 16 ? __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(w, w, false, false))
                           : __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(w, w, false, false));
    };
    const u32x2 lo = both((uint32_t)b), hi = both((uint32_t)(b >> 32));
    return __longlong_as_double((long long)(((uint64_t)hi[0] << 32) | lo[0])) + __longlong_as_double((long long)(((uint64_t)hi[1] << 32) | lo[1]));
}

// the first of 16 lanes: sum[l] += sum[l + 8], + 4, + 2, + 1 (lanes beyond the stride add what nobody reads)
__device__ __forceinline__ double halve_row_f64(double s)
{
    s += row_shift_f64<8>(s);
    s += row_shift_f64<4>(s);
    s += row_shift_f64<2>(s);
    s += row_shift_f64<1>(s);
    return s;
}

__device__ __forceinline__ double first_lane_f64(double x)
{
    const uint64_t b = (uint64_t)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// x[i] += x[i + N / 2], .. x[i + 1]
template <int N> __device__ __forceinline__ double halve(double (&x)[N])
{
#pragma unroll
    for (int stride = N / 2; stride > 0; stride >>= 1) {
#pragma unroll
        for (int i = 0; i < N; i++)
            if (i < stride) x[i] += x[i + stride];
    }
    return x[0];
}

// halve the squares of w[0], w[STEP], .. (exact in double, so that the first level is a fused multiply-add)
template <int STEP = 1, int R> __device__ __forceinline__ double halve_squares(const float (&w)[R], int first = 0)
{
    constexpr int N = R / STEP;
    if constexpr (N == 1) {
        return (double)w[first] * (double)w[first];
    } else {
        double x[N / 2];
#pragma unroll
        for (int i = 0; i < N / 2; i++) {
            const double a = (double)w[first + STEP * i], b = (double)w[first + STEP * (i + N / 2)];
            x[i] = __builtin_fma(b, b, a * a);
        }
        return halve(x);
    }
}

// the sum over the lane's half of the wave, neighbours first, in every lane of it
__device__ __forceinline__ double sum_columns_f64(double x)
{
    const auto add_from = [&](auto ctrl) {
        const uint64_t b = (uint64_t)__double_as_longlong(x);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, decltype(ctrl)::value, 0xf, 0xf, true);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), decltype(ctrl)::value, 0xf, 0xf, true);
        x += __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
    };
    add_from(std::integral_constant<int, 0xB1>());  // quad_perm [1,0,3,2]
    add_from(std::integral_constant<int, 0x4E>());  // quad_perm [2,3,0,1]
    add_from(std::integral_constant<int, 0x141>()); // row_half_mirror
    add_from(std::integral_constant<int, 0x140>()); // row_mirror
    return add_across_f64<16>(x);
}

} // namespace dq
