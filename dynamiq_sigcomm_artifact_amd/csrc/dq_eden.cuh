// EDEN's quantiser on the sixteen consecutive elements of a thread, and the fixed association of its sums: shared by the
// kernels of long slices (dq_eden.hip) and the one of short slices (dq_eden_short.hip).
#pragma once

#include "dq_sums.cuh"
#include "dq_tile16.cuh"

namespace dq {

constexpr int kEdenThreads = 256;
constexpr int kEdenPerThread = 16;
constexpr int kEdenTile = kEdenThreads * kEdenPerThread; // 4096 elements
constexpr int64_t kEdenFoldTiles = 1024;                 // the most tiles whose sums are folded inside other launches

__host__ __device__ inline int64_t eden_tiles(int64_t n) { return (n + kEdenTile - 1) / kEdenTile; }

// sum[l] += sum[l + stride], stride 128 .. 1, over 256 values, one per thread; returns the total in every thread.  t: 0 .. 255,
// lds: 256 doubles of the group's own.  The strides of 128 and 64 meet in LDS, the others inside the first wave, in the same
// order of additions: three barriers instead of ten, and no trips through the LDS crossbar in between.
__device__ __forceinline__ double fold256_of(double *lds, int t) // of the 256 values in lds
{
    __syncthreads();
    if (t < 64) {
        double s = (lds[t] + lds[t + 128]) + (lds[t + 64] + lds[t + 192]);
        s = add_across_f64<32>(s);
        s = add_across_f64<16>(s);
        s = halve_row_f64(s);
        if (t == 0) lds[0] = s;
    }
    __syncthreads();
    const double total = lds[0];
    __syncthreads();
    return total;
}

__device__ __forceinline__ double fold256(double v, double *lds, int t)
{
    lds[t] = v;
    return fold256_of(lds, t);
}

// The boundaries sit in LDS in breadth-first order of the search tree (node 1 = the middle boundary, children of node i at
// 2 i and 2 i + 1): the lanes of a wave read one level of the tree at a time, consecutive words, where the sorted layout
// puts a whole level into a few banks.
template <int NBITS>
__device__ __forceinline__ void eden_tables(const float *__restrict__ boundaries, const float *__restrict__ centroids, float *tree,
                                            float *cen, int tid, int nthreads)
{
    constexpr int L = 1 << NBITS;
    for (int k = tid; k < L; k += nthreads) {
        cen[k] = centroids[k];
        if (k < L - 1) {
            // sorted position k = (2 r + 1) 2^(NBITS - 1 - level) - 1 is node 2^level + r
            const int tz = __builtin_ctz(k + 1);
            tree[(1 << (NBITS - 1 - tz)) + ((k + 1) >> (tz + 1))] = boundaries[k];
        }
    }
}

// bins of the thread's sixteen (eight) elements v, its half word (byte) of every bit plane to `piece` (null: not stored; a plane
// has `words` words), and the sum of centroid * element over sixteen elements in ascending order -- with eight per thread, in the
// odd thread of the two that have them
template <int NBITS, int PER>
__device__ __forceinline__ double eden_bins_of(const float (&v)[PER], float norm, float sqrt_n, const float *tree, const float *cen,
                                               uint8_t *piece, int64_t words)
{
    static_assert(PER == 16 || PER == 8, "a half word or a byte of every plane");
    constexpr int L = 1 << NBITS;
    const uint32_t nb = __float_as_uint(norm);
    const bool ordinary = nb >= 0x0d800000u && nb <= 0x71800000u; // uniform over the slice
    const double yn = ordinary ? recip_f64(norm) : 0.0;
    float x[PER];
    int node[PER];
    if (ordinary) {
#pragma unroll
        for (int k = 0; k < PER; k++) x[k] = div_exact(v[k] * sqrt_n, norm, yn);
    } else {
#pragma unroll
        for (int k = 0; k < PER; k++) x[k] = (v[k] * sqrt_n) / norm;
    }
    // the sixteen searches advance level by level: sixteen independent LDS reads per level; node[] holds the
    // node's byte offset into the table
#pragma unroll
    for (int k = 0; k < PER; k++) node[k] = 4;
#pragma unroll
    for (int level = 0; level < NBITS; level++) {
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const float b = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(tree) + node[k]);
            node[k] = 2 * node[k] + (!(b >= x[k]) ? 4 : 0); // torch's lower bound: a NaN goes right at every level
        }
    }
    // the product of two floats is exact in double, so the fused multiply-add rounds like multiply, then add
    double acc = 0.0;
    float c[PER];
    uint32_t four[PER / 4];
#pragma unroll
    for (int q = 0; q < PER / 4; q++) four[q] = 0;
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const uint32_t off = (uint32_t)(node[k] - 4 * L); // 4 * bin
        c[k] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(cen) + off);
        acc = __builtin_fma((double)c[k], (double)v[k], acc);
        four[k >> 2] |= (k & 3) ? off << (8 * (k & 3) - 2) : off >> 2;
    }
    const uint64_t lo8 = transpose8x8((uint64_t)four[0] | ((uint64_t)four[1] << 32));
    if constexpr (PER == 16) {
        const uint64_t hi8 = transpose8x8((uint64_t)four[2] | ((uint64_t)four[3] << 32));
        if (piece) {
            uint16_t *half = reinterpret_cast<uint16_t *>(piece);
#pragma unroll
            for (int p = 0; p < NBITS; p++)
                half[(int64_t)p * words * 2] = (uint16_t)(((lo8 >> (8 * p)) & 0xffu) | (((hi8 >> (8 * p)) & 0xffu) << 8));
        }
    } else {
        if (piece) {
#pragma unroll
            for (int p = 0; p < NBITS; p++) piece[(int64_t)p * words * 4] = (uint8_t)(lo8 >> (8 * p));
        }
        // the even thread's sum goes on with the odd one's elements
        const uint64_t b = (uint64_t)__double_as_longlong(acc);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, 0xA0, 0xf, 0xf, true); // quad_perm [0,0,2,2]
        const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), 0xA0, 0xf, 0xf, true);
        acc = __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
#pragma unroll
        for (int k = 0; k < PER; k++) acc = __builtin_fma((double)c[k], (double)v[k], acc);
    }
    return acc;
}

} // namespace dq
