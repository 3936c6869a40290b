// The dynamic bit-width rule on the device (testbed_evaluation/new_comm_hooks/comm_hooks.py:64-70) and the two
// norm patterns at which the width changes, shared by the group plan and the search for the offset u.
#pragma once

#include "dq_device.cuh"

namespace dq {

// What stands in for an offset that is a number of the launch and not in device memory, where it is loaded all the same: behind a branch, the
// loads that follow would only leave when the offset has arrived.
static __device__ double kNoOffset = 0.0; // (never written; a constant would lie in another address space and make the load one of either)

__device__ __forceinline__ float round_bf16(float x) { return bf16_bits_to_f32(f32_to_bf16_bits(x)); }

// testbed_evaluation/new_comm_hooks/comm_hooks.py:64-70 on a bf16 norm: every torch op computes in
// binary32 and rounds its result to bf16
__device__ __forceinline__ int64_t qbits_of_norm(uint32_t norm_bits, float u)
{
    const float eps = 1e-20f;
    float x = bf16_bits_to_f32(norm_bits);
    x = (x != x) ? x : round_bf16(x > eps ? x : eps);
    x = round_bf16(log2_det(x));
    x = round_bf16(x * (float)(4.0 / (512.0 / 17.0)));
    x = round_bf16(x + u);
    x = (x != x) ? x : round_bf16(x > eps ? x : eps);
    x = round_bf16(log2_det(x));
    x = __builtin_floorf(x);
    int z = (x != x) ? 1 : (x < 1.0f ? 1 : (x > 3.0f ? 3 : (int)x));
    return (int64_t)1 << z;
}

// The same width as a class (0: 8 bits, 1: 4, 2: 2) for all lanes of a wave, most of the time without the rule's seventy
// instructions: the score s = scale log2(F) + u decides (below 4: 2 bits, below 8: 4, else 8) unless it lies near 4 or 8.
// The rule rounds to bf16 four times in front of its comparison with 4 or 8 (F is bf16 already): log2 F to 2^-9 of at most
// 67 for the F taken here, times the scale 0.133 -> 0.018; the product, at most 8.9, to 2^-9 of it -> 0.018; the sum near
// 8 -> 0.016; and the second log2, of a number near 8, rounds to 3 from 2^-8 below -> a factor 2^(1/256) of s, 0.022.
// Together 0.074; the hardware's log2 and the products here add less than 1e-4.  A band of 0.125 is kept.
__device__ __forceinline__ int width_class_of_norm(uint32_t norm_bits, float u)
{
    const float f = bf16_bits_to_f32(norm_bits);
    const float s = __builtin_fmaf(__builtin_amdgcn_logf(f), (float)(4.0 / (512.0 / 17.0)), u);
    const float off = __builtin_fminf(__builtin_fabsf(s - 4.0f), __builtin_fabsf(s - 8.0f));
    // (NaN fails both comparisons)
    if (__builtin_amdgcn_ballot_w64(!(f >= 0x1p-60f && f <= 0x1p60f && off >= 0.125f)) == 0) return s < 4.0f ? 2 : (s < 8.0f ? 1 : 0);
    const int64_t q = qbits_of_norm(norm_bits, u);
    return q == 8 ? 0 : (q == 4 ? 1 : 2);
}

constexpr int kMaxPattern = 0x7f80; // +infinity: the patterns 0 .. 0x7f80 are the non-negative norms in ascending order

// The width is a monotone step function of the bf16 norm pattern (every operation of the rule is monotone, and
// neighbouring bf16 values are 2^-8 apart, far more than the error of the log2 polynomial), so two patterns
// describe it for a given u.
// index of the first of 64 probes lo + step * (l + 1) (clamped to kMaxPattern) whose width is >= target; 64 if none
__device__ __forceinline__ int first_width_probe(float u, int lo, int step, int lane, int64_t target)
{
    const int p = min(lo + step * (lane + 1), kMaxPattern);
    const uint64_t hit = __builtin_amdgcn_ballot_w64(qbits_of_norm((uint32_t)p, u) >= target);
    return hit ? __builtin_ctzll(hit) : 64;
}

// Where the score scale log2(F) + u of the rule is the target.  The rule changes its width within 0.074 of there (width_class_of_norm), 71
// patterns.  (A NaN gives some pattern, as does what lies beyond binary32: who starts here looks at the widths around it.)
__device__ __forceinline__ int width_near(float u, int64_t target)
{
    return (int)(__float_as_uint(__builtin_amdgcn_exp2f(((float)target - u) * (float)(512.0 / 17.0 / 4.0))) >> 16) & 0x7fff;
}

// The smallest pattern of width >= target (kMaxPattern + 1: none), for one wave, from anywhere: three rounds of probes
__device__ __forceinline__ int width_threshold_anywhere(float u, int lane, int64_t target)
{
    const int a = first_width_probe(u, -1, 512, lane, target);
    if (a >= 64) return kMaxPattern + 1;
    const int from = -1 + 512 * a, next = from + 8 * first_width_probe(u, from, 8, lane, target);
    return next + 1 + first_width_probe(u, next, 1, lane, target);
}

// The same: two rounds, a round being a chain of 0.4 us, on the 256 patterns around the estimate; three where it is not there
__device__ __forceinline__ int width_threshold(float u, int lane, int64_t target)
{
    const int lo = min(max(width_near(u, target) - 128, 0), kMaxPattern - 255);
    const int a = first_width_probe(u, lo - 1, 4, lane, target); // patterns lo + 3, lo + 7, ..
    if (a < 64 || lo + 255 == kMaxPattern) {
        if (a >= 64) return kMaxPattern + 1;
        const int from = lo + 4 * a; // one of from .. from + 3 is the first, unless it is even before those
        const int f = first_width_probe(u, max(from - 2, -1), 1, lane, target);
        if (f > 0 || from == 0) return max(from - 1, 0) + f;
    }
    return width_threshold_anywhere(u, lane, target);
}

// wave 0 finds thr[0] = the smallest pattern of width >= 4, wave 1 thr[1] = that of width 8
// (kMaxPattern + 1 when no pattern reaches it); other waves do nothing.  No barrier inside.
__device__ __forceinline__ void width_thresholds(float u, int *thr, int wave, int lane)
{
    if (wave > 1) return;
    const int t = width_threshold(u, lane, wave == 0 ? 4 : 8);
    if (lane == 0) thr[wave] = t;
}

// ---- histogram of the norm patterns (what the search for u works on) ----------------------------------

constexpr int kNanBin = kMaxPattern + 1; // NaN norms: 2 bits whatever u is

// negative norms (and -0) are clamped to the same epsilon as +0: bin 0
__device__ __forceinline__ int bin_of(uint32_t pattern)
{
    if (pattern <= (uint32_t)kMaxPattern) return (int)pattern;
    return (pattern & 0x7fffu) > (uint32_t)kMaxPattern ? kNanBin : 0;
}

// the largest of the wave's values, in lane 63
__device__ __forceinline__ uint32_t wave_max_upward(uint32_t x)
{
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false)); // row_shr:1, 2, 4, 8
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false)); // row_bcast:15 into rows 1 and 3
    return max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false)); // row_bcast:31 into rows 2 and 3
}

// the sum of the wave's values, in lane 63
__device__ __forceinline__ uint32_t wave_sum_upward(uint32_t x)
{
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);
    return x + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);
}

// A workgroup of kHistThreads threads counts batches of up to 8192 norms in LDS -- 16-bit counters, two per word,
// so the whole range of patterns fits into 64 KB -- and adds the non-zero counters to the histogram in memory
// after each batch: a few hundred atomics per batch instead of one per norm, most of which would hit the same
// few hundred words.  The workgroup takes the batches first, first + stride, ...; local: kHistWords words of LDS.
constexpr int kHistThreads = 1024;
constexpr int kHistBatch = 8192; // norms per batch (a 16-bit counter holds up to 65535)
constexpr int kHistWords = 16384; // 32768 counters

__device__ __forceinline__ void count_norm_patterns(const uint16_t *__restrict__ stats, int64_t nsc, int64_t first,
                                                    int64_t stride, uint32_t *__restrict__ hist, uint32_t *local)
{
    const int t = threadIdx.x;
    for (int64_t batch0 = first; batch0 < nsc; batch0 += stride) {
        for (int w = t; w < kHistWords; w += kHistThreads) local[w] = 0u;
        __syncthreads();
        const int64_t end = min(batch0 + kHistBatch, nsc);
        for (int64_t i = batch0 + t; i < end; i += kHistThreads) {
            const int bin = bin_of(stats[2 * i + 1]);
            atomicAdd(&local[bin >> 1], 1u << (16 * (bin & 1)));
        }
        __syncthreads();
        for (int w = t; w < kHistWords; w += kHistThreads) {
            const uint32_t pair = local[w];
            if (pair & 0xffffu) atomicAdd(&hist[2 * w], pair & 0xffffu);
            if (pair >> 16) atomicAdd(&hist[2 * w + 1], pair >> 16);
        }
        __syncthreads();
    }
}

} // namespace dq
