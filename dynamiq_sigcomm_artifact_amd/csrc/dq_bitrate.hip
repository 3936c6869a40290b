// The search for the offset u of the dynamic bit-width rule
// (testbed_evaluation/new_comm_hooks/comm_hooks.py:73-139) without a pass over the norms per probe.
//
// The reference evaluates the average width at every probe of u with ten torch ops and a reduction over the
// norm tensors of all buckets, and reads the sum back to the host each time (up to 33 probes per search).
// The width of a superchunk depends on its norm only through the bf16 pattern, and as a function of the
// pattern it is a step function with two steps.  So:
//   norm_histogram_kernel   counts the norm patterns of a bucket's statistics into a histogram (one pass per
//                           bucket, accumulated over the buckets of a training step);
//   bitrate_search_kernel   one workgroup: keeps the histogram in LDS with a sum per 256 bins, then runs the reference's
//                           whole bisection (or its incremental correction) in double, each probe being two
//                           threshold searches over the patterns and two sums over a wave.
// The result (u, average width, target - average) equals what the torch ops of the reference give for the same
// norms: the counts are exact integers and the arithmetic of the search is the same IEEE double arithmetic.
#include "dq_bitwidth.cuh"
#include "dq_launch.h"

namespace dq {

namespace {

constexpr int kSearchThreads = 1024;
constexpr int kBinsPerThread = 32;             // 1024 x 32 = 32768 >= kNanBin + 1

__global__ __launch_bounds__(kHistThreads) void norm_histogram_kernel(const uint16_t *__restrict__ stats, int64_t nsc,
                                                                     uint32_t *__restrict__ hist)
{
    __shared__ uint32_t local[kHistWords];
    count_norm_patterns(stats, nsc, (int64_t)blockIdx.x * kHistBatch, (int64_t)gridDim.x * kHistBatch, hist, local);
}

// What bounds the search: one workgroup, so everything is a latency.  The histogram (128 KB) comes in as eight coalesced
// 16-byte loads per thread -- 32 consecutive bins per thread fetched every line eight times over -- and lands in LDS as it
// is, with a sum per 256 bins beside it; a count of the norms from a pattern on is then one more sum over a wave.  (Suffix
// counts of all bins, by shuffles, for the two that a converged correction looks at: 9.1 us instead of 5.0.)  A round of
// probes asks for up to eight values of u at once,
// one pair of waves each: the seven midpoints of the next three steps of the bisection, or the next eight corrections, which
// all follow from the first probe's deficit.  The walk through them is the reference's, probe by probe.  The first round's
// thresholds are found while the histogram is on its way, those of a correction by all waves in one round of 0.5 us (three rounds in two
// waves: 1.2).  What is left of 4.0 us (4.8 with zeros written over zeros, and summed): 2.9 until one CU has the 128 KB.
constexpr int kBins = 32768;                     // >= kNanBin + 1
constexpr int kSlabs = kBins / (4 * kSearchThreads);
constexpr int kSearchWaves = kSearchThreads / 64;
constexpr int kProbes = kSearchWaves / 2;        // values of u per round
static_assert(kBins == kSearchThreads * kBinsPerThread, "the histogram's size is part of the interface");

struct Probe {
    double avg, delta;
};

// the sum over the wave
__device__ __forceinline__ uint32_t wave_sum(uint32_t x)
{
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false); // row_shr:1, 2, 4, 8
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false); // row_bcast:15 into rows 1 and 3
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false); // row_bcast:31 into rows 2 and 3
    return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

// out[0..2] = u, average width, target - average; out[3] = number of probes.  hist: pattern counts in, zeros out.
// prev_u_dev != nullptr: the starting point of the correction is *prev_u_dev (it may be out[0] of the previous search)
__global__ __launch_bounds__(kSearchThreads) void bitrate_search_kernel(uint32_t *__restrict__ hist, int mode, double prev_u,
                                                                       const double *prev_u_dev, double target,
                                                                       double *out)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t bins[]; // the histogram, numbers only
    __shared__ __attribute__((aligned(8))) uint32_t part[kSlabs][kSearchWaves];
    __shared__ uint32_t nans;
    __shared__ uint32_t at_least[2][kProbes]; // norms of width >= 4, >= 8
    __shared__ __attribute__((aligned(16))) uint32_t below[2][kProbes]; // patterns of the window below the width
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;

    // (the first load, without a branch in front of the others; read by every thread long before thread 0 writes out[])
    const double read_u = *(prev_u_dev ? prev_u_dev : &kNoOffset);
    uint4 v[kSlabs]; // bins 4 (t + 1024 k) ..
    const bool whole = (reinterpret_cast<uintptr_t>(hist) & 15) == 0;
    if (whole) {
        const uint4 *h4 = reinterpret_cast<const uint4 *>(hist);
#pragma unroll
        for (int k = 0; k < kSlabs; k++) v[k] = h4[t + kSearchThreads * k];
    } else {
#pragma unroll
        for (int k = 0; k < kSlabs; k++) {
            const uint32_t *h = hist + 4 * (t + kSearchThreads * k);
            v[k] = make_uint4(h[0], h[1], h[2], h[3]);
        }
    }
    if (prev_u_dev) prev_u = read_u;
    // the thresholds of a value of u, for the wave's share of them; they need nothing of the histogram, so those of the first
    // round are found while it is on its way
    const double u_min = -10.0, u_max = 60.0, tol = 0.1;
    const int pair = wave >> 1;
    const auto find = [&](double mine) {
        return width_threshold((float)mine, lane, (wave & 1) ? 8 : 4);
    };
    // the midpoint of this pair's node below [l, h]
    const auto node_mid = [&](double l, double h) {
        double mid = (l + h) * 0.5;
        for (int bit = pair >= 4 ? 1 : (pair >= 2 ? 0 : -1); bit >= 0; bit--) { // from the root down
            if ((pair >> bit) & 1) h = mid;
            else l = mid;
            mid = (l + h) * 0.5;
        }
        return mid;
    };
    const double start = __builtin_fmax(u_min, __builtin_fmin(u_max, prev_u));
    // A correction's first probe is one value of u for all waves: eight of them look at 64 patterns each around either estimate, in one round.
    int p_first = 0, window = 0;
    if (mode == 0) {
        p_first = find(pair == 0 ? u_max : node_mid(u_min, u_max));
    } else {
        const int64_t width = (wave & 1) ? 8 : 4;
        window = min(max(width_near((float)start, width) - 256, 0), kMaxPattern - 511);
        const uint64_t under = __builtin_amdgcn_ballot_w64(qbits_of_norm((uint32_t)(window + 64 * pair + lane), (float)start) < width);
        if (lane == 0) below[wave & 1][pair] = (uint32_t)__popcll(under);
    }
#pragma unroll
    for (int k = 0; k < kSlabs; k++) {
        // Of the 128 times 256 bins most are empty, and nothing is done for those: no zeros to memory or to LDS, no sum over the wave.
        const int p = 4 * (t + kSearchThreads * k);
        const bool some = (v[k].x | v[k].y | v[k].z | v[k].w) != 0u;
        uint32_t sum = 0;
        if (p == kMaxPattern) nans = v[k].y;
        if (__builtin_amdgcn_ballot_w64(some) != 0) {
            if (some) { // (read, then left zeroed for the next accumulation)
                uint32_t *h = hist + p;
                if (whole)
                    *reinterpret_cast<uint4 *>(h) = make_uint4(0u, 0u, 0u, 0u);
                else
                    h[0] = h[1] = h[2] = h[3] = 0u;
            }
            static_assert(kMaxPattern % 4 == 0 && kNanBin == kMaxPattern + 1, "infinity and the NaN norms share a load");
            if (p >= kMaxPattern) v[k] = make_uint4(p == kMaxPattern ? v[k].x : 0u, 0u, 0u, 0u);
            reinterpret_cast<uint4 *>(bins)[t + kSearchThreads * k] = v[k];
            sum = wave_sum(v[k].x + v[k].y + v[k].z + v[k].w);
        }
        if (lane == 0) part[k][wave] = sum;
    }
    __syncthreads();
    if (mode != 0 && pair == 0) {
        static_assert(kProbes == 8, "the window's 512 patterns");
        const uint4 b0 = reinterpret_cast<const uint4 *>(below[wave & 1])[0], b1 = reinterpret_cast<const uint4 *>(below[wave & 1])[1];
        const int count = __builtin_amdgcn_readfirstlane((int)(b0.x + b0.y + b0.z + b0.w + b1.x + b1.y + b1.z + b1.w));
        p_first = window + count;
        if (!((count > 0 || window == 0) && (count < 512 || window + 511 == kMaxPattern)))
            p_first = width_threshold_anywhere((float)start, lane, (wave & 1) ? 8 : 4);
    }
    // entry (k, w) of part is the sum of the 256 bins from 256 (16 k + w) on; lane l of each wave holds entries 2 l and 2 l + 1
    static_assert(kSlabs * kSearchWaves == 128, "two entries per lane");
    const uint2 entries = reinterpret_cast<const uint2 *>(&part[0][0])[lane];
    const uint64_t total = (uint64_t)wave_sum(entries.x + entries.y) + nans;
    // norms of pattern >= p: the entries behind p's, and what lies in p's own
    const auto count_from = [&](int p) {
        if (p > kMaxPattern) return 0u;
        const int e = __builtin_amdgcn_readfirstlane(p >> 8), first = 4 * lane, from = p & 255;
        uint32_t sum = (2 * lane > e ? entries.x : 0u) + (2 * lane + 1 > e ? entries.y : 0u);
        // (an empty entry's bins are not in the LDS)
        if (__builtin_amdgcn_readlane((int)((e & 1) ? entries.y : entries.x), e >> 1) != 0) {
            const uint4 q = reinterpret_cast<const uint4 *>(bins)[64 * e + lane];
            sum += (first >= from ? q.x : 0u) + (first + 1 >= from ? q.y : 0u);
            sum += (first + 2 >= from ? q.z : 0u) + (first + 3 >= from ? q.w : 0u);
        }
        return wave_sum(sum);
    };

    // every thread evaluates the same doubles, so the control flow below is uniform without a broadcast
    int probes = 0;
    // one round: waves 2 k and 2 k + 1 hold the thresholds of candidate k
    const auto publish = [&](int p, bool again) {
        if (again) __syncthreads(); // the previous round has been read
        const uint32_t n = count_from(p);
        if (lane == 0) at_least[wave & 1][wave >> 1] = n;
        __syncthreads();
    };
    const auto result = [&](int k) {
        const uint64_t n4 = at_least[0][k], n8 = at_least[1][k];
        probes++;
        Probe r;
        r.avg = total ? (double)(2 * total + 2 * n4 + 4 * n8) / (double)total : 0.0;
        r.delta = target - r.avg;
        return r;
    };
    double res_u, res_avg, res_delta;
    if (mode == 0) {
        // comm_hooks.py:94-114.  A round holds the nodes 1 .. 7 of the tree of the next three midpoints (node h: below it
        // 2 h when low rises to it, 2 h + 1 when high falls to it); pair 0 of the first round holds the upper end.
        double low = u_min, high = u_max, best_u = high, best_avg = 0.0, best_delta = 0.0;
        bool done = false, first = true;
        for (int it = 0; it < 32 && !done;) {
            publish(first ? p_first : find(pair == 0 ? high : node_mid(low, high)), !first);
            if (first) {
                const Probe r = result(0);
                best_avg = r.avg;
                best_delta = r.delta;
                first = false;
            }
            int node = 1;
            for (int level = 0; level < 3 && it < 32 && !done; level++, it++) {
                const double m = (low + high) * 0.5;
                const Probe r = result(node);
                if (__builtin_fabs(r.delta) < __builtin_fabs(best_delta)) {
                    best_u = m; best_avg = r.avg; best_delta = r.delta;
                }
                if (__builtin_fabs(r.delta) <= tol) {
                    best_u = m; best_avg = r.avg; best_delta = r.delta;
                    done = true;
                } else if (r.delta > 0) {
                    low = m;
                    node = 2 * node;
                } else {
                    high = m;
                    node = 2 * node + 1;
                }
            }
        }
        res_u = best_u; res_avg = best_avg; res_delta = best_delta;
    } else {
        // comm_hooks.py:117-139
        publish(p_first, false);
        Probe r = result(0);
        res_u = start; res_avg = r.avg; res_delta = r.delta;
        if (!(__builtin_fabs(r.delta) <= tol)) {
            const double old_delta = r.delta;
            double step = old_delta;
            bool done = false;
            for (int it = 0; it < 32 && !done; it += kProbes) {
                double mine = step;
                for (int k = 0; k < pair; k++) mine *= 0.5;
                publish(find(__builtin_fmax(u_min, __builtin_fmin(u_max, start + mine))), true);
                for (int k = 0; k < kProbes && !done; k++) {
                    const double cand = __builtin_fmax(u_min, __builtin_fmin(u_max, start + step));
                    r = result(k);
                    if (__builtin_fabs(r.delta) < __builtin_fabs(res_delta)) {
                        res_u = cand; res_avg = r.avg; res_delta = r.delta;
                    }
                    if (__builtin_fabs(r.delta) <= tol || old_delta * r.delta >= 0) {
                        res_u = cand; res_avg = r.avg; res_delta = r.delta;
                        done = true;
                    }
                    step *= 0.5;
                }
            }
        }
    }
    if (t == 0) {
        out[0] = res_u; out[1] = res_avg; out[2] = res_delta; out[3] = (double)probes;
    }
}

} // namespace

int64_t bitrate_hist_ints() { return (int64_t)kSearchThreads * kBinsPerThread; }

hipError_t launch_norm_histogram(const void *stats, int64_t nsc, uint32_t *hist, hipStream_t stream)
{
    const unsigned grid = (unsigned)std::min<int64_t>((nsc + kHistBatch - 1) / kHistBatch, 1024);
    hipLaunchKernelGGL(norm_histogram_kernel, dim3(grid), dim3(kHistThreads), 0, stream, static_cast<const uint16_t *>(stats), nsc,
                       hist);
    return hipGetLastError();
}

hipError_t launch_bitrate_search(uint32_t *hist, int mode, double prev_u, const double *prev_u_dev, double target, double *out,
                                 hipStream_t stream)
{
    constexpr int lds = kBins * (int)sizeof(uint32_t);
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(bitrate_search_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(bitrate_search_kernel, dim3(1), dim3(kSearchThreads), lds, stream, hist, mode, prev_u, prev_u_dev, target,
                       out);
    return hipGetLastError();
}

} // namespace dq
