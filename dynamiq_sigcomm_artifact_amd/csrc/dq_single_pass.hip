// The compressed all-reduce of a bucket without a packed stream in memory.
//
// Where all ranks of a ring live in one GPU's memory -- a ring of one rank, or W simulated ones -- the records that a
// ring step writes are read back by the next step's launch and by nobody else.  A superchunk's way through the ring
// touches no other superchunk: compress on the first rank, decode + add + recompress on each of the others, decode on
// all.  So a wave takes a tile of four superchunks and runs that whole chain in registers (dq_widths.cuh: the levels
// of a chunk instead of its bits), reading every rank's elements once and writing every rank's result once.
//
//   roundtrip_kernel   one rank: statistics, width, centring, compress, decompress, mean add -- one pass over the
//                      bucket, and up to kMaxBuckets buckets per launch
//   tally_kernel       behind it: the widths' counts per bucket and the norm histogram of the search for u
//   ranks_stats_kernel W ranks: every rank's means, and the reduced statistics
//   ring_kernel        W ranks, after a plan of the reduced statistics: the ring
//   ring_parts_kernel  the same on short vectors, one or two superchunks per wave; with drawn values it does without the plan
//
// Measured, start -> now (bit-identical results): 8 ranks x 124,439,808 bf16 elements 2,896 -> 1,070 us per all-reduce (one
// launch per rank and ring step, packed streams and their exchange copies, against three launches whose traffic is the
// vectors alone), 8 x 1,000,003 elements 1,488 -> 20 us (257 launches against 2), a step of nine 25 MB buckets on one rank
// 252 -> 50 us (four launches per bucket on two streams against two launches per step, and the search for u).
//
// Numerics: csrc/cuda_hadamard.cu:1257-1369 (centring, mean add), csrc/cuda_hierarchical_mee.cu:203-696 (codec),
// testbed_evaluation/new_comm_hooks/ring_rdma.py:590-631 (order of the ring), comm_hooks.py:64-70 (widths).
#include <stddef.h>
#include <string.h>

#include <type_traits>

#include "dq_widths.cuh"
#include "dq_bitwidth.cuh"
#include "dq_launch.h"

namespace dq {

namespace {

// the tile's values leave as whole superchunks: through LDS (slots swizzled), then contiguous 16-byte streaming stores.
// sc: the superchunk of this lane's row; stage holds 64 * kSlots 16-byte slots of this wave.
template <int DT> __device__ __forceinline__ void stage_tile(const Raw16<DT> &out, uint4 *stage, int lane)
{
    constexpr int S = Raw16<DT>::kSlots;
#pragma unroll
    for (int k = 0; k < S; k++) stage[swz(S * lane + k)] = out.slot(k);
    wave_lds_sync();
}

template <int DT>
__device__ __forceinline__ void store_tile(void *dst, const Raw16<DT> &out, const uint4 *stage, int64_t sc, int rows_here, int64_t n,
                                           bool vec, int lane)
{
    constexpr int S = Raw16<DT>::kSlots;
    constexpr int ESZ = DT == DQ_F32 ? 4 : 2;
    constexpr int EP = 16 / ESZ;
    char *bytes = static_cast<char *>(dst);
    if (vec) {
#pragma unroll
        for (int k = 0; k < S; k++) {
            const int s = 64 * k + lane;
            const int row = s / (16 * S);
            const int64_t e = (int64_t)__shfl((int)sc, row * 16, 64) * 256 + (s % (16 * S)) * EP;
            if (row < rows_here) {
                const uint4 val = stage[swz(s)];
                if (e + EP <= n) {
                    stream_store(reinterpret_cast<uint4 *>(bytes + e * ESZ), val);
                } else {
                    const uint32_t part[4] = {val.x, val.y, val.z, val.w};
                    const int left = left_here(n, e, EP);
#pragma unroll
                    for (int i = 0; i < EP; i++) {
                        if (i < left) {
                            if (DT == DQ_F32)
                                reinterpret_cast<uint32_t *>(bytes)[e + i] = part[i];
                            else
                                reinterpret_cast<uint16_t *>(bytes)[e + i] = (uint16_t)(part[i >> 1] >> (16 * (i & 1)));
                        }
                    }
                }
            }
        }
    } else if ((lane >> 4) < rows_here) {
        const int64_t e = sc * 256 + (lane & 15) * 16;
        const int left = left_here(n, e, 16);
#pragma unroll
        for (int i = 0; i < 16; i++) {
            if (i < left) {
                if (DT == DQ_F32)
                    reinterpret_cast<uint32_t *>(bytes)[e + i] = out.w[i];
                else
                    reinterpret_cast<uint16_t *>(bytes)[e + i] = (uint16_t)(out.w[i >> 1] >> (16 * (i & 1)));
            }
        }
    }
}

// T(T(level * step) + mean)
template <int DT, class RV> __device__ __forceinline__ void decode_with_mean(RV &out, float (&lev)[RV::kCount], float step, float mean)
{
#pragma unroll
    for (int i = 0; i < RV::kCount; i++) lev[i] = round_element<DT>(lev[i] * step) + mean;
    out.set(lev);
}

// ---- one rank -------------------------------------------------------------------------------------------

struct RoundtripBucket {
    const void *src;
    void *out;
    uint32_t *stats;
    int32_t *counts;
    int64_t n;
    uint64_t step;
    int vec; // src and out 16-byte aligned
};

struct WidthRule {
    float u;
    const double *u_dev; // when set: u is *u_dev
    int thr[2];          // with u a number: the patterns of width 4 and 8 found on the host, else -1
};

// A launch carries arguments for one bucket, kFewBuckets or kMaxBuckets: 296, 952 or 2,152 bytes.  A call on one bucket, us, in a stream,
// with room for one, two, 8, 32: 4,096 elements 7.3, 7.5, 7.8, 7.9; 10^6 elements 7.4, 8.2, 8.4, 8.5.  Steady steps of lists gain less
// than 0.3 by less room, but beyond a kilobyte the host takes longer for the first step of a new object on new tensors: nine buckets of 10^6
// elements, by room, 9: 101, 12: 100, 13 (1,012 bytes): 100, 14 (1,072): 153, 16: 145, 24: 143, 32: 144; twelve 104, and 149 with 32.
constexpr int kFewBuckets = 12;

template <int MOST> struct RoundtripArgs {
    uint32_t first_tile[MOST]; // ascending
    RoundtripBucket bucket[MOST];
    int buckets;
    WidthRule rule;
    WorldDiv wd;
    uint64_t seed;
    const uint64_t *step_dev; // null, or added to every bucket's step
    uint64_t step_more;       // (with step_dev) and this, which tally_kernel leaves in *step_dev
    WidthSet widths;
};

__device__ __forceinline__ int class_of_norm(uint32_t pattern, float u, const int (&thr)[2])
{
    if (thr[0] >= 0 && __builtin_amdgcn_ballot_w64(pattern > (uint32_t)kMaxPattern) == 0)
        return (int)pattern >= thr[1] ? 0 : ((int)pattern >= thr[0] ? 1 : 2);
    return width_class_of_norm(pattern, u);
}

// the last entry of an ascending list that is <= x, by halving (scalar: as a sum of comparisons over the whole list it
// becomes sixty vector instructions)
__device__ __forceinline__ int last_at_most(const uint32_t *list, int count, uint32_t x)
{
    int lo = 0, hi = count - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (list[mid] <= x)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// The one-rank pass is bound by the vector ALU (470 instructions a tile, 504 before) with memory right behind it: a step of nine 25 MB
// buckets 41 us at 5.2 TB/s.  So a tile's elements become numbers once, for the sums and for the quantiser, a row's results come from its
// first lane without the LDS, and a whole tile leaves as the one run it is.  Whole calls, us: 1 x 30,761,978 in MEE 34.0 -> 32.1, 1 x
// 1,761,978 8.2 -> 8.0; with the tally below, 11 buckets of 12.2 M in MEE 134 -> 128, nine of 3 M 31.2 -> 28.6.
// lane 0 of the lane's row of sixteen
__device__ __forceinline__ uint32_t of_row(uint32_t x) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x150, 0xf, 0xf, true); } // row_newbcast:0

template <int DT, bool MEE, int MOST> __global__ __launch_bounds__(64) void roundtrip_kernel(RoundtripArgs<MOST> a)
{
    constexpr int kSlots = Raw16<DT>::kSlots, kStage = 64 * kSlots * 16;
    __shared__ __attribute__((aligned(16))) uint8_t lds[kFloatTileBytes > kStage ? kFloatTileBytes : kStage];
    __shared__ float levels[MEE ? kLevelCount : 1];
    const int lane = threadIdx.x, row = lane >> 4, j = lane & 15;

    // (ahead of the elements' loads, behind which they would be loads of the lanes and wait for those)
    uint64_t step = a.step_dev ? *a.step_dev + a.step_more : 0;
    const float u = a.rule.u_dev ? (float)*a.rule.u_dev : a.rule.u;
    const int at = MOST == 1 ? 0 : last_at_most(a.first_tile, a.buckets, blockIdx.x);
    const RoundtripBucket &b = a.bucket[at];
    const int64_t n = b.n, nsc = (n + 255) >> 8;
    const int64_t sc0 = (int64_t)(blockIdx.x - a.first_tile[at]) * kRowsPerWave;
    if (sc0 >= nsc) return;
    const bool ragged = (sc0 + kRowsPerWave) * 256 > n; // (and fewer than four superchunks, at times)
    const int rows_here = ragged ? (int)min((int64_t)kRowsPerWave, nsc - sc0) : kRowsPerWave;
    const bool active = row < rows_here;
    const int64_t sc = sc0 + (ragged ? min(row, rows_here - 1) : row);
    const int64_t e0 = sc * 256 + j * 16;

    Raw16<DT> v;
    v.zero();
    if (!ragged) {
        v.load(b.src, e0, b.vec != 0);
    } else if (active) {
        load_chunk_guarded<DT>(v, b.src, e0, n);
    }
    if (MEE) levels_to_lds(levels, lane);
    // the rounding stream's arithmetic while the elements are on their way
    Raw16<DQ_PHILOX> r;
    r.generate(RandKey{a.seed, b.step + step}, sc * 16 + j);
    r.pin();

    float t[16];
#pragma unroll
    for (int i = 0; i < 16; i++) t[i] = v.get(i);
    if (!a.wd.pow2) {
        a.wd.divide(t);
    } else if (a.wd.inv != 1.0f) {
#pragma unroll
        for (int i = 0; i < 16; i++) t[i] *= a.wd.inv;
    }
    float sum, sq;
    float_tile_sums(t, reinterpret_cast<float *>(lds), lane, sum, sq);
    const float mean = __uint_as_float(of_row(__float_as_uint(superchunk_mean(sum, sc * 256, n, ragged))));
    const uint32_t norm = of_row(f32_to_bf16_bits(sq));
    const uint32_t mean_bits = f32_to_bf16_bits(mean);
    if (active && j == 0) b.stats[sc] = mean_bits | (norm << 16);
    if (sc0 == 0 && lane < 4) b.counts[lane] = 0; // (tally_kernel adds to them)

    const WidthRegs<MEE> w = width_regs<MEE>(a.widths, class_of_norm(norm, u, a.rule.thr), levels);
    // (v / world - mean: center_loaded forms the same number, in one rounding or two)
#pragma unroll
    for (int i = 0; i < 16; i++) t[i] -= mean;
    finish_centered<DT>(t, e0, n, ragged);
    float lev[16];
    const float scale = quantize_chunk<MEE>(t, r, w, lev);
    decode_with_mean<DT>(v, lev, scale, bf16_bits_to_f32(mean_bits));
    wave_lds_sync(); // the statistics' tile has been read
    stage_tile<DT>(v, reinterpret_cast<uint4 *>(lds), lane);
    if (!ragged && b.vec != 0) {
        // the tile is one run
        const uint4 *stage = reinterpret_cast<const uint4 *>(lds);
        uint4 *to = reinterpret_cast<uint4 *>(static_cast<char *>(b.out) + sc0 * (kStage / kRowsPerWave)) + lane;
#pragma unroll
        for (int k = 0; k < kSlots; k++) stream_store(to + 64 * k, stage[swz(64 * k + lane)]);
    } else {
        store_tile<DT>(b.out, v, reinterpret_cast<const uint4 *>(lds), sc, rows_here, n, b.vec != 0, lane);
    }
}

struct TallyBucket {
    const uint16_t *stats;
    int32_t *counts;
    int64_t nsc;
};

template <int MOST> struct TallyArgs {
    uint32_t first_block[MOST];
    TallyBucket bucket[MOST];
    WidthRule rule;
    uint32_t *hist;
    uint64_t *step_dev;
    uint64_t step_more;
};

// A workgroup takes kTallyBatch superchunks of one bucket.  A wave's norms are alike and meet in a few counters of the LDS, so the
// counting is better spread over more workgroups: 209,716 norms with 8192 each 7.9 us, 4096 6.6, 2048 and 1024 6.4.  What is
// left is a chain of latencies; clearing 64 KB of counters, going over them afterwards and searching the two thresholds for two
// norms per thread were the longest links (6.0 us; 4.6 with the counters in range alone and the rule applied to each norm), then a search
// for the bucket by halving, a load per step, and a barrier of the widths' own.
// (Clearing each norm's own counter and leaving it to whoever found it at 0 spares a barrier, but scatters the atomics on memory:
// 4.8 us here, and 42.9 instead of 12.1 for batches of 8192 of 3,000,000 norms.)
constexpr int kTallyThreads = 1024, kTallyBatch = 2048;

// The norm patterns of a tally's batch, counted in LDS (16-bit counters, two per word) and added to the histogram in memory: begin
// (two barriers), add, a barrier of the caller's, flush.  Thread t holds the patterns k * kTallyThreads + t, of which those
// below `have` count.  Only the counters between the batch's least and greatest pattern are cleared and gone over, where zeros
// (of which a bucket may hold many) and NaN are counted apart.
template <int PER> struct PatternBatch {
    uint32_t low, high; // words of counters in use
    uint32_t zeros_nans; // of wave lane & 15

    // mine: what else the waves have to tell one another (n4 | n8 << 16); returned for wave lane & 15
    __device__ __forceinline__ uint32_t begin(const uint32_t (&pattern)[PER], int have, uint32_t mine, uint32_t *local, uint4 *wave_seen)
    {
        const int t = threadIdx.x, lane = t & 63;
        uint32_t top = 0, under = 0; // the greatest bin, the complement of the least
        uint32_t zeros = 0, nans = 0;
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const uint32_t bin = (uint32_t)bin_of(pattern[k]);
            const bool in = k * kTallyThreads + t < have, zero = bin == 0u, nan = bin == (uint32_t)kNanBin;
            top = max(top, in && !nan ? bin : 0u);
            under = max(under, in && !zero && !nan ? ~bin : 0u);
            zeros += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(in && zero));
            nans += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(in && nan));
        }
        top = wave_max_upward(top);
        under = wave_max_upward(under);
        if (lane == 63) wave_seen[t >> 6] = make_uint4(top, under, zeros | (nans << 16), mine);
        __syncthreads();
        static_assert(kTallyThreads / 64 == 16, "a row of 16 lanes holds a value of every wave");
        const uint4 seen = wave_seen[lane & 15];
        high = (uint32_t)__builtin_amdgcn_readlane((int)wave_max_upward(seen.x), 63) >> 1;
        low = ~(uint32_t)__builtin_amdgcn_readlane((int)wave_max_upward(seen.y), 63) >> 1; // (no bin at all: beyond every word)
        zeros_nans = seen.z;
        for (uint32_t w = low + t; w <= high; w += kTallyThreads) local[w] = 0u;
        __syncthreads();
        return seen.w;
    }

    __device__ __forceinline__ void add(const uint32_t (&pattern)[PER], int have, uint32_t *local) const
    {
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int bin = bin_of(pattern[k]);
            if (k * kTallyThreads + (int)threadIdx.x < have && bin != 0 && bin != kNanBin) atomicAdd(&local[bin >> 1], 1u << (16 * (bin & 1)));
        }
    }

    __device__ __forceinline__ void flush(uint32_t *__restrict__ hist, const uint32_t *local) const
    {
        // (a word per thread: the counters in use lie side by side)
        for (uint32_t w = low + threadIdx.x; w <= high; w += kTallyThreads) {
            const uint32_t pair = local[w];
            if (pair & 0xffffu) atomicAdd(&hist[2 * w], pair & 0xffffu);
            if (pair >> 16) atomicAdd(&hist[2 * w + 1], pair >> 16);
        }
        if (threadIdx.x < 16) { // an entry of wave_seen each
            if (zeros_nans & 0xffffu) atomicAdd(&hist[0], zeros_nans & 0xffffu);
            if (zeros_nans >> 16) atomicAdd(&hist[kNanBin], zeros_nans >> 16);
        }
    }
};

template <bool HIST, int MOST> __global__ __launch_bounds__(kTallyThreads) void tally_kernel(TallyArgs<MOST> a)
{
    __shared__ uint32_t local[HIST ? kHistWords : 1];
    __shared__ uint4 wave_seen[kTallyThreads / 64];
    const int lane = threadIdx.x & 63;
    TallyBucket b;
    uint32_t first = 0;
    if constexpr (MOST == 1) {
        b = a.bucket[0];
    } else {
        // A lane per bucket, and the right lane's: one load's time.  (Behind the last bucket first_block is greater than any block.)
        static_assert(MOST <= 64, "a bucket per lane");
        const int k = min(lane, MOST - 1);
        const uint32_t starts = a.first_block[k];
        const TallyBucket mine = a.bucket[k];
        const int at = __popcll(__builtin_amdgcn_ballot_w64(lane < MOST && starts <= blockIdx.x)) - 1;
        const auto of = [at](uint64_t x) {
            const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, at), hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), at);
            return (uint64_t)lo | ((uint64_t)hi << 32);
        };
        // (addresses of memory, which the compiler knows of an argument but not of a lane's register)
        b.stats = (const uint16_t *)(const __attribute__((address_space(1))) uint16_t *)of(reinterpret_cast<uint64_t>(mine.stats));
        b.counts = (int32_t *)(__attribute__((address_space(1))) int32_t *)of(reinterpret_cast<uint64_t>(mine.counts));
        b.nsc = (int64_t)of((uint64_t)mine.nsc);
        first = (uint32_t)__builtin_amdgcn_readlane((int)starts, at);
    }
    const int64_t begin = (int64_t)(blockIdx.x - first) * kTallyBatch;
    constexpr int kPer = kTallyBatch / kTallyThreads;
    // (the last norm's address beyond the end: behind a comparison each, the loads would wait for one another)
    const int have = (int)min((int64_t)kTallyBatch, b.nsc - begin);
    const uint16_t *mine = b.stats + 2 * begin + 1;
    uint32_t norm[kPer];
#pragma unroll
    for (int k = 0; k < kPer; k++) norm[k] = mine[2 * min(k * kTallyThreads + (int)threadIdx.x, have - 1)];
    const float u = a.rule.u_dev ? (float)*a.rule.u_dev : a.rule.u;
    uint32_t counts = 0; // of the wave: n4 | n8 << 16
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const bool in = k * kTallyThreads + (int)threadIdx.x < have;
        const int c = a.rule.thr[0] >= 0 ? class_of_norm(norm[k], u, a.rule.thr) : width_class_of_norm(norm[k], u);
        counts += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(in && c == 1)) + ((uint32_t)__popcll(__builtin_amdgcn_ballot_w64(in && c == 0)) << 16);
    }
    static_assert(kTallyBatch <= 0xffff, "two counts in a word");
    PatternBatch<kPer> batch;
    if (HIST) {
        counts = batch.begin(norm, have, counts, local, wave_seen);
    } else {
        if (lane == 0) wave_seen[threadIdx.x >> 6].w = counts;
        __syncthreads();
        counts = wave_seen[lane & 15].w;
    }
    if (HIST) {
        batch.add(norm, have, local);
        __syncthreads();
        batch.flush(a.hist, local);
    }
    if (threadIdx.x >= kTallyThreads - 64) { // (the wave with the least to flush)
        // sums over the row of sixteen lanes, a wave's each, in the last of them
        counts += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)counts, 0x111, 0xf, 0xf, true); // row_shr:1, 2, 4, 8
        counts += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)counts, 0x112, 0xf, 0xf, true);
        counts += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)counts, 0x114, 0xf, 0xf, true);
        counts += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)counts, 0x118, 0xf, 0xf, true);
        if (lane == 15) {
            const int c8 = (int)(counts >> 16), c4 = (int)(counts & 0xffffu), c2 = have - c8 - c4;
            if (c8) atomicAdd(&b.counts[0], c8);
            if (c4) atomicAdd(&b.counts[1], c4);
            if (c2) atomicAdd(&b.counts[2], c2);
            if (blockIdx.x == 0 && a.step_dev && a.step_more) *a.step_dev += a.step_more;
        }
    }
}

// ---- W ranks --------------------------------------------------------------------------------------------

struct RankPointers {
    const void *src[kMaxRanks];
};

struct TileWidths {
    uint32_t *words; // null, or one per four superchunks: how many the rule gives 8 bits, and 4 bits in the upper half
    WidthRule rule;
};

constexpr int kStatsWaves = 8; // ranks in flight per workgroup of ranks_stats_kernel
// A workgroup takes GROUPS tiles of four superchunks, a wave of it those of one rank (of every kStatsWaves-th one in a larger
// world): means and norms per rank, and the statistics all-reduce as the reference's chain of bf16 additions in rank order.
// Bound by how much is on the way: a wave that adds up what it has just waited for, and then waits at the barrier for the
// other ranks, asks for nothing meanwhile.  So it has the next tile of its rank on the way while it adds up the current one,
// and meets the others once in GROUPS tiles.  The tiles come as whole lines (a tile goes through LDS anyway).  NT: loads that
// leave the caches to others.
struct StatsArgs {
    RankPointers ranks;
    int world, vec;
    int64_t n;
    uint32_t *total;
    float *mean;
    WorldDiv wd;
    TileWidths widths;
};

template <int DT, int GROUPS, bool NT, bool WORDS> __global__ __launch_bounds__(64 * kStatsWaves, 8) void ranks_stats_kernel(StatsArgs a)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t tiles[];
    const RankPointers &ranks = a.ranks;
    const TileWidths &widths = a.widths;
    const WorldDiv &wd = a.wd;
    uint32_t *__restrict__ total = a.total;
    float *__restrict__ mean_out = a.mean;
    const int world = a.world, vec = a.vec;
    const int64_t n = a.n;
    // asked for ahead of the loads of a single tile; behind the last of several, whose 64 registers have no room for it
    float u = 0.0f;
    if (WORDS && GROUPS == 1) u = widths.rule.u_dev ? (float)*widths.rule.u_dev : widths.rule.u;
    constexpr int kRows = GROUPS * kRowsPerWave;
    __shared__ uint32_t pairs[kMaxRanks][kRows];
    typedef StatsTile<DT> ST;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    constexpr int kSlots = Raw16<DT>::kSlots, kRowBytes = 256 * ST::ESZ;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = min(world, kStatsWaves);
    const int row = lane >> 4, j = lane & 15;
    const int64_t nsc = (n + 255) >> 8;
    const int64_t sc0 = (int64_t)blockIdx.x * kRows;
    const int rows_here = (int)min((int64_t)kRows, nsc - sc0);
    uint8_t *lds = tiles + wave * ST::BYTES;
    if (vec != 0 && (sc0 + kRows) * 256 <= n) {
        for (int rank = wave; rank < world; rank += waves) {
            const u32x4 *from = reinterpret_cast<const u32x4 *>(static_cast<const uint8_t *>(ranks.src[rank]) + sc0 * kRowBytes) + lane;
            u32x4 q[2][kSlots];
#pragma unroll
            for (int k = 0; k < kSlots; k++) q[0][k] = NT ? __builtin_nontemporal_load(from + k * 64) : from[k * 64];
#pragma unroll
            for (int g = 0; g < GROUPS; g++) {
                if (g + 1 < GROUPS) {
#pragma unroll
                    for (int k = 0; k < kSlots; k++) {
                        const u32x4 *next = from + ((g + 1) * kSlots + k) * 64;
                        q[(g + 1) & 1][k] = NT ? __builtin_nontemporal_load(next) : *next;
                    }
                }
                const int r = g * kRowsPerWave + row;
#pragma unroll
                for (int k = 0; k < kSlots; k++) {
                    const int at = k * 1024 + lane * 16;
                    *reinterpret_cast<u32x4 *>(lds + (at / kRowBytes) * ST::RS + at % kRowBytes) = q[g & 1][k];
                }
                wave_lds_sync();
                float sum, sq;
                staged_tile_sums<DT>(wd, lds, lane, sum, sq);
                wave_lds_sync();
                if (j == 0) {
                    const float mean = sum * 0.00390625f;
                    pairs[rank][r] = f32_to_bf16_bits(mean) | (f32_to_bf16_bits(sq) << 16);
                    mean_out[rank * nsc + sc0 + r] = mean;
                }
            }
        }
    } else {
        for (int rank = wave; rank < world; rank += waves) {
            for (int g = 0; g * kRowsPerWave < rows_here; g++) {
                const int r = g * kRowsPerWave + row;
                const int64_t first = (sc0 + r) * 256;
                const bool ragged = (sc0 + (g + 1) * kRowsPerWave) * 256 > n;
                Raw16<DT> v;
                v.zero();
                if (r < rows_here) load_chunk<DT>(v, ranks.src[rank], first + j * 16, n, vec != 0, ragged);
                float sum, sq;
                tile_sums<DT>(v, wd, lds, lane, sum, sq);
                wave_lds_sync();
                if (j == 0 && r < rows_here) {
                    const float mean = superchunk_mean(sum, first, n, ragged);
                    pairs[rank][r] = f32_to_bf16_bits(mean) | (f32_to_bf16_bits(sq) << 16);
                    mean_out[rank * nsc + sc0 + r] = mean;
                }
            }
        }
    }
    if (WORDS && GROUPS > 1) u = widths.rule.u_dev ? (float)*widths.rule.u_dev : widths.rule.u;
    __syncthreads();
    if (threadIdx.x < rows_here) {
        uint32_t acc = pairs[0][threadIdx.x];
        for (int rank = 1; rank < world; rank++) {
            const uint32_t p = pairs[rank][threadIdx.x];
            const float lo = bf16_bits_to_f32(acc & 0xffffu) + bf16_bits_to_f32(p & 0xffffu);
            const float hi = bf16_bits_to_f32(acc >> 16) + bf16_bits_to_f32(p >> 16);
            acc = f32_to_bf16_bits(lo) | (f32_to_bf16_bits(hi) << 16);
        }
        total[sc0 + threadIdx.x] = acc;
        if (WORDS) {
            const int cls = class_of_norm(acc >> 16, u, widths.rule.thr);
            const uint64_t eights = __builtin_amdgcn_ballot_w64(cls == 0), fours = __builtin_amdgcn_ballot_w64(cls == 1);
            if ((threadIdx.x & 3) == 0)
                widths.words[(sc0 + threadIdx.x) >> 2] = (uint32_t)__popcll((eights >> threadIdx.x) & 15u) |
                                                         ((uint32_t)__popcll((fours >> threadIdx.x) & 15u) << 16);
        }
    }
}

// rounding randomness out of the compressors' pools: which rank uses which rows of which pool in which step
struct FromTileWidths {
    const uint32_t *words; // of ranks_stats_kernel
    int32_t *counts;       // written: group sizes
    WidthRule rule;
};
struct Pools {
    const void *pool[3][kMaxPoolRanks];                          // one per width (8, 4, 2 bits) and rank
    int32_t first[3][kMaxPoolRanks][kMaxPoolRanks];              // first row of 16 values: [width][rank][step]
};

template <bool POOL> struct RingArgs {
    const void *src[kMaxRanks];
    void *out[kMaxRanks];
    const float *mean;      // [world][nsc]
    const uint16_t *total;  // reduced statistics
    const int32_t *order;   // the plan: row lists and group sizes
    const int32_t *counts;
    int64_t n;
    int nsc, world, vec;
    RandKey key;
    WorldDiv wd;
    WidthSet widths;
    typename std::conditional<POOL, Pools, FromTileWidths>::type more;
};

// Workgroup (x, y): tile x of ring chunk y -- rank y compresses it first, rank y + 1 decodes, adds and recompresses, and
// so on around the ring; the last one's records are what every rank decodes.  The runs of the chunk follow one another as in
// dq_scaling_mixed.hip (8-bit, 4-bit, 2-bit), so a wave has one width and one first rank.
// (Held to five waves per SIMD, 96 registers, where the compiler takes 97 by itself: the longest vectors wait for memory.)
template <int DT, int RDT, bool MEE>
__global__ __launch_bounds__(64, DT == DQ_BF16 && RDT == DQ_PHILOX && !MEE ? 5 : 1) void ring_kernel(RingArgs<RDT != DQ_PHILOX> a)
{
    __shared__ __attribute__((aligned(16))) uint4 stage[64 * Raw16<DT>::kSlots];
    __shared__ float levels[MEE ? kLevelCount : 1];
    const int lane = threadIdx.x, row = lane >> 4, j = lane & 15;
    const int chunk = blockIdx.y, world = a.world;
    // the run this tile lies in: group sizes clamped so that a corrupt count cannot lead outside the lists
    int cls = 3, tile = blockIdx.x, cnt = 0;
    int64_t row0 = 0;
    {
        int used = 0;
        const int counts[3] = {a.counts[0], a.counts[1], a.counts[2]};
#pragma unroll
        for (int g = 0; g < 3; g++) {
            const int m = min(max(counts[g], 0), a.nsc - used);
            const int per = (m + world - 1) / world;
            const int begin = (int)min((int64_t)per * chunk, (int64_t)m);
            const int here = min(per, m - begin);
            const int tiles = (here + kRowsPerWave - 1) / kRowsPerWave;
            if (cls == 3) {
                if (tile < tiles) {
                    cls = g; cnt = here; row0 = (int64_t)g * a.nsc + begin;
                } else {
                    tile -= tiles;
                }
            }
            used += m;
        }
    }
    if (cls == 3) return;
    const int k0 = tile * kRowsPerWave;
    const int rows_here = min(kRowsPerWave, cnt - k0);
    const bool active = row < rows_here;
    const int64_t sc = a.order[row0 + k0 + min(row, rows_here - 1)];
    const int64_t e0 = sc * 256 + j * 16;
    const bool ragged = __builtin_amdgcn_ballot_w64(e0 + 16 > a.n) != 0;
    if (MEE) levels_to_lds(levels, lane);
    const WidthRegs<MEE> w = width_regs<MEE>(a.widths, cls, levels);
    const uint32_t total_mean = a.total[2 * sc];

    // the next rank's elements (and random values) are on their way while this rank's are quantised
    Raw16<DT> next;
    Raw16<RDT> next_r;
    float next_mean = 0.0f;
    next.zero();
    next_r.zero();
    const auto fetch = [&](int step) {
        int rank = chunk + step;
        if (rank >= world) rank -= world;
        if (active) {
            load_chunk<DT>(next, a.src[rank], e0, a.n, a.vec & 1, ragged);
            next_mean = a.mean[(int64_t)rank * a.nsc + sc];
            if constexpr (RDT != DQ_PHILOX)
                next_r.load(a.more.pool[cls][rank], ((int64_t)a.more.first[cls][rank][step] + k0 * 16 + lane) * 16, (a.vec & 4) != 0);
        }
    };
    fetch(0);
    float lev[16], scale = 0.0f;
#pragma unroll 1
    for (int step = 0; step < world; step++) {
        const Raw16<DT> v = next;
        Raw16<RDT> r = next_r;
        const float mean = next_mean;
        if (step + 1 < world) fetch(step + 1);
        if constexpr (RDT == DQ_PHILOX) {
            int rank = chunk + step;
            if (rank >= world) rank -= world;
            r.generate(RandKey{a.key.seed + (uint64_t)rank, (uint64_t)step}, sc * 16 + j);
        }
        float x[16];
        center_loaded<DT>(x, v, a.wd, mean, e0, a.n, ragged);
        if (step > 0) { // the sum, in the element type
#pragma unroll
            for (int i = 0; i < 16; i++) x[i] = round_element<DT>(__builtin_fmaf(lev[i], scale, x[i]));
        }
        scale = quantize_chunk<MEE>(x, r, w, lev);
    }
    Raw16<DT> out;
    decode_with_mean<DT>(out, lev, scale, bf16_bits_to_f32(total_mean));
    stage_tile<DT>(out, stage, lane);
    for (int rank = 0; rank < world; rank++) store_tile<DT>(a.out[rank], out, stage, sc, rows_here, a.n, (a.vec & 2) != 0, lane);
}

// a lane's part of a chunk, side by side with those of its neighbours
template <int DT, int N> __device__ __forceinline__ void store_part(void *dst, const RawPart<DT, N> &out, int64_t e, int64_t n, bool vec, bool ragged)
{
    constexpr int W = RawPart<DT, N>::kWords;
    if (vec && !ragged) {
        uint32_t *p = static_cast<uint32_t *>(dst) + e * W / N;
        if constexpr (W == 2) {
            typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
            const u32x2 t = {out.w[0], out.w[1]};
            __builtin_nontemporal_store(t, reinterpret_cast<u32x2 *>(p));
        } else {
#pragma unroll
            for (int k = 0; k < W; k += 4) stream_store(reinterpret_cast<uint4 *>(p + k), make_uint4(out.w[k], out.w[k + 1], out.w[k + 2], out.w[k + 3]));
        }
        return;
    }
    const int left = left_here(n, e, N);
#pragma unroll
    for (int i = 0; i < N; i++) {
        if (i < left) {
            if constexpr (DT == DQ_F32)
                static_cast<uint32_t *>(dst)[e + i] = out.w[i];
            else
                static_cast<uint16_t *>(dst)[e + i] = (uint16_t)(out.w[i >> 1] >> (16 * (i & 1)));
        }
    }
}

// x / y for 0 <= x < 2^23, 0 < y, inv = 1 / y to within an ulp or two
__device__ __forceinline__ int small_quotient(int x, int y, float inv)
{
    int q = (int)((float)x * inv);
    const int r = x - q * y;
    return q + (r >= y ? 1 : 0) - (r < 0 ? 1 : 0);
}

constexpr int kPartWaves = 4;

// ring_kernel with N = 4 or 8 elements per lane, a superchunk or two per wave: short vectors, where a wave's chain of `world` steps is all
// there is to wait for (2 us a step with one wave of ring_kernel per SIMD, 0.7 us with four elements).
//
// PLANS: without a plan launch in front.  A superchunk's way through the ring depends on the others only by where it starts: on its
// place among those of its width.  The statistics leave a word per four superchunks with their widths' counts; a workgroup takes
// neighbouring superchunks and adds up the words, all of them and those before its own, while the norms of its own are on their way.
//
// Fours with drawn values are held to 64 vector registers and stay within 80 scalar ones, or a SIMD has room for seven waves instead of eight,
// whatever the compiler counts: with 81, 96 and the trap handler's 16 are taken.  MEE from 7,169 superchunks on, all vectors an element off the
// 16 bytes, with 81 -> 79, us: 2 x 8,192 23.6 -> 22.5, 8 x 8,192 71.0 -> 65.2.
template <int DT, int RDT, bool MEE, int N, bool PLANS>
__global__ __launch_bounds__(64 * kPartWaves, N == 4 && RDT == DQ_PHILOX ? 8 : 1) void ring_parts_kernel(RingArgs<RDT != DQ_PHILOX> a)
{
    constexpr int P = N / 4, kLanes = 64 / P, kHere = P * kPartWaves; // superchunks of a wave, lanes of one, superchunks of the workgroup
    constexpr bool POOL = RDT != DQ_PHILOX;
    __shared__ float levels[MEE ? kLevelCount : 1];
    // What a step needs besides its elements, by rank and once more, so that the ranks from any on lie side by side: the address of the
    // vector and the mean.  (Loaded step by step through the scalar cache they are half of a step's time.)
    __shared__ uint4 of_rank[kPartWaves][P][2 * kMaxRanks];
    __shared__ uint64_t pool_of_step[POOL ? kPartWaves : 1][kMaxPoolRanks];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), world = a.world;
    const int half = lane / kLanes; // (0 where a wave has one superchunk)
    const int rank_here = lane & (2 * kMaxRanks - 1), my_rank = min(rank_here < world ? rank_here : rank_here - world, world - 1);
    const int which = P == 1 ? 0 : lane >> 5; // superchunk whose ranks the lane fetches
    const uint64_t my_src = reinterpret_cast<uint64_t>(a.src[my_rank]);
    if (MEE) {
        if (wave == 0) levels_to_lds(levels, lane);
        if (!PLANS) __syncthreads();
    }
    const int at0 = ((int)blockIdx.x * kPartWaves + wave) * P;
    int cls[P], chunk[P], in_run[P];
    int64_t sc[P];
    float my_mean = 0.0f;
    uint32_t total_mean = 0;
    int have = 0; // of the wave's superchunks; the others repeat the first
    if constexpr (PLANS) {
        static_assert(kHere % kRowsPerWave == 0, "a workgroup's superchunks are those of whole words");
        __shared__ uint2 part[kPartWaves];
        const FromTileWidths &f = a.more;
        const int first_word = (int)blockIdx.x * P, words = (a.nsc + 3) >> 2;
        const uint32_t norm = a.total[2 * min(kHere * (int)blockIdx.x + (lane & (kHere - 1)), a.nsc - 1) + 1];
        // (neither waits for the place in the list)
        my_mean = a.mean[(int64_t)my_rank * a.nsc + min(at0 + which, a.nsc - 1)];
        total_mean = a.total[2 * min(at0 + half, a.nsc - 1)];
        const double u_dev = *(f.rule.u_dev ? f.rule.u_dev : &kNoOffset);
        uint32_t all = 0, before = 0;
        constexpr int kTogether = 4, kThreads = 64 * kPartWaves;
        for (int first = 0; first < words; first += kTogether * kThreads) {
            uint32_t got[kTogether];
#pragma unroll
            for (int i = 0; i < kTogether; i++) got[i] = f.words[min(first + i * kThreads + (int)threadIdx.x, words - 1)];
#pragma unroll
            for (int i = 0; i < kTogether; i++) {
                const int word = first + i * kThreads + (int)threadIdx.x;
                all += word < words ? got[i] : 0u;
                before += word < first_word ? got[i] : 0u;
            }
        }
        all = wave_sum_upward(all);
        before = wave_sum_upward(before);
        if (lane == 63) part[wave] = make_uint2(all, before);
        const float u = f.rule.u_dev ? (float)u_dev : f.rule.u;
        const int mine = class_of_norm(norm, u, f.rule.thr); // (of lane & (kHere - 1))
        __syncthreads();
        const uint2 p0 = part[0], p1 = part[1], p2 = part[2], p3 = part[3];
        all = (uint32_t)__builtin_amdgcn_readfirstlane((int)(p0.x + p1.x + p2.x + p3.x));
        before = (uint32_t)__builtin_amdgcn_readfirstlane((int)(p0.y + p1.y + p2.y + p3.y));
        const int m8 = (int)(all & 0xffffu), m4 = (int)(all >> 16), m2 = a.nsc - m8 - m4;
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            f.counts[0] = m8;
            f.counts[1] = m4;
            f.counts[2] = m2;
            f.counts[3] = 0;
        }
        have = min(a.nsc - at0, P);
        if (have <= 0) return;
        const int b8 = (int)(before & 0xffffu), b4 = (int)(before >> 16);
#pragma unroll
        for (int h = 0; h < P; h++) {
            const int of = h < have ? h : 0, bit = wave * P + of;
            sc[h] = at0 + of;
            cls[h] = __builtin_amdgcn_readlane(mine, bit);
            const int m = cls[h] == 0 ? m8 : (cls[h] == 1 ? m4 : m2);
            const int k = (cls[h] == 0 ? b8 : (cls[h] == 1 ? b4 : kRowsPerWave * first_word - b8 - b4)) +
                          __popcll(__builtin_amdgcn_ballot_w64(mine == cls[h]) & ((1u << bit) - 1u));
            // (within the ranks also with words that are not these norms')
            const int per = max(small_quotient(max(m + world - 1, 0), world, a.wd.inv), 1);
            chunk[h] = max(min(small_quotient(max(k, 0), per, __builtin_amdgcn_rcpf((float)per)), world - 1), 0);
            in_run[h] = 0;
        }
    } else {
        // entry at0 + h of the three lists end to end; sizes clamped as in ring_kernel
        const int counts[3] = {a.counts[0], a.counts[1], a.counts[2]};
#pragma unroll
        for (int h = 0; h < P; h++) {
            int used = 0, k = 0;
            cls[h] = 3;
#pragma unroll
            for (int g = 0; g < 3; g++) {
                const int m = min(max(counts[g], 0), a.nsc - used);
                if (cls[h] == 3 && at0 + h - used < m) {
                    const int per = small_quotient(m + world - 1, world, a.wd.inv);
                    cls[h] = g;
                    k = at0 + h - used;
                    chunk[h] = small_quotient(k, per, __builtin_amdgcn_rcpf((float)per));
                    in_run[h] = k - chunk[h] * per;
                }
                used += m;
            }
            if (cls[h] == 3) {
                if (h == 0) return;
                cls[h] = cls[0]; chunk[h] = chunk[0]; in_run[h] = in_run[0]; sc[h] = sc[0];
            } else {
                sc[h] = a.order[(int64_t)cls[h] * a.nsc + k];
                have = h + 1;
            }
        }
        my_mean = a.mean[(int64_t)my_rank * a.nsc + sc[P - 1 < which ? P - 1 : which]];
        total_mean = a.total[2 * sc[half]];
    }
    const int64_t my_sc = P == 1 || half == 0 ? sc[0] : sc[P - 1];
    const int my_chunk = P == 1 || half == 0 ? chunk[0] : chunk[P - 1], my_cls = P == 1 || half == 0 ? cls[0] : cls[P - 1];
    const int64_t e0 = my_sc * 256 + (lane & (kLanes - 1)) * N;
    const bool ragged = max(sc[0], sc[P - 1]) * 256 + 256 > a.n;
    // The vector's end may lie inside a lane's elements: it loads the last N there are and drops those before its own when it comes to
    // them.  (Loaded one by one and put together on the spot, the one ragged wave of a launch waited for memory in every step and
    // outlasted all others: 15.8 us where they had ended at 11 to 13, 8 x 1,000,003 elements.)  Vectors off the 16 bytes are loaded in one piece
    // too: element by element, a lane waited for each.  Statistics and ring, all vectors an element off, us: 8 x 7,000 superchunks 57.7 -> 50.1,
    // 16 x 7,000 111 -> 96, 2 x 12,288 29.8 -> 27.8, fp32 8 x 3,907 52.0 -> 47.8.
    const bool whole_loads = a.n >= N;
    const int64_t from = min(e0, a.n - N);
    const WidthRegs<MEE> w = width_regs<MEE>(a.widths, my_cls, levels);
    uint64_t my_pool = 0; // of step `lane`
    if constexpr (POOL) {
        static_assert(P == 1, "pools are for a superchunk per wave");
        const int step = min(lane & (kMaxPoolRanks - 1), world - 1), rank = chunk[0] + step < world ? chunk[0] + step : chunk[0] + step - world;
        my_pool = reinterpret_cast<uint64_t>(a.more.pool[cls[0]][rank]) +
                  (int64_t)(a.more.first[cls[0]][rank][step] + in_run[0] * 16) * (16 * (RDT == DQ_F32 ? 4 : 2));
    }

    // (memory, and the compiler is told so: what it only knows as an address it loads through instructions that may also mean the LDS,
    // and every read of the LDS then waits for the elements of the step to come)
    typedef const __attribute__((address_space(1))) void *global;
    const auto pointer = [](uint64_t at) { return (const void *)(global)at; };
    RawPart<DT, N> next;
    RawPart<RDT, N> next_r;
    next_r.zero();
    float next_mean = 0.0f;
    const auto load = [&](uint64_t src, uint64_t pool) {
        if (whole_loads)
            next.load_anywhere(pointer(src), from);
        else
            load_chunk_guarded<DT>(next, pointer(src), e0, a.n);
        if constexpr (POOL) next_r.load(pointer(pool), lane * N, (a.vec & 4) != 0);
    };
    // With lists the means wait for an entry of the list, and the first step's elements not for them: its addresses come from the lanes
    // instead of the table (fixed proportions, 4 x 64 superchunks 13.9 -> 13.4 us, 2 x 256 in MEE 12.6 -> 12.4).
    if constexpr (!PLANS) {
        const auto of_lane = [](uint64_t x, int at) {
            return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, at) |
                   (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), at) << 32;
        };
        const uint64_t first = of_lane(my_src, chunk[0]), second = P == 1 ? first : of_lane(my_src, chunk[P - 1]);
        load(half == 0 ? first : second, POOL ? of_lane(my_pool, 0) : 0);
    }
    if (rank_here < 2 * world && (P > 1 || lane < 2 * kMaxRanks))
        of_rank[wave][which][rank_here] = make_uint4((uint32_t)my_src, (uint32_t)(my_src >> 32), __float_as_uint(my_mean), 0u);
    if constexpr (POOL) {
        if (lane < kMaxPoolRanks) pool_of_step[wave][lane] = my_pool;
    }
    wave_lds_sync();
    const uint4 *ranks = of_rank[wave][half] + my_chunk;
    const auto fetch = [&](int step) {
        const uint4 of = ranks[step];
        next_mean = __uint_as_float(of.z);
        load((uint64_t)of.x | ((uint64_t)of.y << 32), POOL ? pool_of_step[wave][step] : 0);
    };
    if (PLANS)
        fetch(0);
    else
        next_mean = __uint_as_float(ranks[0].z);
    uint32_t draws[4];
    float lev[N], scale = 0.0f;
#pragma unroll 1
    for (int step = 0; step < world; step++) {
        RawPart<DT, N> v = next;
        RawPart<RDT, N> r = next_r;
        const float mean = next_mean;
        if (step + 1 < world) fetch(step + 1);
        if (whole_loads && ragged) v.drop((int)min((int64_t)N, e0 - from));
        if constexpr (!POOL) {
            constexpr int kTogether = 16 / N; // lanes of a chunk
            if ((step & (kTogether - 1)) == 0) {
                const int mine = step + (lane & (kTogether - 1));
                int of = my_chunk + mine; // (draws of steps beyond the last go unused)
                if (of >= world) of -= world;
                part_words<N>(RandKey{a.key.seed + (uint64_t)of, (uint64_t)mine}, my_sc * 16 + ((lane & (kLanes - 1)) / kTogether), lane, draws);
            }
#pragma unroll
            for (int k = 0; k < N / 4; k++) r.w[k] = draws[k];
#pragma unroll
            for (int k = 0; k < 4 - N / 4; k++) draws[k] = draws[k + N / 4];
        }
        float x[N];
        center_loaded<DT>(x, v, a.wd, mean, e0, a.n, ragged);
        if (step > 0) { // the sum, in the element type
#pragma unroll
            for (int i = 0; i < N; i++) x[i] = round_element<DT>(__builtin_fmaf(lev[i], scale, x[i]));
        }
        scale = quantize_chunk<MEE>(x, r, w, lev);
    }
    RawPart<DT, N> out;
    decode_with_mean<DT>(out, lev, scale, bf16_bits_to_f32(total_mean));
    if (half >= have) return;
    for (int rank = 0; rank < world; rank++) store_part<DT, N>(a.out[rank], out, e0, a.n, (a.vec & 2) != 0, ragged);
}

// How many elements a lane of the ring takes, 16 being ring_kernel.  Fewer issue more per element (160 instructions per superchunk and step
// with four, 110 with eight, 95 with sixteen), and from five waves per SIMD on that is what counts.  Statistics and ring without a plan,
// bf16, us, before there were eights (and with four elements loaded as in ring_parts_kernel's comment) -> four -> eight elements:
//   2 ranks  x 4,000 superchunks 10.9 9.8 10.8 (AEE), 11.5 11.3 11.3 (MEE), x 5,300 12.5 12.1 11.8, 13.3 13.0 12.8, x 8,000 13.4 12.7 12.9,
//            14.3 14.9 13.8, x 12,000 17.1 16.9 14.9, 18.5 18.7 17.4
//   5 ranks  x 4,000 15.7 15.2 15.5, 16.7 16.5 16.6, x 5,000 18.1 17.4 18.2, 19.8 19.1 19.9, x 8,000 23.3 22.6 21.0, 25.5 25.3 23.1,
//            x 12,000 30.8 29.5 26.4, 33.6 32.9 30.4
//   8 ranks  x 2,000 (500,000 elements) 16.2 15.1 17.1, x 4,000 20.6 19.3 20.0, 22.3 21.0 21.7, x 5,000 24.0 22.6 24.0, 26.2 24.8 26.4,
//            x 8,000 31.8 29.3 28.6, 34.9 32.8 31.3, x 12,000 40.8 37.5 34.9, 44.7 42.6 40.9
// With fp32 elements eight are 32 bytes of a lane and its loads half lines: 5 ranks x 8,000 27.8 26.8 31.3, so fp32 stays with four; pools
// do as well (bf16, 4 x 4,600 18.0 -> 18.7, 8 x 5,200 27.2 -> 28.5, in MEE 19.3 -> 20.4, 29.0 -> 30.3).  Outputs off the 16 bytes are stored element by
// element, of which eight lie twice as far from the neighbour's, and fours stay at every length: 2 x 8,192 14.6 -> 15.6, 4 x 12,288 26.6 -> 32.0,
// 8 x 16,000 53.1 -> 70.4, in MEE 58.4 -> 74.3.  (Vectors off them alone are loaded in one piece: 2 x 8,192 19.4 -> 17.9, 4 x 12,288 42.7 -> 43.2, 8 x
// 16,000 94.8 -> 91.6.)
// From five ranks without a plan on, three with one, the steps are most of the time, and fours keep the lead up to seven waves per SIMD.  Of
// the time before there were eights, eight / four: 8 ranks x 5,200 0.994 / 0.932 (AEE), 1.000 / 0.936 (MEE), x
// 7,000 1.012 / 0.926, 1.044 / 0.951, x 7,300 0.943 / 0.933, 0.931 / 0.935; 5 x 7,000 0.992 / 0.964, 1.007 / 0.965; 4 x 7,000 0.958 / 0.959,
// 0.969 / 0.963; with lists 8 x 7,000 0.986 / 0.946, 0.994 / 0.947, 3 x 7,000 0.986 / 0.965, 1.001 / 0.982, 2 x 7,000 0.975 / 0.998, 0.976 / 0.986.
constexpr int kFoursTo = 5120, kFoursToMany = 7168;
constexpr int fours_to(int world, bool plans) { return world >= (plans ? 5 : 3) ? kFoursToMany : kFoursTo; }

// With lists from a plan, up to so many superchunks in parts.  bf16 with drawn values, plan and all, us, sixteen -> eight: 2 ranks x 10,240 19.1 ->
// 17.3 (AEE), 20.3 -> 18.4 (MEE), x 12,000 18.0 -> 17.9, 20.8 -> 20.2, x 16,000 19.5 -> 20.0; 5 x 16,000 35.9 -> 34.5, 40.2 -> 40.0, x 20,000 41.9 -> 40.0, 47.1 -> 45.6; 8 x 20,000
// 54.8 -> 52.7, 63.1 -> 60.1.  The others, kernel alone, sixteen -> four: 8 ranks x 256 superchunks 12.2 -> 7.8 (AEE), 15.9 -> 8.9 (MEE),
// 19.5 -> 8.3 (AEE from pools); x 8,192 from pools 26.2 -> 20.6, fp32 24.6 -> 23.2, 29.0 -> 23.9.  Two ranks in fp32 AEE with drawn values
// have their line at five waves per SIMD: x 4,900 6.8 -> 6.5, x 5,700 6.8 -> 7.2.
constexpr int kParts = 8192;
int parts_to(int world, bool bf16, bool mee, bool pooled)
{
    if (pooled) return kParts;
    if (bf16) return world >= 4 ? 20480 : 12288;
    return !mee && world < 3 ? kFoursTo : kParts;
}

// Up to so many superchunks a ring with drawn values finds its groups itself (ring_parts_kernel, PLANS) in the place of a plan launch of 4 to
// 6 us, which is also worth fewer elements per lane a little longer.  Statistics, (plan,) ring, us, with plan and ring_kernel -> without,
// bf16: 2 ranks x 16,000 19.6 -> 18.2 (AEE), 21.5 -> 20.4 (MEE), x 24,000 24.4 -> 24.4, 27.6 -> 28.5; 3 x 16,000 25.3 -> 23.7, 27.5 -> 26.7,
// x 24,000 31.5 -> 32.2, 35.5 -> 37.1; 8 x 16,000 48.6 -> 42.8, 53.9 -> 47.9, x 24,000 65.0 -> 61.8, 73.5 -> 70.0.  fp32, with four elements per
// lane: 2 x 12,000 20.3 -> 19.3, 22.0 -> 20.4, x 16,000 24.5 -> 24.1, 24.5 -> 25.7; 5 x 16,000 49.7 -> 46.9, 51.1 -> 48.4; 8 x 16,000 78.5 ->
// 74.9, 77.9 -> 75.8, x 20,000 96.9 -> 96.9, 98.9 -> 98.5.  Few ranks of bf16 near their line, with a plan -> without: 2 x 18,432 21.1 -> 19.8, 24.5 ->
// 22.8, x 19,000 21.4 -> 21.4, 24.6 -> 24.5, x 19,500 21.5 -> 21.3, 24.5 -> 24.9, x 20,480 21.6 -> 21.4, 26.0 -> 24.8; 3 x 18,432 27.9 -> 26.2, 31.7 ->
// 29.6, x 19,500 27.4 -> 28.1, 31.8 -> 32.1, x 20,000 28.1 -> 27.9, 31.7 -> 31.8, x 20,480 30.4 -> 27.9, 34.1 -> 31.9.
constexpr int kPlansItself = 20480, kPlansItself32 = 16384, kPlansItselfFew32 = 12288;
static_assert(kPlansItself <= 0xffff, "a width's count over all superchunks is half a word (ring_parts_kernel, PLANS)");

WidthRule make_rule(float u, const double *u_dev)
{
    WidthRule r{u, u_dev, {-1, -1}};
    if (!u_dev && u == u) {
        r.thr[0] = host_width_threshold(u, 4);
        r.thr[1] = host_width_threshold(u, 8);
    }
    return r;
}

} // namespace

template <int MOST>
static hipError_t run_roundtrip(const RoundtripDesc *desc, int count, int world, float u, const double *u_dev, uint64_t seed,
                            uint64_t *step_dev, uint64_t step_more, uint32_t *hist, int dtype, bool mee, const MeeParams *mp,
                            hipStream_t stream)
{
    RoundtripArgs<MOST> a;
    TallyArgs<MOST> t;
    static_assert(MOST > kFewBuckets || sizeof(a) <= 1024, "see RoundtripArgs");
    memset(&t, 0, sizeof(t));
    memset(t.first_block, 0xff, sizeof(t.first_block));
    memset(&a, 0, offsetof(RoundtripArgs<MOST>, rule));
    uint32_t tiles = 0, blocks = 0;
    for (int k = 0; k < MOST; k++) {
        if (k >= count) break;
        const RoundtripDesc &d = desc[k];
        const int64_t nsc = (d.n + 255) / 256;
        a.first_tile[k] = tiles;
        t.first_block[k] = blocks;
        a.bucket[k] = RoundtripBucket{d.src, d.out, static_cast<uint32_t *>(d.stats), d.counts, d.n, d.step,
                                      aligned16(d.src) && aligned16(d.out) ? 1 : 0};
        t.bucket[k] = TallyBucket{static_cast<const uint16_t *>(d.stats), d.counts, nsc};
        tiles += (uint32_t)((nsc + kRowsPerWave - 1) / kRowsPerWave);
        blocks += (uint32_t)((nsc + kTallyBatch - 1) / kTallyBatch);
    }
    a.buckets = count;
    a.rule = t.rule = make_rule(u, u_dev);
    a.wd = make_world_div(world, dtype == DQ_F32 ? 4 : 2);
    a.seed = seed;
    a.step_dev = step_dev;
    a.step_more = step_more;
    a.widths = make_width_set(mp, mee);
    t.hist = hist;
    t.step_dev = step_dev;
    t.step_more = step_more;
    hipError_t e;
    if (dtype == DQ_BF16)
        e = mee ? launch_with(roundtrip_kernel<DQ_BF16, true, MOST>, dim3(tiles), dim3(64), stream, a)
                : launch_with(roundtrip_kernel<DQ_BF16, false, MOST>, dim3(tiles), dim3(64), stream, a);
    else
        e = mee ? launch_with(roundtrip_kernel<DQ_F32, true, MOST>, dim3(tiles), dim3(64), stream, a)
                : launch_with(roundtrip_kernel<DQ_F32, false, MOST>, dim3(tiles), dim3(64), stream, a);
    if (e != hipSuccess) return e;
    return hist ? launch_with(tally_kernel<true, MOST>, dim3(blocks), dim3(kTallyThreads), stream, t)
                : launch_with(tally_kernel<false, MOST>, dim3(blocks), dim3(kTallyThreads), stream, t);
}

// count <= kMaxBuckets
hipError_t launch_roundtrip(const RoundtripDesc *desc, int count, int world, float u, const double *u_dev, uint64_t seed,
                            uint64_t *step_dev, uint64_t step_more, uint32_t *hist, int dtype, bool mee, const MeeParams *mp,
                            hipStream_t stream)
{
    const auto run = count == 1 ? run_roundtrip<1> : (count <= kFewBuckets ? run_roundtrip<kFewBuckets> : run_roundtrip<kMaxBuckets>);
    return run(desc, count, world, u, u_dev, seed, step_dev, step_more, hist, dtype, mee, mp, stream);
}

// ranks_stats_kernel, us, a tile per wave -> four -> eight (-> eight that pass the caches by): 2 ranks x 6,400 tiles 7.0 -> 6.8 -> 8.3
// (9.3), 8 x 1,954 7.8 -> 8.2 -> 8.6, 8 x 3,907 14.4 -> 12.9 -> 12.9 (12.8), 8 x 15,625 42.5 -> 39.4 -> 39.6 (39.4), 8 x 32,227 110 ->
// 102 -> 106 (82), 8 x 121,524 425 -> 375 (324).  The ring that follows reads the vectors again: out of the cache behind the L2
// (256 MB) if they are there, which loads that pass it by cost 10 us at 8 x 15,625 and nothing at 8 x 32,227.  Both launches,
// keeping -> passing by: 280 MB 147 -> 151, 320 MB 168 -> 170, 384 MB 215 -> 205.
// Vectors off the 16 bytes load element by element, each wave one tile and then the next with nothing on the way: a tile per wave
// whatever their length (in fours and eights -> one by one: bf16 8 x 2,051 tiles 42 -> 37.5, 8 x 15,626 283 -> 255, 8 x 121,524
// 1,895 -> 1,794; fp32 8 x 3,907 105 -> 73, 8 x 15,626 409 -> 298, 3 x 29,297 285 -> 220; bf16 8 x 3,907 goes the other way, 60 ->
// 64.5).
// Near the lines, a tile per wave -> four, statistics and ring together: bf16 8 x 2,075 28.8 -> 29.1, 8 x 2,500 30.0 -> 30.6, 8 x 2,550
// 34.5 -> 30.6, 8 x 2,750 34.6 -> 31.8, 2 x 10,000 27.4 -> 27.4; fp32 8 x 2,075 37.0 -> 37.5, 8 x 2,500 41.2 -> 41.3, 8 x 2,750 46.3 -> 44.4,
// 3 x 6,500 40.7 -> 41.2, 4 x 4,500 38.7 -> 38.9; in fp32, a tile per wave -> eight that pass the caches by: 2 x 37,500 (307 MB) 147 -> 146,
// 4 x 19,500 (319 MB) 156.5 -> 159.5, 8 x 10,000 (327 MB) 169 -> 166, 2 x 47,500 202 -> 193.
constexpr int64_t kStatsOneTile = 19 << 10, kStatsCache = (int64_t)300 << 20;

hipError_t launch_ranks_stats(const void *const *src, int world, int64_t n, void *total, float *mean, int dtype, uint32_t *tile_widths,
                              float u, const double *u_dev, hipStream_t stream)
{
    RankPointers p;
    int vec = 1;
    for (int r = 0; r < kMaxRanks; r++) {
        p.src[r] = r < world ? src[r] : nullptr;
        if (r < world && !aligned16(src[r])) vec = 0;
    }
    const int64_t nsc = (n + 255) / 256;
    const int64_t tiles = (nsc + kRowsPerWave - 1) / kRowsPerWave;
    const int waves = world < kStatsWaves ? world : kStatsWaves;
    const StatsArgs args{p, world, vec, n, static_cast<uint32_t *>(total), mean, make_world_div(world, dtype == DQ_F32 ? 4 : 2),
                         TileWidths{tile_widths, tile_widths ? make_rule(u, u_dev) : WidthRule{0.0f, nullptr, {-1, -1}}}};
    const auto run = [&](auto kernel, int groups, int tile_bytes) {
        return launch_with(kernel, dim3((unsigned)((tiles + groups - 1) / groups)), dim3(64 * waves), stream, args, waves * tile_bytes);
    };
    const auto launch = [&](auto type) {
        constexpr int DT = decltype(type)::value, kTile = StatsTile<DT>::BYTES;
        if (vec && tiles * world * StatsTile<DT>::ESZ * 1024 > kStatsCache && !tile_widths) return run(ranks_stats_kernel<DT, 8, true, false>, 8, kTile);
        if (vec && tiles * world > kStatsOneTile)
            return tile_widths ? run(ranks_stats_kernel<DT, 4, false, true>, 4, kTile) : run(ranks_stats_kernel<DT, 4, false, false>, 4, kTile);
        return tile_widths ? run(ranks_stats_kernel<DT, 1, false, true>, 1, kTile) : run(ranks_stats_kernel<DT, 1, false, false>, 1, kTile);
    };
    return dtype == DQ_BF16 ? launch(std::integral_constant<int, DQ_BF16>()) : launch(std::integral_constant<int, DQ_F32>());
}

template <int DT, int RDT>
static hipError_t run_ring(const RingDesc &d, bool mee, const MeeParams *mp, hipStream_t stream)
{
    constexpr bool POOL = RDT != DQ_PHILOX;
    RingArgs<POOL> a;
    memset(&a, 0, sizeof(a));
    bool in = true, out = true, pool = true;
    for (int r = 0; r < d.world; r++) {
        a.src[r] = d.src[r];
        a.out[r] = d.out[r];
        in = in && aligned16(d.src[r]);
        out = out && aligned16(d.out[r]);
        if constexpr (POOL) {
            for (int g = 0; g < 3; g++) {
                a.more.pool[g][r] = d.pool[g][r];
                pool = pool && aligned16(d.pool[g][r]);
                for (int s = 0; s < d.world; s++) a.more.first[g][r][s] = d.first[g][r][s];
            }
        }
    }
    a.mean = d.mean;
    a.total = static_cast<const uint16_t *>(d.total);
    a.order = d.order;
    a.counts = d.counts;
    a.n = d.n;
    a.nsc = (int)((d.n + 255) / 256);
    a.world = d.world;
    a.vec = (in ? 1 : 0) | (out ? 2 : 0) | (pool ? 4 : 0);
    a.key = RandKey{d.seed, 0};
    a.wd = make_world_div(d.world, DT == DQ_F32 ? 4 : 2);
    a.widths = make_width_set(mp, mee);
    const auto parts = [&](auto plans) {
        const auto go = [&](auto kernel, int here) {
            return launch_with(kernel, dim3((unsigned)((a.nsc + here - 1) / here)), dim3(64 * kPartWaves), stream, a);
        };
        constexpr bool PLANS = decltype(plans)::value;
        if constexpr (DT == DQ_BF16 && !POOL) {
            if (a.nsc > fours_to(d.world, PLANS) && (a.vec & 2) != 0)
                return mee ? go(ring_parts_kernel<DT, RDT, true, 8, PLANS>, 2 * kPartWaves) : go(ring_parts_kernel<DT, RDT, false, 8, PLANS>, 2 * kPartWaves);
        }
        return mee ? go(ring_parts_kernel<DT, RDT, true, 4, PLANS>, kPartWaves) : go(ring_parts_kernel<DT, RDT, false, 4, PLANS>, kPartWaves);
    };
    if constexpr (!POOL) {
        if (d.tile_widths) {
            a.more = FromTileWidths{d.tile_widths, d.work, make_rule(d.u, d.u_dev)};
            return parts(std::integral_constant<bool, true>());
        }
    }
    if (a.nsc <= parts_to(d.world, DT == DQ_BF16, mee, POOL)) return parts(std::integral_constant<bool, false>());
    // every run rounds its superchunks per ring chunk up to whole tiles
    const dim3 grid((unsigned)(a.nsc / (kRowsPerWave * d.world) + 4), (unsigned)d.world);
    return mee ? launch_with(ring_kernel<DT, RDT, true>, grid, dim3(64), stream, a)
               : launch_with(ring_kernel<DT, RDT, false>, grid, dim3(64), stream, a);
}

bool ring_plans_itself(int64_t n, int world, int dtype)
{
    return (n + 255) / 256 <= (dtype == DQ_BF16 ? kPlansItself : (world < 4 ? kPlansItselfFew32 : kPlansItself32));
}

hipError_t launch_ring(const RingDesc &d, int dtype, bool mee, const MeeParams *mp, hipStream_t stream)
{
    if (dtype == DQ_BF16) {
        if (d.pooled) return run_ring<DQ_BF16, DQ_BF16>(d, mee, mp, stream);
        return run_ring<DQ_BF16, DQ_PHILOX>(d, mee, mp, stream);
    }
    if (d.pooled) return run_ring<DQ_F32, DQ_F32>(d, mee, mp, stream);
    return run_ring<DQ_F32, DQ_PHILOX>(d, mee, mp, stream);
}

} // namespace dq
