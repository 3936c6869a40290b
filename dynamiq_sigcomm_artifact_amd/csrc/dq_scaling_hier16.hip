// Vectorised hierarchical scaling-quantisation kernels for the production
// shape: chunk 16, superchunk 16 chunks (256 elements), bf16 or fp32 elements,
// strategies 2 (AEE) and 3 (MEE), code widths 2..8.
//
// Work decomposition (wave64, one wave per workgroup, no barriers):
//   * one lane owns one chunk: 16 consecutive elements = 32 B (bf16) / 64 B
//     (fp32) of 128-bit loads, so the chunk maximum needs no cross-lane traffic
//     and every per-chunk scalar is computed once per 16 elements;
//   * one 16-lane DPP row owns one superchunk: the superchunk maximum is four
//     DPP max steps, no LDS;
//   * one wave owns a tile of 4 consecutive superchunks = one contiguous run of
//     4 records (328..1096 bytes) of the packed stream.  Records are 82/146/274
//     bytes and never 16-byte aligned, so a run is assembled in an LDS window
//     whose offset equals the global address modulo 16 and streamed out with
//     aligned 128-bit stores (ragged head / tail bytes singly); packed input is
//     pulled through the same kind of window with aligned 128-bit loads;
//   * one single-wave workgroup per tile, ~50 VGPRs, 8 waves per SIMD: many
//     small workgroups let the dispatcher balance the chip better than a
//     persistent loop with software prefetch did (4.7 -> 5.4 TB/s at 1 GiB), and
//     a 25 MB bucket (6400 tiles) fits the machine in one resident round.
//
// VALU budget.  The quantiser is VALU-bound if written naively (IEEE division,
// NaN/Inf/out-of-range guards per element).  Two measures keep it HBM-bound:
//   * exact division by a chunk-constant: x/d == (float)((double)x * (1/d in
//     double)).  The product carries a relative error < 2^-51 while a binary32
//     quotient of binary32 operands is never closer than 2^-49 (relative) to a
//     rounding boundary without being exactly representable, so the result is
//     the correctly rounded quotient for every finite x -- three full-rate
//     instructions per element instead of the ~10-instruction division
//     expansion;
//   * a wave-uniform fast path: if every element of the wave is finite and
//     below 2^100 and every random value lies in [0, 1] (one packed integer
//     maximum per element finds out), the guards of the general formula cannot
//     fire and are skipped; otherwise the whole wave takes the guarded path.
//     Both paths produce the same bytes on the inputs the fast path accepts.
//
// Numerics: csrc/cuda_hierarchical_mee.cu:203-343 (compress), 345-505
// (decompress) and 526-696 (fused decompress-accumulate-recompress).
#include "dq_hier16_tiles.cuh"
#include "dq_launch.h"

namespace dq {



// ---- kernels ------------------------------------------------------------------------------------

// workgroup = one wave = one tile; the bodies live in dq_hier16_tiles.cuh
template <class MP> struct CompressArgs {
    const void *src;
    const uint8_t *recv;
    uint8_t *dst;
    const void *rnd;
    const int32_t *rows;
    int64_t nsc;
    int vec;
    RandKey key;
    MP mp;
};

template <class MP> struct DecompressArgs {
    const uint8_t *src;
    void *dst;
    const int32_t *rows;
    const uint16_t *stats;
    int64_t limit, nsc;
    int vec;
    MP mp;
};

template <int DT, int RDT, int NBITS, bool MEE, bool FUSED>
__global__ __launch_bounds__(64) void hier16_compress_kernel(CompressArgs<MeeArg<NBITS, MEE>> a)
{
    typedef Rec<NBITS> RC;
    __shared__ __attribute__((aligned(16))) uint8_t win_out[RC::WIN];
    __shared__ __attribute__((aligned(16))) uint8_t win_in[FUSED ? RC::WIN : 16];
    __shared__ float table[(MEE && FUSED) ? (1 << NBITS) : 1];
    const Center none{nullptr, 0, {0.0f, 0.0, 0, 0, 0, 0.0f}};
    const int64_t tile = blockIdx.x;
    compress_tile<DT, RDT, NBITS, MEE, FUSED>(a.src, a.recv, a.dst, a.rnd, row_ids_plain(a.rows), a.nsc, tile, a.vec, a.key, none, a.mp,
                                              win_out, win_in, table, threadIdx.x);
}

// LONG: the wave takes kTilesPerWaveLong consecutive tiles of a row list and fetches their entries with one load (RowIds).
// A variant of its own: the loop costs registers (about 50 instead of 20), which the one-tile kernel need not pay.  The
// encoder has no such variant: its time on long buckets goes into arithmetic, not into the wait for the row list, and
// looped it holds every literal of its tile body in a register of its own (over 100 registers).
constexpr int kTilesPerWaveLong = 4;

template <int DT, int NBITS, bool MEE, bool ADD, bool LONG>
__global__ __launch_bounds__(64) void hier16_decompress_kernel(DecompressArgs<MeeArg<NBITS, MEE>> a)
{
    __shared__ __attribute__((aligned(16))) uint8_t win_in[Rec<NBITS>::WIN];
    __shared__ __attribute__((aligned(16))) uint4 tile_out[64 * Raw16<DT>::kSlots];
    __shared__ float table[MEE ? (1 << NBITS) : 1];
    if constexpr (LONG) {
        const int64_t tile0 = (int64_t)blockIdx.x * kTilesPerWaveLong;
        const RowIds ids = row_ids_prefetch(a.rows, tile0 * kRowsPerWave, kTilesPerWaveLong * kRowsPerWave, a.nsc, threadIdx.x);
#pragma unroll 1
        for (int t = 0; t < kTilesPerWaveLong; t++) {
            decompress_tile<DT, NBITS, MEE, ADD>(a.src, a.dst, ids, a.stats, a.limit, a.nsc, tile0 + t, a.vec, a.mp, win_in, tile_out, table);
            wave_lds_sync(); // window, table and output tile are reused by the next tile
        }
    } else {
        const int64_t tile = blockIdx.x;
        decompress_tile<DT, NBITS, MEE, ADD>(a.src, a.dst, row_ids_plain(a.rows), a.stats, a.limit, a.nsc, tile, a.vec, a.mp, win_in,
                                             tile_out, table);
    }
}

// ---- launchers ------------------------------------------------------------------------------------


// one single-wave workgroup per tile of 4 superchunks (per kTilesPerWaveLong tiles in the LONG decoder)
static inline unsigned grid_for(int64_t nsc, int tiles = 1)
{
    const int64_t per = (int64_t)kRowsPerWave * tiles;
    return (unsigned)((nsc + per - 1) / per);
}

constexpr int64_t kLongRun = 262144; // superchunks of a row list: 16384 waves of four tiles, two rounds of a full chip

// Vectors without a row list that take eight elements per lane (dq_scaling_hier16_short.hip).  Kernels in a graph, us, sixteen -> eight:
//   superchunks                              1,024         2,048         3,072         6,144         10,240        16,384
//   compress  bf16, 4 bits, AEE, pool        2.56 -> 2.51  2.66 -> 2.60  2.70 -> 2.86  3.14 -> 3.30
//             bf16, 5 bits, MEE, drawn       2.84 -> 2.79  2.90 -> 2.82  2.99 -> 3.18  3.54 -> 3.64
//             bf16, 8 bits, MEE, pool        3.07 -> 2.73  3.20 -> 2.83  3.34 -> 3.20  4.09 -> 3.79  6.02 -> 5.31  6.87 -> 6.35
//             bf16, 6 bits, MEE, pool        3.15 -> 2.66  3.21 -> 2.80  3.25 -> 3.08  4.22 -> 3.75  5.88 -> 5.10  7.00 -> 6.18
//             bf16, 7 bits, MEE, pool        3.13 -> 2.73  3.23 -> 2.78  3.40 -> 3.13  4.07 -> 3.74  5.98 -> 5.12  6.87 -> 6.23
//             fp32, 5 bits, MEE, pool                                    3.16 -> 3.08  4.60 -> 4.03  5.94 -> 5.34  7.22 -> 6.79
//             fp32, 6 bits, MEE, pool        3.14 -> 2.64  3.26 -> 2.79  3.34 -> 3.07  5.16 -> 4.49  6.13 -> 5.43  7.49 -> 6.87
//             fp32, 7 bits, MEE, pool        3.17 -> 2.66  3.27 -> 2.78  3.41 -> 3.09  5.19 -> 4.49  6.26 -> 5.43  7.57 -> 6.90
//             fp32, 8 bits, AEE, pool                                    3.09 -> 2.92  4.31 -> 3.89  5.49 -> 5.19  6.92 -> 6.66
//   ring step bf16, 4 bits, AEE, pool        2.73 -> 2.66  2.88 -> 2.80  2.93 -> 3.05  3.73 -> 3.86
//             bf16, 8 bits, MEE, pool        3.46 -> 3.08  3.65 -> 3.25  3.72 -> 3.70  5.19 -> 5.05  6.94 -> 6.56  7.93 -> 8.07
//             fp32, 8 bits, AEE, pool                                    3.51 -> 3.40  5.16 -> 4.74  6.21 -> 5.76  7.73 -> 7.65
//             fp32, 8 bits, MEE, pool        3.69 -> 3.01  3.89 -> 3.17  4.15 -> 3.59  6.02 -> 5.53  7.36 -> 6.68  8.76 -> 8.46
//             bf16, 7 bits, MEE, pool                                    3.60 -> 3.78  4.76 -> 5.09
//   decompress bf16, 4 bits, AEE             2.10 -> 2.03  2.24 -> 2.11  2.39 -> 2.26  2.76 -> 2.67  (8,192: 2.84 -> 3.02)
//             bf16, 7 bits, AEE              2.20 -> 2.10  2.40 -> 2.27  2.45 -> 2.50  (2,560: 2.40 -> 2.39; 2,944: 2.44 -> 2.49)
//             bf16, 7 bits, MEE              2.29 -> 2.14  2.44 -> 2.27  2.49 -> 2.53  (2,560: 2.48 -> 2.44)
//             bf16, 8 bits, AEE              2.10 -> 2.03  2.28 -> 2.12  2.34 -> 2.24
//             bf16, 8 bits, MEE              2.23 -> 2.08  2.42 -> 2.19  2.52 -> 2.36
//             fp32, 8 bits, MEE              2.56 -> 2.18  2.61 -> 2.35  2.76 -> 2.66  3.21 -> 3.51
// (in the columns of 3,072 of 5 bits, of 8 bits in AEE encoding, and of the ring step at 7: 3,584).  Up to 2,048 superchunks every wave of eights has a SIMD to
// itself, and half of the SIMDs would have none of sixteens.  Beyond, a short chain is worth the chunk's work done twice where the chain is
// long and nothing is drawn: at 16-bit elements MEE from 6 bits on, at 32 bits from 5 bits MEE and from 8 bits AEE on; a ring step, which decodes on top, at
// 8 bits only, and less far: with vectors that no cache holds, us, MEE bf16 x 9,728 7.19 -> 6.90, x 10,240 7.38 -> 7.30, x 11,264 7.78 -> 7.68 but read
// again 5.52 -> 5.75, x 12,288 5.62 -> 5.97; fp32 x 10,240 8.45 -> 8.34, x 12,288 9.16 -> 9.29; AEE fp32 x 9,216 7.17 -> 7.11, x 10,240 7.51 -> 7.68,
// x 12,288 8.30 -> 8.62.  (Compress of 7 bits in MEE, bf16, x 12,288 6.08 -> 5.50, x 16,384 7.05 -> 6.73, but the same vector again and
// again 4.68 -> 4.86, 5.32 -> 5.50.)  Half a chunk of 7-bit codes is seven bytes that a lane reads one by one, and 16-bit elements do not hide that as long.
constexpr int64_t kShortRun = 2048, kShortDecode = 3072, kShortDecode7 = 2560, kLongChainRun = 16384, kLongChainStepMee = 10240, kLongChainStep = 9216;

static bool short_encode(int64_t nsc, bool fused, int nbits, bool f32, bool mee, bool drawn)
{
    if (nsc <= kShortRun) return true;
    if (drawn) return false;
    if (fused) return nbits == 8 && (mee ? nsc <= kLongChainStepMee : f32 && nsc <= kLongChainStep);
    return nsc <= kLongChainRun && (mee ? nbits >= (f32 ? 5 : 6) : nbits == 8 && f32);
}

template <int DT, int RDT, int NBITS, bool MEE>
static hipError_t run_compress(const void *src, const uint8_t *recv, uint8_t *dst, const void *rnd, const int32_t *rows,
                               int64_t nsc, bool fused, const MeeParams &mp, RandKey key, hipStream_t stream)
{
    const CompressArgs<MeeArg<NBITS, MEE>> args{src, recv, dst, rnd, rows, nsc, (aligned16(src) ? 1 : 0) | (aligned16(rnd) ? 2 : 0), key,
                                                make_arg<NBITS, MEE>(mp)};
    static_assert(sizeof(args) <= 128, "beyond, a launch takes 0.8 us longer (MeeTable)");
    const dim3 grid(grid_for(nsc)), block(64);
    if (fused) return launch_with(hier16_compress_kernel<DT, RDT, NBITS, MEE, true>, grid, block, stream, args);
    return launch_with(hier16_compress_kernel<DT, RDT, NBITS, MEE, false>, grid, block, stream, args);
}

template <int DT, int NBITS, bool MEE>
static hipError_t run_decompress(const uint8_t *src, void *dst, const int32_t *rows, const uint16_t *stats, int64_t limit,
                                 int64_t nsc, int add, const MeeParams &mp, hipStream_t stream)
{
    const DecompressArgs<MeeArg<NBITS, MEE>> args{src, dst, rows, stats, limit, nsc, aligned16(dst) ? 1 : 0, make_arg<NBITS, MEE>(mp)};
    static_assert(sizeof(args) <= 128, "beyond, a launch takes 0.8 us longer (MeeTable)");
    const dim3 block(64);
    if (rows && nsc >= kLongRun && !add) {
        // a long row list (the decoder of the grouped pipelines on the reference's whole-model buckets)
        return launch_with(hier16_decompress_kernel<DT, NBITS, MEE, false, true>, dim3(grid_for(nsc, kTilesPerWaveLong)), block, stream, args);
    }
    const dim3 grid(grid_for(nsc));
    if (add) return launch_with(hier16_decompress_kernel<DT, NBITS, MEE, true, false>, grid, block, stream, args);
    return launch_with(hier16_decompress_kernel<DT, NBITS, MEE, false, false>, grid, block, stream, args);
}

#define DQ_COMMA ,

static hipError_t dispatch_compress(const void *src, const uint8_t *recv, uint8_t *dst, const void *rnd,
                                    const int32_t *rows, int64_t nsc, bool fused, int nbits, int dtype, bool mee,
                                    const MeeParams &mp, hipStream_t stream, const RandKey *philox = nullptr)
{
    if (!rows && short_encode(nsc, fused, nbits, (dtype & 0xf) == DQ_F32, mee, philox != nullptr))
        return launch_hier16_short_compress(src, fused ? recv : nullptr, dst, rnd, nsc, nbits, dtype, mee, mp, philox, stream);
    const bool rb16 = (dtype & DQ_RAND_BF16) != 0;
    dtype &= 0xf;
    const RandKey key = philox ? *philox : RandKey{0, 0};
    if (philox) {
        if (dtype == DQ_BF16) {
            DQ_NBITS_MEE(run_compress, DQ_BF16 DQ_COMMA DQ_PHILOX, src, recv, dst, rnd, rows, nsc, fused, mp, key, stream)
        } else {
            DQ_NBITS_MEE(run_compress, DQ_F32 DQ_COMMA DQ_PHILOX, src, recv, dst, rnd, rows, nsc, fused, mp, key, stream)
        }
    }
    if (dtype == DQ_BF16) {
        DQ_NBITS_MEE(run_compress, DQ_BF16 DQ_COMMA DQ_BF16, src, recv, dst, rnd, rows, nsc, fused, mp, key, stream)
    } else if (rb16) {
        DQ_NBITS_MEE(run_compress, DQ_F32 DQ_COMMA DQ_BF16, src, recv, dst, rnd, rows, nsc, fused, mp, key, stream)
    } else {
        DQ_NBITS_MEE(run_compress, DQ_F32 DQ_COMMA DQ_F32, src, recv, dst, rnd, rows, nsc, fused, mp, key, stream)
    }
}

hipError_t launch_hier16_compress(const void *src, uint8_t *dst, const void *rnd, int64_t n, int nbits, int dtype,
                                  bool mee, const MeeParams &mp, hipStream_t stream)
{
    return dispatch_compress(src, nullptr, dst, rnd, nullptr, n / 256, false, nbits, dtype, mee, mp, stream);
}

hipError_t launch_hier16_dec_comp(const uint8_t *recv, const void *inp, uint8_t *send, const void *rnd, int64_t n,
                                  int nbits, int dtype, bool mee, const MeeParams &mp, hipStream_t stream)
{
    return dispatch_compress(inp, recv, send, rnd, nullptr, n / 256, true, nbits, dtype, mee, mp, stream);
}

hipError_t launch_hier16_compress_philox(const void *src, const uint8_t *recv, uint8_t *dst, int64_t n, int nbits, int dtype,
                                         bool mee, const MeeParams &mp, uint64_t seed, uint64_t step, hipStream_t stream)
{
    const RandKey key{seed, step};
    return dispatch_compress(src, recv, dst, nullptr, nullptr, n / 256, recv != nullptr, nbits, dtype, mee, mp, stream, &key);
}

hipError_t launch_hier16_compress_rows(const void *src, const uint8_t *recv, const int32_t *rows, uint8_t *dst,
                                       const void *rnd, int64_t nrows, int nbits, int dtype, bool mee,
                                       const MeeParams &mp, hipStream_t stream)
{
    return dispatch_compress(src, recv, dst, rnd, rows, nrows, recv != nullptr, nbits, dtype, mee, mp, stream);
}

static hipError_t dispatch_decompress(const uint8_t *src, void *dst, const int32_t *rows, const uint16_t *stats,
                                      int64_t limit, int64_t nsc, int nbits, int dtype, bool mee, const MeeParams &mp,
                                      int add, hipStream_t stream)
{
    if (!rows && !stats && !add && limit >= nsc * 256 && nsc <= (nbits == 7 && (dtype & 0xf) == DQ_BF16 ? kShortDecode7 : kShortDecode))
        return launch_hier16_short_decompress(src, dst, nsc, nbits, dtype, mee, mp, stream);
    if ((dtype & 0xf) == DQ_BF16) {
        DQ_NBITS_MEE(run_decompress, DQ_BF16, src, dst, rows, stats, limit, nsc, add, mp, stream)
    } else {
        DQ_NBITS_MEE(run_decompress, DQ_F32, src, dst, rows, stats, limit, nsc, add, mp, stream)
    }
}

hipError_t launch_hier16_decompress(const uint8_t *src, void *dst, int64_t n, int nbits, int dtype, bool mee,
                                    const MeeParams &mp, int add, hipStream_t stream)
{
    return dispatch_decompress(src, dst, nullptr, nullptr, n, n / 256, nbits, dtype, mee, mp, add, stream);
}

hipError_t launch_hier16_decompress_rows(const uint8_t *src, void *dst, const int32_t *rows, const void *stats,
                                         int64_t limit, int64_t nrows, int nbits, int dtype, bool mee,
                                         const MeeParams &mp, int add, hipStream_t stream)
{
    return dispatch_decompress(src, dst, rows, static_cast<const uint16_t *>(stats), limit, nrows, nbits, dtype, mee, mp,
                               add, stream);
}

} // namespace dq
