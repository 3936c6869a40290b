// The codec of dq_scaling_hier16.hip for vectors that give it only one or two waves per SIMD: eight elements per lane instead of
// sixteen, two superchunks per wave instead of four.
//
// A launch then has twice the waves, each with half the chain of instructions between its loads and its stores; what a chunk costs once
// (scale, step, their reciprocals, the draws) is worked out twice, which is why longer vectors keep sixteen.  Bound: latency, of the launch
// (2 us), the loads and the chain.  Up to 2,048 superchunks 2 to 15 % less than with sixteen; the figures stand where the line is drawn
// (dq_scaling_hier16.hip).
//
// Layout: a chunk is a pair of lanes, a superchunk half a wave.  Eight codes are NBITS whole bytes, so a lane puts its half of the chunk's
// code bytes into the window by itself, and the second of the pair the scale byte.  Records, windows and numbers are those of the
// other kernels (dq_hier16_tiles.cuh), bit for bit.
//
// Numerics: csrc/cuda_hierarchical_mee.cu:203-343 (compress), 345-505 (decompress) and 526-696 (fused
// decompress-accumulate-recompress).
#include "dq_hier16_tiles.cuh"
#include "dq_launch.h"

namespace dq {

namespace {

constexpr int kPart = 8;                  // elements per lane
constexpr int kParts = 256 / kPart;       // lanes per superchunk
constexpr int kRows = 64 / kParts;        // superchunks per wave

template <class MP> struct ShortCompressArgs {
    const void *src;
    const uint8_t *recv;
    uint8_t *dst;
    const void *rnd;
    int64_t nsc;
    int vec;
    RandKey key;
    MP mp;
};

template <class MP> struct ShortDecompressArgs {
    const uint8_t *src;
    void *dst;
    int64_t nsc;
    int vec;
    MP mp;
};

// a run of at most 64 aligned pieces (window_fetch and window_commit take up to 128)
__device__ __forceinline__ u32x4 run_fetch(const uint8_t *g, int total, int lane)
{
    const int mis = (int)(reinterpret_cast<uintptr_t>(g) & 15);
    return reinterpret_cast<const u32x4 *>(g - mis)[min(lane, ((mis + total + 15) >> 4) - 1)];
}

__device__ __forceinline__ int run_commit(uint8_t *win, const u32x4 &piece, const uint8_t *g, int total, int lane)
{
    const int mis = (int)(reinterpret_cast<uintptr_t>(g) & 15);
    if (lane < (mis + total + 15) >> 4) reinterpret_cast<u32x4 *>(win)[lane] = piece;
    return mis;
}

// what the codes of a lane take: NBITS bytes
template <int NBITS> struct PartWords {
    static constexpr int kWords = (kPart * NBITS + 31) / 32;
    uint32_t w[kWords];
    __device__ __forceinline__ void read(const uint8_t *p)
    {
#pragma unroll
        for (int k = 0; k < kWords; k++) w[k] = 0;
#pragma unroll
        for (int k = 0; k < NBITS; k++) w[k >> 2] |= (uint32_t)p[k] << (8 * (k & 3));
    }
    __device__ __forceinline__ void write(uint8_t *p) const
    {
#pragma unroll
        for (int k = 0; k < NBITS; k++) p[k] = (uint8_t)(w[k >> 2] >> (8 * (k & 3)));
    }
};

template <int NBITS> __device__ __forceinline__ uint32_t unit_of(const uint8_t *rec)
{
    return (uint32_t)rec[16 * Rec<NBITS>::CB] | ((uint32_t)rec[16 * Rec<NBITS>::CB + 1] << 8);
}

template <int DT, int RDT, int NBITS, bool MEE, bool FUSED>
__global__ __launch_bounds__(64) void hier16_short_compress_kernel(ShortCompressArgs<MeeArg<NBITS, MEE>> a)
{
    typedef Rec<NBITS> RC;
    static_assert(window_bytes<NBITS>(kRows) <= 64 * 16, "a run is one piece per lane");
    __shared__ __attribute__((aligned(16))) uint8_t win_out[window_bytes<NBITS>(kRows)];
    __shared__ __attribute__((aligned(16))) uint8_t win_in[FUSED ? window_bytes<NBITS>(kRows) : 16];
    __shared__ float table[(MEE && FUSED) ? (1 << NBITS) : 1];
    const int lane = threadIdx.x, row = lane / kParts, part = lane % kParts, j = part >> 1, second = part & 1;
    const int64_t sc0 = (int64_t)blockIdx.x * kRows;
    const int rows_here = (int)min((int64_t)kRows, a.nsc - sc0), total = rows_here * RC::REC;
    const bool active = row < rows_here;

    u32x4 piece;
    if (FUSED) piece = run_fetch(a.recv + sc0 * RC::REC, total, lane);
    TableRegs<NBITS> tr;
    if (MEE && FUSED) tr = table_fetch<NBITS>(a.mp, lane);
    RawPart<DT, kPart> v;
    RawPart<RDT, kPart> r;
    v.zero();
    r.halves();
    if (active) {
        const int64_t e0 = (sc0 + row) * 256 + part * kPart;
        if constexpr (RDT != DQ_PHILOX) r.load(a.rnd, e0, a.vec & 2);
        v.load(a.src, e0, a.vec & 1);
    }
    if constexpr (RDT == DQ_PHILOX) r.generate(a.key, (sc0 + row) * 16 + j, second);

    if (FUSED) {
        const int mis = run_commit(win_in, piece, a.recv + sc0 * RC::REC, total, lane);
        if (MEE) table_commit<NBITS>(table, tr, lane);
        wave_lds_sync();
        if (active) {
            const uint8_t *rec = win_in + mis + row * RC::REC;
            PartWords<NBITS> codes;
            codes.read(rec + j * RC::CB + second * NBITS);
            float t[kPart];
#pragma unroll
            for (int i = 0; i < kPart; i++) t[i] = v.get(i);
            chunk_decode<NBITS, MEE, true, kPart>(codes.w, rec[j * RC::CB + RC::PB], unit_of<NBITS>(rec), table, t);
            v.set(t); // rounds the sum to the element type
        }
    }

    PartWords<NBITS> codes;
    uint32_t q, ub;
    const uint32_t amax = chunk_max<kPart>(v.absmax_bits());
    const bool lane_fast = amax <= kFastMaxBits && r.unit_interval();
    if (DQ_UNLIKELY(__builtin_amdgcn_ballot_w64(!lane_fast) != 0))
        chunk_encode_guarded<NBITS, MEE, kPart>(v, r, a.mp, codes.w, q, ub);
    else
        chunk_encode_fast<NBITS, MEE, kPart>(v, r, amax, a.mp, codes.w, q, ub);

    uint8_t *gout = a.dst + sc0 * RC::REC;
    const int mis = (int)(reinterpret_cast<uintptr_t>(gout) & 15);
    if (active) {
        uint8_t *rec = win_out + mis + row * RC::REC;
        codes.write(rec + j * RC::CB + second * NBITS);
        if (second) rec[j * RC::CB + RC::PB] = (uint8_t)q;
        if (part == 0) {
            rec[16 * RC::CB] = (uint8_t)ub;
            rec[16 * RC::CB + 1] = (uint8_t)(ub >> 8);
        }
    }
    wave_lds_sync();
    window_flush(win_out, gout, mis, total, lane);
}

template <int DT, int NBITS, bool MEE>
__global__ __launch_bounds__(64) void hier16_short_decompress_kernel(ShortDecompressArgs<MeeArg<NBITS, MEE>> a)
{
    typedef Rec<NBITS> RC;
    __shared__ __attribute__((aligned(16))) uint8_t win_in[window_bytes<NBITS>(kRows)];
    __shared__ float table[MEE ? (1 << NBITS) : 1];
    const int lane = threadIdx.x, row = lane / kParts, part = lane % kParts, j = part >> 1, second = part & 1;
    const int64_t sc0 = (int64_t)blockIdx.x * kRows;
    const int rows_here = (int)min((int64_t)kRows, a.nsc - sc0), total = rows_here * RC::REC;

    const u32x4 piece = run_fetch(a.src + sc0 * RC::REC, total, lane);
    TableRegs<NBITS> tr;
    if (MEE) tr = table_fetch<NBITS>(a.mp, lane);
    const int mis = run_commit(win_in, piece, a.src + sc0 * RC::REC, total, lane);
    if (MEE) table_commit<NBITS>(table, tr, lane);
    wave_lds_sync();
    if (row >= rows_here) return;
    const uint8_t *rec = win_in + mis + row * RC::REC;
    PartWords<NBITS> codes;
    codes.read(rec + j * RC::CB + second * NBITS);
    float t[kPart];
    chunk_decode<NBITS, MEE, false, kPart>(codes.w, rec[j * RC::CB + RC::PB], unit_of<NBITS>(rec), table, t);
    RawPart<DT, kPart> out;
    out.set(t);
    out.store(a.dst, (sc0 + row) * 256 + part * kPart, a.vec);
}

static unsigned waves_for(int64_t nsc) { return (unsigned)((nsc + kRows - 1) / kRows); }

template <int DT, int RDT, int NBITS, bool MEE>
static hipError_t run_compress(const void *src, const uint8_t *recv, uint8_t *dst, const void *rnd, int64_t nsc, const MeeParams &mp,
                               RandKey key, hipStream_t stream)
{
    const ShortCompressArgs<MeeArg<NBITS, MEE>> args{src, recv, dst, rnd, nsc, (aligned16(src) ? 1 : 0) | (aligned16(rnd) ? 2 : 0), key,
                                                     make_arg<NBITS, MEE>(mp)};
    static_assert(sizeof(args) <= 128, "beyond, a launch takes 0.8 us longer (MeeTable)");
    if (recv) return launch_with(hier16_short_compress_kernel<DT, RDT, NBITS, MEE, true>, dim3(waves_for(nsc)), dim3(64), stream, args);
    return launch_with(hier16_short_compress_kernel<DT, RDT, NBITS, MEE, false>, dim3(waves_for(nsc)), dim3(64), stream, args);
}

template <int DT, int NBITS, bool MEE>
static hipError_t run_decompress(const uint8_t *src, void *dst, int64_t nsc, const MeeParams &mp, hipStream_t stream)
{
    const ShortDecompressArgs<MeeArg<NBITS, MEE>> args{src, dst, nsc, aligned16(dst) ? 1 : 0, make_arg<NBITS, MEE>(mp)};
    static_assert(sizeof(args) <= 128, "beyond, a launch takes 0.8 us longer (MeeTable)");
    return launch_with(hier16_short_decompress_kernel<DT, NBITS, MEE>, dim3(waves_for(nsc)), dim3(64), stream, args);
}

} // namespace

#define DQ_COMMA ,

hipError_t launch_hier16_short_compress(const void *src, const uint8_t *recv, uint8_t *dst, const void *rnd, int64_t nsc, int nbits,
                                        int dtype, bool mee, const MeeParams &mp, const RandKey *philox, hipStream_t stream)
{
    const bool rb16 = (dtype & DQ_RAND_BF16) != 0;
    dtype &= 0xf;
    const RandKey key = philox ? *philox : RandKey{0, 0};
    if (philox) {
        if (dtype == DQ_BF16) {
            DQ_NBITS_MEE(run_compress, DQ_BF16 DQ_COMMA DQ_PHILOX, src, recv, dst, rnd, nsc, mp, key, stream)
        } else {
            DQ_NBITS_MEE(run_compress, DQ_F32 DQ_COMMA DQ_PHILOX, src, recv, dst, rnd, nsc, mp, key, stream)
        }
    }
    if (dtype == DQ_BF16) {
        DQ_NBITS_MEE(run_compress, DQ_BF16 DQ_COMMA DQ_BF16, src, recv, dst, rnd, nsc, mp, key, stream)
    } else if (rb16) {
        DQ_NBITS_MEE(run_compress, DQ_F32 DQ_COMMA DQ_BF16, src, recv, dst, rnd, nsc, mp, key, stream)
    } else {
        DQ_NBITS_MEE(run_compress, DQ_F32 DQ_COMMA DQ_F32, src, recv, dst, rnd, nsc, mp, key, stream)
    }
}

hipError_t launch_hier16_short_decompress(const uint8_t *src, void *dst, int64_t nsc, int nbits, int dtype, bool mee, const MeeParams &mp,
                                          hipStream_t stream)
{
    if ((dtype & 0xf) == DQ_BF16) {
        DQ_NBITS_MEE(run_decompress, DQ_BF16, src, dst, nsc, mp, stream)
    } else {
        DQ_NBITS_MEE(run_decompress, DQ_F32, src, dst, nsc, mp, stream)
    }
}

} // namespace dq
