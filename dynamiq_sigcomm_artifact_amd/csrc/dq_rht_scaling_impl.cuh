// Blocked randomized Hadamard transform fused with the hierarchical chunk-16 quantiser, and -- with the same lane = chunk
// structure -- the passes of the transform alone (rht_tile_kernel, rht_tile_split_kernel, rht_strided_kernel), with or
// without THC's / EDEN's quantisers at the ends; dq_hadamard.hip plans which passes a transform takes.
//
// rht_blocked followed by scaling_compress moves every element through HBM three times (read, write the
// rotated vector, read it again); the inverse pair likewise.  Here the rotated tile never leaves the
// workgroup: a workgroup owns a tile of 2^kt consecutive floats (whole transform blocks of up to 2^15) in
// LDS.  One lane owns one chunk of 16 consecutive floats at both ends: it loads the chunk (64 bytes), flips
// the signs and does the stages of strides 1..8 on its registers, the remaining stages run as LDS passes of
// up to five stages each, and the lane then reads its chunk back and quantises it.  The LDS index is padded by
// one float per 32 (dq_fwht.cuh): the chunk-wise accesses, the passes and the coalesced stores are then all free
// of bank conflicts.  The inverse kernel decodes records into registers, does the first
// stages there, finishes in LDS and stores fp32 with coalesced 16-byte stores.
//
// Results are bit for bit those of the two-call sequences: the butterflies run in the same order
// (dq_fwht.cuh), the scale is applied by the same single multiplication, and the quantiser is the tile body
// of the hier16 kernels (dq_hier16_tiles.cuh).  Numerics of the quantiser: csrc/cuda_hierarchical_mee.cu:203-505;
// of the transform: csrc/cuda_hadamard.cu:66-157,534-605 with the sign flip and 1/sqrt(block) of
// testbed_evaluation/new_comm_hooks/thc_hooks.py:95-107 folded in.
//
// This file is the body of several translation units (the kernel templates have a few hundred instantiations between
// them, and one compiler run over all of them takes minutes): each .hip file that includes it defines DQ_RHT_PART as the
// set of entry points it emits --
//   DQ_RHT_TRANSFORM          launch_rht_tile, launch_rht_strided, launch_rht_compress (the dispatcher), the matrix-core variant
//   DQ_RHT_COMPRESS_PHILOX    launch_rht_compress_philox      (dq_rht_compress_philox.hip)
//   DQ_RHT_COMPRESS_BF16      launch_rht_compress_bf16_pool   (dq_rht_compress_bf16.hip)
//   DQ_RHT_COMPRESS_F32       launch_rht_compress_f32_pool    (dq_rht_compress_f32.hip)
//   DQ_RHT_DECOMPRESS         launch_irht_decompress          (dq_rht_decompress.hip)
// -- and only the templates those use are instantiated there.
#pragma once

#include <algorithm>
#include <type_traits>

#include "dq_fwht.cuh"
#include "dq_hier16_tiles.cuh"
#include "dq_launch.h"
#include "dq_sums.cuh"

#define DQ_RHT_TRANSFORM 1
#define DQ_RHT_COMPRESS_PHILOX 2
#define DQ_RHT_COMPRESS_BF16 4
#define DQ_RHT_COMPRESS_F32 8
#define DQ_RHT_DECOMPRESS 16
#ifndef DQ_RHT_PART
#error "define DQ_RHT_PART before including dq_rht_scaling_impl.cuh"
#endif

namespace dq {

namespace {

struct RhtTileArgs {
    const void *sign;  // may be null: fp32 +-1 values, or (sign_bits) one bit per element, set = negative
    int sign_bits;
    int64_t n;         // elements, a multiple of 256 and of the transform block
    int kt;            // log2 tile elements
    int kb;            // log2 transform block, <= kt
    float scale;
    int vec;           // 16-byte accesses to the fp32 vector and the sign vector allowed
};

// The diagonal drawn where it is applied (sign is then null); flip4 and flip16 serve it.  A type of its own: the kernels
// fused with the codec run on 64 registers, and a test for a seed that they never have costs them time (2^30 elements there
// and back 2134 us with it, 2118 without, as before there were drawn diagonals).
struct RhtPassArgs : RhtTileArgs {
    SignSeed gen;
};
// threads of a tile of 2^kt elements: a chunk each.  (Asked of the launch, their number costs 256 bytes of hidden arguments.)
__host__ __device__ constexpr int tile_threads(int kt) { return kt < 10 ? 64 : (kt > 14 ? 1024 : 1 << (kt - 4)); }

template <bool ENDS> using PassArgs = typename std::conditional<ENDS, RhtPassArgs, RhtTileArgs>::type;

// Element g of the diagonal of rand_diag (srrcomp.py:61-106; rand_diag_word of dq_hadamard.hip in 32-bit arithmetic: only
// the low word of every product is used, and the one carry that is, of the addition, is added back by hand).  The two
// congruential steps at its head are one affine function of the column, so the next column's state is an addition away: two
// multiplications at a quarter of the rate are left, about 15 instruction slots per element (25 with four).  Cheaper than a
// launch that writes the bits while the vector is short (the rule is in launch_eden_compress).
constexpr uint32_t kDiagFirst = 1103515245u, kDiagSecond = 1140671485u, kDiagStep = kDiagFirst * kDiagSecond;

__device__ __forceinline__ uint32_t rand_diag_state(const SignSeed &s, uint32_t j)
{
    return kDiagStep * j + (kDiagSecond * (kDiagFirst * s.ss + 12345u + s.ss) + 12820163u + s.ss);
}

__device__ __forceinline__ uint32_t rand_diag_mix(uint32_t r)
{
    const uint32_t q = r + 0x9e3779b9u;
    const uint32_t carry = q < r ? 0x10000u : 0u;
    r = (q ^ ((q >> 16) | carry)) * 0x85ebca6bu;
    r = (r ^ (r >> 13)) * 0xc2b2ae35u;
    return r ^ (r >> 16);
}

__device__ __forceinline__ uint32_t rand_diag_column(const SignSeed &s, uint32_t j) { return rand_diag_mix(rand_diag_state(s, j)); }

// the sign bit of element j of segment k: +1 where the nibble is >= 8
__device__ __forceinline__ uint32_t nibble_negative(uint32_t r, uint32_t k) { return ~(r << (28 - 4 * k)) & 0x80000000u; }

__device__ __forceinline__ uint32_t rand_diag_negative(const SignSeed &s, uint32_t k, uint32_t j)
{
    return nibble_negative(rand_diag_column(s, j), k);
}

// the sign flip of elements g .. g + 3 (g a multiple of 4) / of element g.  A packed sign flips the sign bit,
// which is what the multiplication by -1.0f does to every number
__device__ __forceinline__ void flip4(float4 &v, const RhtTileArgs &a, int64_t g)
{
    if (!a.sign) return;
    if (a.sign_bits) {
        const uint32_t w = static_cast<const uint32_t *>(a.sign)[g >> 5] >> (g & 31);
        v.x = __uint_as_float(__float_as_uint(v.x) ^ ((w & 1u) << 31));
        v.y = __uint_as_float(__float_as_uint(v.y) ^ ((w & 2u) << 30));
        v.z = __uint_as_float(__float_as_uint(v.z) ^ ((w & 4u) << 29));
        v.w = __uint_as_float(__float_as_uint(v.w) ^ ((w & 8u) << 28));
    } else {
        const float4 s = *reinterpret_cast<const float4 *>(static_cast<const float *>(a.sign) + g);
        v.x *= s.x; v.y *= s.y; v.z *= s.z; v.w *= s.w;
    }
}

__device__ __forceinline__ void flip4(float4 &v, const RhtPassArgs &a, int64_t g)
{
    if (a.gen.bits != 0) {
        const uint32_t k = (uint32_t)(g >> a.gen.bits), j = (uint32_t)g & ((1u << a.gen.bits) - 1u); // the four share a segment
        const uint32_t r = rand_diag_state(a.gen, j);
        v.x = __uint_as_float(__float_as_uint(v.x) ^ nibble_negative(rand_diag_mix(r), k));
        v.y = __uint_as_float(__float_as_uint(v.y) ^ nibble_negative(rand_diag_mix(r + kDiagStep), k));
        v.z = __uint_as_float(__float_as_uint(v.z) ^ nibble_negative(rand_diag_mix(r + 2 * kDiagStep), k));
        v.w = __uint_as_float(__float_as_uint(v.w) ^ nibble_negative(rand_diag_mix(r + 3 * kDiagStep), k));
        return;
    }
    flip4(v, static_cast<const RhtTileArgs &>(a), g);
}

__device__ __forceinline__ float flip1(float v, const RhtTileArgs &a, int64_t g)
{
    if (!a.sign) return v;
    if (a.sign_bits) {
        const uint32_t w = static_cast<const uint32_t *>(a.sign)[g >> 5] >> (g & 31);
        return __uint_as_float(__float_as_uint(v) ^ (w << 31));
    }
    return v * static_cast<const float *>(a.sign)[g];
}

// 16 consecutive elements starting at g (a multiple of 16), sign-flipped; zeros at and beyond n
__device__ __forceinline__ void load_chunk(float (&v)[16], const float *__restrict__ x, const RhtTileArgs &a, int64_t g)
{
    if (g + 16 <= a.n && a.vec) {
        const float4 *p = reinterpret_cast<const float4 *>(x + g);
        float4 q[4] = {p[0], p[1], p[2], p[3]};
        if (a.sign && a.sign_bits) {
            const uint32_t w = static_cast<const uint32_t *>(a.sign)[g >> 5] >> (g & 31);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                q[k].x = __uint_as_float(__float_as_uint(q[k].x) ^ (((w >> (4 * k)) & 1u) << 31));
                q[k].y = __uint_as_float(__float_as_uint(q[k].y) ^ (((w >> (4 * k + 1)) & 1u) << 31));
                q[k].z = __uint_as_float(__float_as_uint(q[k].z) ^ (((w >> (4 * k + 2)) & 1u) << 31));
                q[k].w = __uint_as_float(__float_as_uint(q[k].w) ^ (((w >> (4 * k + 3)) & 1u) << 31));
            }
        } else if (a.sign) {
            const float4 *sp = reinterpret_cast<const float4 *>(static_cast<const float *>(a.sign) + g);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float4 sg = sp[k];
                q[k].x *= sg.x; q[k].y *= sg.y; q[k].z *= sg.z; q[k].w *= sg.w;
            }
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            v[4 * k] = q[k].x; v[4 * k + 1] = q[k].y; v[4 * k + 2] = q[k].z; v[4 * k + 3] = q[k].w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = g + i < a.n ? flip1(x[g + i], a, g + i) : 0.0f;
    }
}

// floats of LDS holding the padded tile, rounded up so that what follows is 16-byte aligned
__host__ __device__ constexpr int padded_tile_floats(int kt) { return padded_floats(1 << kt); }

// The stages of strides 1..8 of 64 chunks as one matrix product on the matrix cores: Y = X H16, X the wave's 64 x 16
// block of chunks, H16[i][j] = (-1)^popcount(i & j).  v_mfma_f32_16x16x4_f32 takes a 16 x 4 slice of X (lane l: row
// l % 16, column l / 16 of the slice) against a 4 x 16 slice of H16 (lane l: row l / 16, column l % 16) and leaves a
// 16 x 16 block of Y with lane l holding rows 4 (l / 16) .. + 3 of column l % 16.  With slice j made of the columns
// 4 (l / 16) + j of X, a lane's four slice operands are one aligned float4 of its row.  The sums of a product are not
// formed in the butterfly order, so the last bits differ from the stage-by-stage transform (the reference's own
// tolerance for the transform is 1e-5 relative): a measurement variant, not the default.
typedef float mfma_f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void chunk_stages_mfma16(const float *__restrict__ x, const RhtTileArgs &a, int64_t origin, int chunk0,
                                                    int lane, float *lds)
{
    const int m = lane & 15, kk = lane >> 4;
    float h[4];
#pragma unroll
    for (int j = 0; j < 4; j++) h[j] = (__builtin_popcount((4 * kk + j) & m) & 1) ? -1.0f : 1.0f;
#pragma unroll
    for (int b = 0; b < 4; b++) {
        const int64_t g = origin + (int64_t)(chunk0 + 16 * b + m) * 16 + 4 * kk;
        float4 q = *reinterpret_cast<const float4 *>(x + g);
        flip4(q, a, g);
        mfma_f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(q.x, h[0], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(q.y, h[1], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(q.z, h[2], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(q.w, h[3], acc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) lds[chunk_word(chunk0 + 16 * b + 4 * kk + i) + m] = acc[i];
    }
}

template <int RDT, int NBITS, bool MEE, bool MFMA16 = false>
__global__ __attribute__((amdgpu_waves_per_eu(8, 8))) void rht_compress_kernel(const float *__restrict__ x, uint8_t *__restrict__ dst, const void *__restrict__ rnd,
                                    RhtTileArgs a, int rvec, RandKey key, MeeArg<NBITS, MEE> mp)
{
    typedef Rec<NBITS> RC;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = threadIdx.x, nthreads = tile_threads(a.kt);
    const int tile = 1 << a.kt;
    const int64_t origin = (int64_t)blockIdx.x << a.kt;

    // every lane loads chunks of 16 consecutive floats (64 bytes, as the quantiser's own kernels do), flips the
    // signs and does the stages of strides 1..8 on its registers; elements beyond n (a ragged last tile) are zero
    const int nchunks = tile >> 4;
    if constexpr (MFMA16) {
        // whole tiles, 16-byte aligned, blocks of at least 16 (checked by the launcher)
        for (int c0 = (tid >> 6) * 64; c0 < nchunks; c0 += nthreads) chunk_stages_mfma16(x, a, origin, c0, tid & 63, lds);
    } else {
    for (int c = tid; c < nchunks; c += nthreads) {
        float v[16];
        load_chunk(v, x, a, origin + c * 16);
        chunk_stages(v, a.kb);
        float *mine = lds + chunk_word(c);
#pragma unroll
        for (int i = 0; i < 16; i++) mine[i] = v[i];
    }
    }
    fwht_lds_stages_after4(lds, a.kt, a.kb, tid, nthreads);

    // quantise: the tile holds one run of 64 chunks (4 superchunks, one contiguous run of records) per wave.
    // Every wave first takes its chunks into registers; after the barrier the tile is dead and the record
    // windows reuse its LDS.
    const int lane = tid & 63, wave = tid >> 6;
    const int64_t nsc_total = a.n >> 8, sc_origin = origin >> 8;
    const int tile_sc = max(1, tile >> 8);
    const int64_t sc0 = sc_origin + wave * kRowsPerWave;
    const int rows_here = (wave * kRowsPerWave < tile_sc && sc0 < nsc_total)
                              ? (int)min((int64_t)min(kRowsPerWave, tile_sc - wave * kRowsPerWave), nsc_total - sc0)
                              : 0;
    Raw16<DQ_F32> v;
    Raw16<RDT> r;
    if ((lane >> 4) < rows_here) {
        if constexpr (RDT == DQ_PHILOX)
            r.generate(key, sc0 * 16 + lane);
        else
            r.load(rnd, (sc0 * 16 + lane) * 16, rvec);
        const float *mine = lds + chunk_word(wave * 64 + lane);
#pragma unroll
        for (int i = 0; i < 16; i++) v.w[i] = __float_as_uint(mine[i] * a.scale);
    } else {
        v.zero();
        r.halves();
    }
    __syncthreads();
    if (rows_here > 0)
        encode_store_run<NBITS, MEE, kRowsPerWave, false>(v, r, mp, dst + sc0 * RC::REC, rows_here, reinterpret_cast<uint8_t *>(lds) + wave * RC::WIN, threadIdx.x & 63);
}

// blocks below 2^10 elements, several to a tile
template <int NBITS, bool MEE>
__global__ void irht_decompress_tile_kernel(const uint8_t *__restrict__ src, float *__restrict__ x, RhtTileArgs a,
                                       MeeArg<NBITS, MEE> mp)
{
    typedef Rec<NBITS> RC;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = threadIdx.x, nthreads = tile_threads(a.kt);
    const int tile = 1 << a.kt;
    const int64_t origin = (int64_t)blockIdx.x << a.kt;
    const int lane = tid & 63, wave = tid >> 6, nwaves = nthreads >> 6;
    // the record windows and the MEE table use the tile's LDS before the tile itself does
    uint8_t *windows = reinterpret_cast<uint8_t *>(lds);
    uint8_t *win_in = windows + wave * RC::WIN;
    float *table = reinterpret_cast<float *>(windows + nwaves * RC::WIN);
    if (MEE) {
        for (int k = tid; k < (1 << NBITS); k += nthreads) table[k] = f16_bits_to_f32(mp.levels()[k]);
        __syncthreads();
    }

    // decode the wave's run of records into registers, one lane per chunk; chunks beyond n become zeros
    const int64_t nsc_total = a.n >> 8, sc_origin = origin >> 8;
    const int tile_sc = max(1, tile >> 8);
    const int64_t sc0 = sc_origin + wave * kRowsPerWave;
    const int rows_here = (wave * kRowsPerWave < tile_sc && sc0 < nsc_total)
                              ? (int)min((int64_t)min(kRowsPerWave, tile_sc - wave * kRowsPerWave), nsc_total - sc0)
                              : 0;
    const int row = lane >> 4, j = lane & 15;
    float t[16];
#pragma unroll
    for (int i = 0; i < 16; i++) t[i] = 0.0f;
    if (rows_here > 0) {
        const int total = rows_here * RC::REC;
        const uint8_t *g = src + sc0 * RC::REC;
        const WinRegs wr = window_fetch(g, total, lane);
        const int mis = window_commit(win_in, wr, g, total, lane);
        wave_lds_sync();
        if (row < rows_here) {
            const uint8_t *rec = win_in + mis + row * RC::REC;
            uint32_t cw[RC::WORDS], cq;
            chunk_read<NBITS>(rec + j * RC::CB, cw, cq);
            const uint32_t ub = (uint32_t)rec[16 * RC::CB] | ((uint32_t)rec[16 * RC::CB + 1] << 8);
            chunk_decode<NBITS, MEE, false>(cw, cq, ub, table, t);
        }
    }
    __syncthreads(); // windows and table are done with: the tile takes the LDS
    {
        const int c = wave * 64 + lane;
        if (c * 16 < tile) {
            chunk_stages(t, a.kb);
            float *mine = lds + chunk_word(c);
#pragma unroll
            for (int i = 0; i < 16; i++) mine[i] = t[i];
        }
    }
    fwht_lds_stages_after4(lds, a.kt, a.kb, tid, nthreads);

    // store (coalesced): scale, then sign flip
    if (a.vec) {
        for (int i = tid * 4; i < tile; i += nthreads * 4) {
            const int64_t g = origin + i;
            if (g >= a.n) continue;
            const int q = pad_idx(i);
            float4 v = make_float4(lds[q], lds[q + 1], lds[q + 2], lds[q + 3]);
            v.x *= a.scale; v.y *= a.scale; v.z *= a.scale; v.w *= a.scale;
            flip4(v, a, g);
            stream_store(reinterpret_cast<float4 *>(x + g), v);
        }
    } else {
        for (int i = tid; i < tile; i += nthreads) {
            const int64_t g = origin + i;
            if (g >= a.n) continue;
            x[g] = flip1(lds[pad_idx(i)] * a.scale, a, g);
        }
    }
}

// ---- quantisers folded into the ends of the plain transform (TransformEnds) ------------------------------------

// the sign flip of a chunk that is already in registers (g a multiple of 16; 16-byte accesses to a float sign vector)
__device__ __forceinline__ bool has_diagonal(const RhtTileArgs &a) { return a.sign != nullptr; }
__device__ __forceinline__ bool has_diagonal(const RhtPassArgs &a) { return a.sign || a.gen.bits != 0; }

// sixteen signs from the low half of a word, the first element's in bit 0
__device__ __forceinline__ void flip16_bits(float (&v)[16], uint32_t w)
{
    // from the last element down, its bit at the top: doubling shifts and issues in half the time of a shift
    w <<= 16;
#pragma unroll
    for (int k = 15; k >= 0; k--) {
        v[k] = __uint_as_float(__float_as_uint(v[k]) ^ (w & 0x80000000u));
        w += w;
    }
}

template <class A> __device__ __forceinline__ void flip16(float (&v)[16], const A &a, int64_t g)
{
    if (!has_diagonal(a)) return;
    if (a.sign && a.sign_bits) {
        flip16_bits(v, static_cast<const uint32_t *>(a.sign)[g >> 5] >> (g & 31));
        return;
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
        float4 q = make_float4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
        flip4(q, a, g + 4 * k);
        v[4 * k] = q.x; v[4 * k + 1] = q.y; v[4 * k + 2] = q.z; v[4 * k + 3] = q.w;
    }
}

// lowest level and spacing of THC's grid
__device__ __forceinline__ void grid_of(const ThcGrid &d, const float *lo_p, const float *spacing_p, float &lo, float &spacing)
{
    if (d.kind == ThcGrid::NORM) {
        const float a = d.t * *d.norm, top = a * d.inv_sqrt;
        const float b = (top + top) * d.inv_levels;
        lo = -top;
        spacing = b + 1e-23f;
    } else if (d.kind == ThcGrid::HOST) {
        lo = d.lo;
        spacing = d.spacing;
    } else {
        lo = *lo_p;
        spacing = *spacing_p;
    }
}

// sixteen elements of a source of another type or length than the transform
__device__ __forceinline__ void load_source(float (&v)[16], const InEnds &e, int64_t g)
{
    const bool whole = g + 16 <= e.in_count && (reinterpret_cast<uintptr_t>(e.in_src) & 15) == 0;
    if (e.in_dtype == DQ_F32) {
        const float *p = static_cast<const float *>(e.in_src) + g;
        if (whole) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float4 q = reinterpret_cast<const float4 *>(p)[k];
                v[4 * k] = q.x; v[4 * k + 1] = q.y; v[4 * k + 2] = q.z; v[4 * k + 3] = q.w;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 16; i++) v[i] = g + i < e.in_count ? p[i] : 0.0f;
        }
        return;
    }
    const uint16_t *p = static_cast<const uint16_t *>(e.in_src) + g;
    uint32_t w[8];
    if (whole) {
        const uint4 a = reinterpret_cast<const uint4 *>(p)[0], b = reinterpret_cast<const uint4 *>(p)[1];
        w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w; w[4] = b.x; w[5] = b.y; w[6] = b.z; w[7] = b.w;
    } else {
#pragma unroll
        for (int k = 0; k < 8; k++) {
            w[k] = g + 2 * k < e.in_count ? p[2 * k] : 0u;
            if (g + 2 * k + 1 < e.in_count) w[k] |= (uint32_t)p[2 * k + 1] << 16;
        }
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
        v[2 * k] = e.in_dtype == DQ_BF16 ? bf16_bits_to_f32(w[k] & 0xffffu) : f16_bits_to_f32(w[k] & 0xffffu);
        v[2 * k + 1] = e.in_dtype == DQ_BF16 ? bf16_bits_to_f32(w[k] >> 16) : f16_bits_to_f32(w[k] >> 16);
    }
}

// four elements of a destination of another type or length (out_dst aligned to four elements, or element by element)
__device__ __forceinline__ void store_destination(const OutEnds &e, float4 v, int64_t g)
{
    if (g >= e.out_count) return;
    const float f[4] = {v.x, v.y, v.z, v.w};
    if (e.out_dtype == DQ_F32) {
        float *p = static_cast<float *>(e.out_dst) + g;
        if (g + 4 <= e.out_count && (reinterpret_cast<uintptr_t>(e.out_dst) & 15) == 0) {
            *reinterpret_cast<float4 *>(p) = v;
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (g + i < e.out_count) p[i] = f[i];
        }
        return;
    }
    uint16_t *p = static_cast<uint16_t *>(e.out_dst) + g;
    uint32_t h[4];
#pragma unroll
    for (int i = 0; i < 4; i++) h[i] = e.out_dtype == DQ_BF16 ? f32_to_bf16_bits(f[i]) : f32_to_f16_bits(f[i]);
    if (g + 4 <= e.out_count && (reinterpret_cast<uintptr_t>(e.out_dst) & 7) == 0) {
        *reinterpret_cast<uint2 *>(p) = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (g + i < e.out_count) p[i] = (uint16_t)h[i];
    }
}

// the centroids of sixteen consecutive bins, from the thread's half word of every plane (two 8 x 8 bit transposes)
__device__ __forceinline__ void load_planes(float (&v)[16], const InEnds &e, const float *cen, int64_t g, int64_t words)
{
    const uint16_t *half = reinterpret_cast<const uint16_t *>(e.in_planes) + (g >> 4);
    // (eight loads whatever the width, the last plane's again: in a loop over the planes they wait for one another)
    uint32_t h[8];
#pragma unroll
    for (int p = 0; p < 8; p++) h[p] = half[(int64_t)min(p, e.in_nbits - 1) * words * 2];
    uint64_t lo8 = 0, hi8 = 0;
#pragma unroll
    for (int p = 0; p < 8; p++) {
        const uint32_t w = p < e.in_nbits ? h[p] : 0u;
        lo8 |= (uint64_t)(w & 0xffu) << (8 * p);
        hi8 |= (uint64_t)(w >> 8) << (8 * p);
    }
    lo8 = transpose8x8(lo8);
    hi8 = transpose8x8(hi8);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        v[k] = cen[(lo8 >> (8 * k)) & 0xffu];
        v[8 + k] = cen[(hi8 >> (8 * k)) & 0xffu];
    }
}

// The chunk at g (a multiple of 16; n is a multiple of 32, so the chunk is inside the vector or outside) as the first
// pass sees it: the floats of x, or THC's levels times step plus lo (thc_hooks.py:176-178: two roundings), or the
// centroids of EDEN's bins, read from the bit planes (srrcomp.py:343-354); then the sign flip of a forward transform.
// cen: the centroid table in LDS.
template <bool ENDS, class E>
__device__ __forceinline__ void fetch_chunk(float (&v)[16], const float *__restrict__ x, const PassArgs<ENDS> &in,
                                            const E &e, const float *cen, int64_t g)
{
    if (!ENDS || (!e.in_levels && !e.in_planes && !e.in_src)) {
        load_chunk(v, x, in, g);
        if constexpr (ENDS) {
            if (in.gen.bits != 0) flip16(v, in, g);
        }
        return;
    }
    if (g >= in.n) {
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = 0.0f;
        return;
    }
    if (e.in_src) {
        load_source(v, e, g);
    } else if (e.in_levels) {
        const uint4 *p = reinterpret_cast<const uint4 *>(e.in_levels + g);
        const uint4 l0 = p[0], l1 = p[1];
        const uint32_t w[8] = {l0.x, l0.y, l0.z, l0.w, l1.x, l1.y, l1.z, l1.w};
        float step, lo;
        grid_of(e.grid, e.in_lo, e.in_step, lo, step);
        if (e.grid.kind == ThcGrid::NORM) step = step * e.grid.inv_clients;
        if (e.grid.kind == ThcGrid::HOST) step = e.grid.step;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const float p0 = bf16_bits_to_f32(w[k] & 0xffffu) * step, p1 = bf16_bits_to_f32(w[k] >> 16) * step;
            v[2 * k] = p0 + lo;
            v[2 * k + 1] = p1 + lo;
        }
    } else {
        load_planes(v, e, cen, g, in.n >> 5);
    }
    flip16(v, in, g);
}

// four consecutive elements of the last pass on their way out: scale, sign flip of an inverse transform, EDEN's scale,
// then the float store or THC's quantiser (thc_hooks.py:161-166) and a bf16 store
template <bool ENDS>
__device__ __forceinline__ void store4(float *__restrict__ x, float4 v, const PassArgs<ENDS> &a, const TransformEnds &e, int sign_mode,
                                       int apply_scale, int64_t g)
{
    if (apply_scale) { v.x *= a.scale; v.y *= a.scale; v.z *= a.scale; v.w *= a.scale; }
    if (sign_mode == 2) flip4(v, a, g);
    if (ENDS && e.post_scale) {
        const float ps = *e.post_scale;
        v.x *= ps; v.y *= ps; v.z *= ps; v.w *= ps;
    }
    if (ENDS && e.out_levels) {
        const float4 u = *reinterpret_cast<const float4 *>(e.uniform + g);
        float lo, delta;
        grid_of(e.grid, e.out_lo, e.out_delta, lo, delta);
        uint2 o;
        o.x = f32x2_to_bf16x2(thc_level(v.x, u.x, lo, delta, e.out_top), thc_level(v.y, u.y, lo, delta, e.out_top));
        o.y = f32x2_to_bf16x2(thc_level(v.z, u.z, lo, delta, e.out_top), thc_level(v.w, u.w, lo, delta, e.out_top));
        *reinterpret_cast<uint2 *>(e.out_levels + g) = o;
    } else if (ENDS && e.out_dst) {
        store_destination(e, v, g);
    } else {
        *reinterpret_cast<float4 *>(x + g) = v;
    }
}

// lane bit 4 (16) or 5 (32) changes places with register bit RB: one instruction per two registers
template <int LANES, int RB> __device__ __forceinline__ void swap_lane_bit(float (&v)[16])
{
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < 16; i++) {
        if ((i >> RB) & 1) continue;
        const uint32_t a = __float_as_uint(v[i]), b = __float_as_uint(v[i | (1 << RB)]);
        const u32x2 r = LANES == 16 ? __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(a, b, false, false))
                                    : __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(a, b, false, false));
        v[i] = __uint_as_float(r[0]);
        v[i | (1 << RB)] = __uint_as_float(r[1]);
    }
}

// the stage of register bit RB
template <int RB> __device__ __forceinline__ void stage_of(float (&v)[16])
{
#pragma unroll
    for (int i = 0; i < 16; i++) {
        if ((i >> RB) & 1) continue;
        const float p = v[i], q = v[i | (1 << RB)];
        v[i] = p + q;
        v[i | (1 << RB)] = p - q;
    }
}

// A tile of 2^KT elements with a chunk per thread, in two trips through the LDS: which chunk a thread takes; the stages of strides 1 ..
// 8, for 2^13 and 2^14 elements one or two more by lane bit 5 (and 4) changing places with a register bit, and the chunk into the LDS;
// (a barrier;) the next stages; (a barrier.)  What is left then are the four highest stages, on elements tid + j 2^(KT - 4).
template <int KT> __device__ __forceinline__ int chunk_of(int tid)
{
    const int lane = tid & 63;
    if (KT == 13) return (tid & ~63) | ((lane & 31) << 1) | (lane >> 5);
    if (KT == 14) return (tid & ~63) | ((lane & 15) << 2) | (((lane >> 4) & 1) << 1) | (lane >> 5);
    return tid;
}

template <int KT> __device__ __forceinline__ void chunk_into_tile(float (&v)[16], float *lds, int tid)
{
    const int lane = tid & 63, c = chunk_of<KT>(tid);
    butterflies<4>(v);
    if constexpr (KT == 13) {
        swap_lane_bit<32, 0>(v);
        stage_of<0>(v); // e4
        float *slot = lds + pad_idx(((c >> 1) << 5) | (lane >> 5));
#pragma unroll
        for (int i = 0; i < 16; i++) slot[((i & 1) << 4) | (i & 14)] = v[i];
    } else if constexpr (KT == 14) {
        swap_lane_bit<32, 1>(v);
        stage_of<1>(v); // e4
        swap_lane_bit<16, 0>(v);
        stage_of<0>(v); // e5
        float *slot = lds + pad_idx(((c >> 2) << 6) | ((lane >> 5) << 1) | ((lane >> 4) & 1));
#pragma unroll
        for (int i = 0; i < 16; i++) slot[pad_idx(((i & 1) << 5) | (((i >> 1) & 1) << 4) | (i & 12))] = v[i];
    } else {
        float *slot = lds + chunk_word(c);
#pragma unroll
        for (int i = 0; i < 16; i++) slot[i] = v[i];
    }
}

template <int KT> __device__ __forceinline__ void middle_stages(float *lds, int tid, int nthreads)
{
    static_assert(KT >= 10 && KT <= 14, "two trips");
    if (KT == 13)
        lds_pass<5, 4>(lds, KT, tid, nthreads);
    else if (KT == 14)
        lds_pass<6, 4>(lds, KT, tid, nthreads);
    else
        lds_pass<4, KT < 13 ? KT - 8 : 4>(lds, KT, tid, nthreads);
}

// First passes with a source of another type or length store so many elements with the non-temporal hint: what waits in the L2 until the
// kernel ends, more than half of its 32 MB, is then on its way while others still load.  2^23 elements from bf16 levels 13.8 -> 9.5 us, from
// a 25 MB gradient 12.8 -> 11.7.  The pass that reads them takes 0.5 to 1 longer, which costs fewer elements more than they gain, and more
// than 32 MB fill the L2 long before the end.  Where the pass reads what it overwrites it gains nothing.  The whole call, us, without ->
// with:
//   THC compress    4,194,304 18.0 18.2; of 2^23: 4,300,000 25.7 23.8, 6,553,600 25.9 24.2, all 26.3 25.3; of 2^24: 4,300,000 30.2 30.0,
//                   6,553,600 31.7 30.1, 8,300,000 33.4 32.8, 10,000,000 40.0 41.4, all 49.7 53.5
//   THC decompress  2^22 19.5 19.6, 2^23 25.3 24.4, 2^24 46.5 49.4
//   EDEN            compress 2^22 32.8 33.2, 2^23 46.7 47.0, 2^24 81.8 86.0; decompress 20.4 20.9, 36.3 34.8, 54.1 57.4
//   in place        forward, blocks of 2^18: 4.5 x 2^20 22.5 22.2, 6 x 2^20 21.6 21.9, 7 x 2^20 21.0 21.7, 2^23 22.7 23.8, 2^24 42.3 42.9
constexpr int64_t kEarlyFrom = ((int64_t)1 << 22) + 1, kEarlyTo = (int64_t)1 << 23;

// lds_pass whose results go to memory: consecutive lanes hold consecutive elements (P >= 6)
template <int P, int M> __device__ __forceinline__ void lds_pass_out(const float *lds, int kt, int tid, int nthreads, float *__restrict__ out, bool early)
{
    for (int u = tid; u < 1 << (kt - M); u += nthreads) {
        const int base = tuple_base<P, M>(u, kt - P - M);
        const float *q = lds + pad_idx(base);
        float v[1 << M];
#pragma unroll
        for (int j = 0; j < (1 << M); j++) v[j] = q[tuple_step<P>(j)];
        butterflies<M>(v);
        if (early) {
            asm volatile(""); // (the compiler would make one store of the two, without the hint)
#pragma unroll
            for (int j = 0; j < (1 << M); j++) __builtin_nontemporal_store(v[j], out + base + (j << P));
            asm volatile("");
        } else {
#pragma unroll
            for (int j = 0; j < (1 << M); j++) out[base + (j << P)] = v[j];
        }
    }
}

// The transform alone (dq_rht_blocked, the first pass of a long dq_hadamard) with the structure of the two kernels
// above: a lane loads its chunk of 16 consecutive floats, does the stages of strides 1..8 on its registers, the rest
// runs as LDS passes of up to five stages, and the tile leaves as coalesced 16-byte stores with the scale and (inverse
// direction) the sign flip.  Against the all-in-LDS kernel of dq_hadamard.hip: two or three LDS passes instead of four,
// and a thread's loads issued together.  In place: a workgroup reads and writes only its own tile.
// sign_mode: 0 no flip, 1 flip on load, 2 flip on store
// ENDS: a quantiser may sit at either end (TransformEnds; 16-byte accesses only: a.vec is set)
template <bool ENDS>
__device__ __forceinline__ void tile_pass(float *__restrict__ x, const PassArgs<ENDS> &a, int sign_mode, int apply_scale,
                                          const TransformEnds &e, unsigned block, float *lds)
{
    const int tid = threadIdx.x, nthreads = tile_threads(a.kt);
    const int tile = 1 << a.kt;
    const int64_t origin = (int64_t)block << a.kt;
    PassArgs<ENDS> in = a;
    if (sign_mode != 1) {
        in.sign = nullptr;
        if constexpr (ENDS) in.gen.bits = 0;
    }
    const float *cen = lds + padded_tile_floats(a.kt); // EDEN's centroids sit behind the tile
    if (ENDS && e.in_planes) {
        for (int k = tid; k < (1 << e.in_nbits); k += nthreads) lds[padded_tile_floats(a.kt) + k] = e.in_centroids[k];
        __syncthreads();
    }
    const int nchunks = tile >> 4;
    if (nchunks == 2 * nthreads) {
        // 2^15 tiles: both chunks of a thread are loaded before either is used
        float v[16], w[16];
        fetch_chunk<ENDS>(v, x, in, e, cen, origin + tid * 16);
        fetch_chunk<ENDS>(w, x, in, e, cen, origin + (tid + nthreads) * 16);
        chunk_stages(v, a.kb);
        chunk_stages(w, a.kb);
        float *mine = lds + chunk_word(tid), *other = lds + chunk_word(tid + nthreads);
#pragma unroll
        for (int i = 0; i < 16; i++) mine[i] = v[i];
#pragma unroll
        for (int i = 0; i < 16; i++) other[i] = w[i];
    } else {
        for (int c = tid; c < nchunks; c += nthreads) {
            float v[16];
            fetch_chunk<ENDS>(v, x, in, e, cen, origin + c * 16);
            chunk_stages(v, a.kb);
            float *mine = lds + chunk_word(c);
#pragma unroll
            for (int i = 0; i < 16; i++) mine[i] = v[i];
        }
    }
    fwht_lds_stages_after4(lds, a.kt, a.kb, tid, nthreads);
    if (a.vec) {
        for (int i = tid * 4; i < tile; i += nthreads * 4) {
            const int64_t g = origin + i;
            if (g >= a.n) continue;
            const int q = pad_idx(i);
            store4<ENDS>(x, make_float4(lds[q], lds[q + 1], lds[q + 2], lds[q + 3]), a, e, sign_mode, apply_scale, g);
        }
    } else {
        for (int i = tid; i < tile; i += nthreads) {
            const int64_t g = origin + i;
            if (g >= a.n) continue;
            float v = lds[pad_idx(i)];
            if (apply_scale) v *= a.scale;
            x[g] = sign_mode == 2 ? flip1(v, a, g) : v;
        }
    }
}

// The first pass of a long transform: the tile is one block of 2^10 .. 2^14 elements, a chunk per thread, with nothing to do on
// the way out.  The last stages store from registers, as whole 256-byte runs: one trip through the LDS and one barrier less
// than tile_pass.  Bound like the strided passes; 2^23 elements from bf16 levels 13.4 -> 11.8 us, from a 25 MB gradient 17.3 -> 15.0.
template <bool ENDS, class E>
__device__ __forceinline__ void first_pass(float *__restrict__ x, const PassArgs<ENDS> &a, int sign_mode, const E &e, unsigned block,
                                           float *lds, int threads, bool early)
{
    const int tid = threadIdx.x;
    const int64_t origin = (int64_t)block << a.kt;
    PassArgs<ENDS> in = a;
    if (sign_mode != 1) {
        in.sign = nullptr;
        if constexpr (ENDS) in.gen.bits = 0;
    }
    const float *cen = lds + padded_tile_floats(a.kt); // EDEN's centroids sit behind the tile
    if (ENDS && e.in_planes) {
        for (int k = tid; k < (1 << e.in_nbits); k += threads) lds[padded_tile_floats(a.kt) + k] = e.in_centroids[k];
        __syncthreads();
    }
    const int nthreads = 1 << (a.kt - 4);
    const auto fetch_into = [&](auto kt) { // (a launch of several passes has the threads of the largest; they come in whole waves)
        if (tid >= nthreads) return;
        float v[16];
        fetch_chunk<ENDS>(v, x, in, e, cen, origin + chunk_of<decltype(kt)::value>(tid) * 16);
        chunk_into_tile<decltype(kt)::value>(v, lds, tid);
    };
    if (a.kt == 13)
        fetch_into(std::integral_constant<int, 13>());
    else if (a.kt == 14)
        fetch_into(std::integral_constant<int, 14>());
    else
        fetch_into(std::integral_constant<int, 12>()); // (and below)
    __syncthreads();
    const int step = threads;
    switch (a.kt) {
    case 10: middle_stages<10>(lds, tid, step); break;
    case 11: middle_stages<11>(lds, tid, step); break;
    case 12: middle_stages<12>(lds, tid, step); break;
    case 13: middle_stages<13>(lds, tid, step); break;
    default: middle_stages<14>(lds, tid, step); break;
    }
    __syncthreads();
    float *out = x + origin;
    switch (a.kt) {
    case 10: lds_pass_out<6, 4>(lds, 10, tid, step, out, early); break;
    case 11: lds_pass_out<7, 4>(lds, 11, tid, step, out, early); break;
    case 12: lds_pass_out<8, 4>(lds, 12, tid, step, out, early); break;
    case 13: lds_pass_out<9, 4>(lds, 13, tid, step, out, early); break;
    default: lds_pass_out<10, 4>(lds, 14, tid, step, out, early); break;
    }
}

template <bool ENDS>
__global__ void rht_tile_kernel(float *__restrict__ x, PassArgs<ENDS> a, int sign_mode, int apply_scale, TransformEnds e)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    tile_pass<ENDS>(x, a, sign_mode, apply_scale, e, blockIdx.x, lds);
}

// Uniform values of a stream as torch's generator hands them to the threads of a kernel: thread k of 2^bits takes the blocks
// counter, counter + 1, ... of subsequence k, and the four words of a block go to elements 2^bits apart.  u[i] is that of element
// first + i 2^shift.  The bits of i from P on are the number of the word in its block (where they lie outside i, its bits are those
// of first): one block serves up to four of the elements.  Drawn here while the elements are on their way, they need neither the
// launch that writes them nor its 33 MB there and back: THC's compress of a 25 MB bucket 46 -> 27 us.
template <int B, int P>
__device__ __forceinline__ void draw_rows(float (&u)[1 << B], const UniformDraw &d, int64_t first, int shift)
{
    constexpr int kLow = P >= 0 && P < B ? 1 << P : 0, kHigh = P + 1 >= 0 && P + 1 < B ? 1 << (P + 1) : 0;
#pragma unroll
    for (int i = 0; i < (1 << B); i++) {
        if (i & (kLow | kHigh)) continue;
        const int64_t g = first + ((int64_t)i << shift);
        const uint32_t at = (uint32_t)(g >> d.bits);
        const uint64_t counter = d.counter + (at >> 2);
        uint32_t w[4] = {(uint32_t)counter, (uint32_t)(counter >> 32), (uint32_t)g & ((1u << d.bits) - 1u), 0u};
        philox4x32_10(w, (uint32_t)d.seed, (uint32_t)(d.seed >> 32));
        if (!kLow) {
            w[0] = (at & 1) ? w[1] : w[0];
            w[2] = (at & 1) ? w[3] : w[2];
        }
        if (!kHigh) {
            w[0] = (at & 2) ? w[2] : w[0];
            w[1] = (at & 2) ? w[3] : w[1];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if ((!kLow && (k & 1)) || (!kHigh && (k & 2))) continue;
            // (0, 1] with 1 replaced by 0
            const float f = __builtin_fmaf((float)w[k], 0x1p-32f, 0x1p-32f);
            u[i | (k & 1 ? kLow : 0) | (k & 2 ? kHigh : 0)] = f == 1.0f ? 0.0f : f;
        }
    }
}

template <int B> __device__ __forceinline__ void draw_rows(float (&u)[1 << B], const UniformDraw &d, int64_t first, int shift)
{
    switch (d.bits - shift) {
    case -1: draw_rows<B, -1>(u, d, first, shift); break;
    case 0: draw_rows<B, 0>(u, d, first, shift); break;
    case 1: draw_rows<B, 1>(u, d, first, shift); break;
    case 2: draw_rows<B, 2>(u, d, first, shift); break;
    case 3: draw_rows<B, 3>(u, d, first, shift); break;
    default: draw_rows<B, B>(u, d, first, shift); break;
    }
}

// A later pass of a transform longer than one tile: index bits [sbits, sbits + A + B) of the vector.  A tile is 2^(A + B)
// rows of 32 consecutive floats (128 bytes), row stride 2^sbits elements.  A thread owns column tid % 32 of 2^A consecutive
// rows: it loads them (every load instruction of a wave covers two whole 128-byte row segments), does the A lowest row
// stages on its registers, hands the rows over through the LDS once, does the other B stages on rows 2^A apart and stores
// them from its registers, as whole row segments again.  The LDS needs no padding: 32 lanes are the 32 columns of a row.
// A = 4 (5 for 512 and 1024 rows), so a thread has 16 (32) values and a tile tile / 16 (512 and 1024) threads.
// Bound by the memory's latency: all workgroups of a pass are on the chip at once, load together and store together.
// One trip through the LDS instead of three or four: 2^23 elements, 1024 rows back to a 25 MB vector 17.2 -> 13.3 us, to THC's
// levels 19.0 -> 17.8 (67 MB read); both directions of THC on 25 MB 82.6 -> 70.2, on 16,000,000 elements 146.7 -> 118.7, EDEN on
// 500,000 36.5 -> 31.7, on 12,000,000 157 -> 136 (with the first pass below).
// sign_mode: 0, or 2 = flip on store (the last pass of an inverse).
// e.sums (the whole vector, its last pass): the sum of the squares of what the workgroup stores, in the order of dq_sums.cuh: EDEN's
// norm without a pass over the vector for it, 3.1 us of 34 at 2^20 elements, 12 of 137 at 2^24.  The workgroup has 2^(A + B - 4)
// pieces of 32 columns.  With A = 4 they are its groups of 32 threads, whose rows are the loop's last 4 - B digits below the
// B of the registers; with A = 5 a group has two, and the piece's number has one more digit in front of the group's.
// DRAW: the pass stores THC's levels and draws their uniform values, while the elements are on their way; it knows e.zeros_from.  A variant of its own: beside
// loads of uniform values, which may be pending in the registers that the draws go to as far as the compiler can tell, every draw
// waited for elements it does not need.  2^23 elements to THC's levels, with thc_levels in groups: both ways 54.1 -> 52.8 us, 2^24 103.5 ->
// 100.5, padded 25 MB (with e.zeros_from) 50.7 -> 48.
template <bool ENDS, int A, int B, bool DRAW = false, class E>
__device__ __forceinline__ void strided_rows(float *__restrict__ x, const PassArgs<ENDS> &a, int sbits, int sign_mode, int apply_scale,
                                             const E &e, unsigned block, float *lds)
{
    constexpr int R1 = 1 << A, R2 = 1 << B;
    const int tid = threadIdx.x;
    // (shift and mask: written as a quotient and remainder by the power of two, the compiler expands a 64-bit
    // division in front of the kernel's first loads)
    const int64_t hi = (int64_t)(block >> (sbits - 5)), mid = (int64_t)(block & ((1u << (sbits - 5)) - 1u));
    const int64_t origin = (hi << (sbits + A + B)) + (mid << 5);
    const int col = tid & 31, group = tid >> 5;
    const bool mine = group < R2; // (a launch of several passes has the threads of the largest)
    float v[R1];
    // of the thread's rows: those behind them are zeros that nobody has written (the last written row's address is asked for instead:
    // behind a comparison each, the loads would wait for one another)
    int have = R1;
    bool whole = true;
    if (DRAW && e.zeros_from >= 0) {
        have = min(max((int)(e.zeros_from >> sbits) - (group << A), 0), R1);
        whole = __builtin_amdgcn_ballot_w64(have < R1) == 0;
    }
    if (mine) {
        const float *from = x + origin + ((int64_t)(group << A) << sbits) + col;
        if (whole) {
#pragma unroll
            for (int j = 0; j < R1; j++) v[j] = from[(int64_t)j << sbits];
        } else if (__builtin_amdgcn_ballot_w64(have > 0) != 0) {
#pragma unroll
            for (int j = 0; j < R1; j++) v[j] = from[(int64_t)min(j, max(have - 1, 0)) << sbits];
        }
    }
    // THC's uniform values are drawn while the elements are on their way; or they are on their way while the stages run, where one
    // workgroup has a CU to itself (1024 rows; with 256 that gains nothing)
    static_assert(!DRAW || (ENDS && A == B), "a thread has one row of the registers' 2^B to draw for");
    constexpr bool kAhead = ENDS && !DRAW && A == 5 && B == 5;
    const bool levels_out = DRAW || (ENDS && e.out_levels);
    float u[R2];
    bool have_u = DRAW;
    if constexpr (DRAW || kAhead) {
        if (levels_out && mine) {
            const int64_t at = origin + ((int64_t)group << sbits) + col;
            if constexpr (DRAW) {
                draw_rows<B>(u, e.draw, at, A + sbits);
            } else {
#pragma unroll
                for (int i = 0; i < R2; i++) u[i] = e.uniform[at + ((int64_t)i << (A + sbits))];
                have_u = true;
            }
        }
    }
    if (!whole) {
#pragma unroll
        for (int j = 0; j < R1; j++) v[j] = j < have ? v[j] : 0.0f;
    }
    if (mine) butterflies<A>(v);
    float post = 1.0f, lo = 0.0f, delta = 1.0f;
    if (ENDS && !DRAW && e.post_scale) post = *e.post_scale;
    if (levels_out) grid_of(e.grid, e.out_lo, e.out_delta, lo, delta);
    if constexpr (B > 0) {
        if (mine) {
#pragma unroll
            for (int j = 0; j < R1; j++) lds[((group << A) + j) * 32 + col] = v[j];
        }
        __syncthreads();
    }
    constexpr int kSums = A == 5 ? 2 : 1 << (4 - B);
    double sums[kSums];
    if constexpr (ENDS && !DRAW) {
#pragma unroll
        for (int q = 0; q < kSums; q++) sums[q] = 0.0;
    }
    const bool flips = !DRAW && sign_mode == 2;
    bool drawn = false;
    if constexpr (ENDS) drawn = flips && a.gen.bits != 0;
    // rows i 2^A + row, i < 2^B, of one column
    const auto finish = [&](float (&w)[R2], int row) {
        const int64_t first = origin + ((int64_t)row << sbits) + col;
        if (apply_scale) {
#pragma unroll
            for (int i = 0; i < R2; i++) w[i] *= a.scale;
        }
        if (drawn) {
            if constexpr (ENDS) {
                const uint32_t column_mask = (1u << a.gen.bits) - 1u;
                if constexpr (B >= 3) {
                    if (a.gen.bits + 3 == sbits + A + B) {
                        // the whole vector: the eight elements of a column of the diagonal are 2^(B - 3) of these rows apart
#pragma unroll
                        for (int i = 0; i < R2 / 8; i++) {
                            const uint32_t r = rand_diag_column(a.gen, (uint32_t)(first + ((int64_t)i << (A + sbits))) & column_mask);
#pragma unroll
                            for (int k = 0; k < 8; k++) {
                                const int at = k * (R2 / 8) + i;
                                w[at] = __uint_as_float(__float_as_uint(w[at]) ^ nibble_negative(r, k));
                            }
                        }
                        drawn = false;
                    }
                }
                if (drawn) {
#pragma unroll
                    for (int i = 0; i < R2; i++) {
                        const int64_t g = first + ((int64_t)i << (A + sbits));
                        w[i] = __uint_as_float(__float_as_uint(w[i]) ^ rand_diag_negative(a.gen, (uint32_t)(g >> a.gen.bits), (uint32_t)g & column_mask));
                    }
                }
                drawn = true;
            }
        } else if (flips && a.sign && a.sign_bits) {
            // a row's 32 signs are one word: lane i (and R2 + i) fetches that of row i of the lower (upper) half of the wave, and
            // the two make the lane mask of a select
            const int lane = tid & 63;
            const int low_row = B > 0 ? (row & ~1) + ((lane >> B) & 1) : row;
            const int64_t at = origin + ((int64_t)(((lane & (R2 - 1)) << A) + low_row) << sbits);
            const uint32_t word = static_cast<const uint32_t *>(a.sign)[at >> 5];
#pragma unroll
            for (int i = 0; i < R2; i++) {
                const uint32_t low = (uint32_t)__builtin_amdgcn_readlane((int)word, i), high = (uint32_t)__builtin_amdgcn_readlane((int)word, R2 + i);
                const uint64_t mask = (uint64_t)low | ((uint64_t)high << 32);
                // (the two wait states behind a readlane are the compiler's only for its own instructions)
                asm("s_nop 1\n\tv_cndmask_b32_e64 %0, %0, -%0, %1" : "+v"(w[i]) : "s"(mask));
            }
        } else if (flips && a.sign) {
#pragma unroll
            for (int i = 0; i < R2; i++) w[i] *= static_cast<const float *>(a.sign)[first + ((int64_t)i << (A + sbits))];
        }
        // on their way out: EDEN's scale, then the float store, THC's quantiser (thc_hooks.py:161-166) or a destination of
        // another type
        if (ENDS && !DRAW && e.post_scale) {
#pragma unroll
            for (int i = 0; i < R2; i++) w[i] *= post;
        }
        if (levels_out) {
            if (!have_u) {
#pragma unroll
                for (int i = 0; i < R2; i++) u[i] = e.uniform[first + ((int64_t)i << (A + sbits))];
            }
            uint32_t levels[R2];
            thc_levels(w, u, lo, delta, e.out_top, levels);
#pragma unroll
            for (int i = 0; i < R2; i++) e.out_levels[first + ((int64_t)i << (A + sbits))] = (uint16_t)(levels[i] >> 16);
        } else if (ENDS && e.out_dst) {
            // rows that lie inside the destination for the whole wave need no test
            const int last_row = __builtin_amdgcn_readfirstlane(B > 0 ? row | 1 : row);
            const int64_t whole = ((e.out_count - 32 - origin - ((int64_t)last_row << sbits)) >> (A + sbits)) + 1;
            const int rows = (int)min(whole, (int64_t)R2);
            const auto store = [&](auto *out, auto convert) {
                if (rows == R2) {
#pragma unroll
                    for (int i = 0; i < R2; i++) out[first + ((int64_t)i << (A + sbits))] = convert(w[i]);
                    return;
                }
#pragma unroll
                for (int i = 0; i < R2; i++) {
                    const int64_t g = first + ((int64_t)i << (A + sbits));
                    if (i < rows)
                        out[g] = convert(w[i]);
                    else if (g < e.out_count)
                        out[g] = convert(w[i]);
                }
            };
            if (e.out_dtype == DQ_F32)
                store(static_cast<float *>(e.out_dst), [](float f) { return f; });
            else if (e.out_dtype == DQ_BF16)
                store(static_cast<uint16_t *>(e.out_dst), [](float f) { return (uint16_t)f32_to_bf16_bits(f); });
            else
                store(static_cast<uint16_t *>(e.out_dst), [](float f) { return (uint16_t)f32_to_f16_bits(f); });
        } else {
#pragma unroll
            for (int i = 0; i < R2; i++) x[first + ((int64_t)i << (A + sbits))] = w[i];
            if (ENDS && e.sums) {
                if constexpr (B == 5) {
                    sums[0] = halve_squares<2>(w);
                    sums[1] = halve_squares<2>(w, 1);
                } else {
                    const double sum = halve_squares(w);
#pragma unroll
                    for (int q = 0; q < kSums; q++) sums[q] = q == row >> B ? sum : sums[q];
                }
            }
        }
    };
    if constexpr (B > 0) {
#pragma unroll 1
        for (int row = mine ? group : R1; row < R1; row += R2) {
            float w[R2];
#pragma unroll
            for (int i = 0; i < R2; i++) w[i] = lds[((i << A) + row) * 32 + col];
            butterflies<B>(w);
            finish(w, row);
        }
    } else if (mine) {
#pragma unroll
        for (int j = 0; j < R1; j++) {
            float w[1] = {v[j]};
            finish(w, j);
        }
    }
    if constexpr (ENDS && !DRAW) {
        if (e.sums) {
            double sum;
            if constexpr (A == 5)
                sum = sum_columns_f64(sums[0]) + sum_columns_f64(sums[1]);
            else
                sum = sum_columns_f64(halve(sums));
            double *part = reinterpret_cast<double *>(lds + (32 << (A + B))); // (behind the tile: strided_lds_bytes)
            if (mine && col == 0) part[group] = sum;
            __syncthreads();
            if (tid < 64) {
                double all = tid < R2 ? part[tid] : 0.0;
                if (B == 5) all = add_across_f64<16>(all);
                all = halve_row_f64(all);
                if (tid == 0) e.sums[block] = all;
            }
        }
    }
}

// a tile, and a double for each of up to 32 groups
__host__ constexpr size_t strided_lds_bytes(int rbits) { return (sizeof(float) << (rbits + 5)) + 32 * sizeof(double); }
// threads of the tile of a strided pass
__host__ __device__ constexpr int strided_threads(int rbits) { return rbits >= 9 ? 1 << rbits : 1 << (rbits + 1); }

template <bool ENDS, class E>
__device__ __forceinline__ void strided_pass(float *__restrict__ x, const PassArgs<ENDS> &a, int rbits, int sbits, int sign_mode,
                                             int apply_scale, const E &e, unsigned block, float *lds)
{
    switch (rbits) {
    case 4: strided_rows<ENDS, 4, 0>(x, a, sbits, sign_mode, apply_scale, e, block, lds); break;
    case 5: strided_rows<ENDS, 4, 1>(x, a, sbits, sign_mode, apply_scale, e, block, lds); break;
    case 6: strided_rows<ENDS, 4, 2>(x, a, sbits, sign_mode, apply_scale, e, block, lds); break;
    case 7: strided_rows<ENDS, 4, 3>(x, a, sbits, sign_mode, apply_scale, e, block, lds); break;
    default: strided_rows<ENDS, 4, 4>(x, a, sbits, sign_mode, apply_scale, e, block, lds); break;
    }
}

// the arguments of a pass, and the ends that it looks at
struct FirstEnds : InEnds {
    ThcGrid grid;
};
struct LastEnds : OutEnds {
    ThcGrid grid;
};

// The same as kernel arguments.  Beyond 128 bytes of them a launch takes 0.7 us longer (MeeTable of dq_tile16.cuh), and as they stand the
// arguments, ends and grid are 176 and 224: what excludes one another shares a place, and small numbers take a byte.
enum { kNoEnd, kOther, kLevelsEnd, kPlanesEnd };

struct FirstPass {
    float *x;
    const void *sign, *in, *p; // the source, levels or planes; with levels the step or the norm, with planes the centroids
    const float *in_lo;
    int64_t n, in_count;
    float scale, grid[7]; // lo, spacing, step, t, inv_sqrt, inv_levels, inv_clients
    uint32_t gen_ss;
    uint8_t kt, kb, vec, sign_bits, sign_mode, gen_bits, end, in_dtype, in_nbits, grid_kind;
};
static_assert(sizeof(FirstPass) <= 128, "see above");

struct StridedPass {
    float *x;
    const void *sign;
    void *out;                  // the destination or levels
    const void *p;              // with levels the uniform values, else the scale of the last pass
    const void *q, *r;          // with levels its grid: lowest level or norm, spacing; else the sums
    int64_t n, count;           // with levels zeros_from, else out_count
    uint64_t draw_seed, draw_counter;
    float scale, out_top, grid[3]; // lo, spacing; or t, inv_sqrt, inv_levels
    uint32_t gen_ss;
    uint8_t rbits, sbits, sign_mode, apply_scale, end, out_dtype, gen_bits, vec, sign_bits, kt, grid_kind;
    int8_t draw_bits;
};
static_assert(sizeof(StridedPass) <= 128, "see above");

template <bool ENDS> __device__ __forceinline__ PassArgs<ENDS> pass_args(const FirstPass &p)
{
    PassArgs<ENDS> a;
    a.sign = p.sign; a.sign_bits = p.sign_bits; a.n = p.n; a.kt = p.kt; a.kb = p.kb; a.scale = p.scale; a.vec = p.vec;
    if constexpr (ENDS) {
        a.gen.bits = p.gen_bits;
        a.gen.ss = p.gen_ss;
    }
    return a;
}

template <bool ENDS> __device__ __forceinline__ PassArgs<ENDS> pass_args(const StridedPass &p)
{
    PassArgs<ENDS> a;
    a.sign = p.sign; a.sign_bits = p.sign_bits; a.n = p.n; a.kt = p.kt; a.kb = 0; a.scale = p.scale; a.vec = p.vec;
    if constexpr (ENDS) {
        a.gen.bits = p.gen_bits;
        a.gen.ss = p.gen_ss;
    }
    return a;
}

__device__ __forceinline__ FirstEnds ends_of(const FirstPass &p)
{
    FirstEnds e;
    const bool levels = p.end == kLevelsEnd, planes = p.end == kPlanesEnd;
    e.in_src = p.end == kOther ? p.in : nullptr;
    e.in_dtype = p.in_dtype;
    e.in_count = p.in_count;
    e.in_levels = levels ? static_cast<const uint16_t *>(p.in) : nullptr;
    e.in_step = e.grid.norm = static_cast<const float *>(p.p);
    e.in_lo = p.in_lo;
    e.in_planes = planes ? static_cast<const uint32_t *>(p.in) : nullptr;
    e.in_centroids = static_cast<const float *>(p.p);
    e.in_nbits = p.in_nbits;
    e.grid.kind = p.grid_kind;
    e.grid.lo = p.grid[0]; e.grid.spacing = p.grid[1]; e.grid.step = p.grid[2];
    e.grid.t = p.grid[3]; e.grid.inv_sqrt = p.grid[4]; e.grid.inv_levels = p.grid[5]; e.grid.inv_clients = p.grid[6];
    return e;
}

__device__ __forceinline__ LastEnds ends_of(const StridedPass &p)
{
    LastEnds e;
    const bool levels = p.end == kLevelsEnd;
    e.zeros_from = levels ? p.count : -1;
    e.out_dst = p.end == kOther ? p.out : nullptr;
    e.out_dtype = p.out_dtype;
    e.out_count = p.count;
    e.out_levels = levels ? static_cast<uint16_t *>(p.out) : nullptr;
    e.uniform = static_cast<const float *>(p.p);
    e.out_lo = e.grid.norm = static_cast<const float *>(p.q);
    e.out_delta = static_cast<const float *>(p.r);
    e.out_top = p.out_top;
    e.draw.bits = p.draw_bits; e.draw.seed = p.draw_seed; e.draw.counter = p.draw_counter;
    e.post_scale = levels ? nullptr : static_cast<const float *>(p.p);
    e.sums = levels ? nullptr : const_cast<double *>(static_cast<const double *>(p.q));
    e.grid.kind = p.grid_kind;
    e.grid.lo = e.grid.t = p.grid[0];
    e.grid.spacing = e.grid.inv_sqrt = p.grid[1];
    e.grid.inv_levels = p.grid[2];
    return e;
}

inline FirstPass first_of(float *x, const RhtPassArgs &a, int sign_mode, const TransformEnds &e)
{
    FirstPass p;
    const bool norm = e.grid.kind == ThcGrid::NORM;
    p.x = x; p.sign = a.sign; p.n = a.n; p.scale = a.scale;
    p.kt = (uint8_t)a.kt; p.kb = (uint8_t)a.kb; p.vec = (uint8_t)a.vec; p.sign_bits = (uint8_t)a.sign_bits; p.sign_mode = (uint8_t)sign_mode;
    p.gen_bits = (uint8_t)a.gen.bits; p.gen_ss = a.gen.ss;
    p.end = e.in_levels ? kLevelsEnd : (e.in_planes ? kPlanesEnd : (e.in_src ? kOther : kNoEnd));
    p.in = e.in_levels ? (const void *)e.in_levels : (e.in_planes ? (const void *)e.in_planes : e.in_src);
    p.p = e.in_planes ? e.in_centroids : (norm ? e.grid.norm : e.in_step);
    p.in_lo = e.in_lo; p.in_count = e.in_count;
    p.in_dtype = (uint8_t)e.in_dtype; p.in_nbits = (uint8_t)e.in_nbits;
    p.grid_kind = (uint8_t)e.grid.kind;
    const float grid[7] = {e.grid.lo, e.grid.spacing, e.grid.step, e.grid.t, e.grid.inv_sqrt, e.grid.inv_levels, e.grid.inv_clients};
    for (int k = 0; k < 7; k++) p.grid[k] = grid[k];
    return p;
}

inline StridedPass strided_of(float *x, const RhtPassArgs &a, int rbits, int sbits, int sign_mode, int apply_scale, const TransformEnds &e)
{
    StridedPass p;
    const bool norm = e.grid.kind == ThcGrid::NORM, levels = e.out_levels != nullptr;
    p.x = x; p.sign = a.sign; p.n = a.n; p.scale = a.scale;
    p.kt = (uint8_t)a.kt; p.vec = (uint8_t)a.vec; p.sign_bits = (uint8_t)a.sign_bits; p.sign_mode = (uint8_t)sign_mode;
    p.rbits = (uint8_t)rbits; p.sbits = (uint8_t)sbits; p.apply_scale = (uint8_t)apply_scale;
    p.gen_bits = (uint8_t)a.gen.bits; p.gen_ss = a.gen.ss;
    p.end = levels ? kLevelsEnd : (e.out_dst ? kOther : kNoEnd);
    p.out = levels ? (void *)e.out_levels : e.out_dst;
    p.p = levels ? e.uniform : e.post_scale;
    p.q = levels ? (const void *)(norm ? e.grid.norm : e.out_lo) : (const void *)e.sums;
    p.r = e.out_delta;
    p.count = levels ? e.zeros_from : e.out_count;
    p.out_dtype = (uint8_t)e.out_dtype; p.out_top = e.out_top;
    p.draw_bits = (int8_t)e.draw.bits; p.draw_seed = e.draw.seed; p.draw_counter = e.draw.counter;
    p.grid_kind = (uint8_t)e.grid.kind;
    p.grid[0] = norm ? e.grid.t : e.grid.lo;
    p.grid[1] = norm ? e.grid.inv_sqrt : e.grid.spacing;
    p.grid[2] = e.grid.inv_levels;
    return p;
}

// 30 to 50 KB of code a kernel: where it begins shows in passes of 10 us.  THC on 25 MB, nearly the same instructions 2.8 KB further on,
// 45.7 -> 46.7 us; begun at a multiple of 1 KB 46.5, of 4 KB 45.8, of 64 KB 45.5.
#define DQ_OWN_PAGES __attribute__((aligned(4096)))

template <bool ENDS> __global__ __launch_bounds__(512) void rht_strided_kernel(StridedPass p)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    strided_pass<ENDS>(p.x, pass_args<ENDS>(p), p.rbits, p.sbits, p.sign_mode, p.apply_scale, ends_of(p), blockIdx.x, lds);
}

// 512 (B = 4) or 1024 rows (B = 5)
template <bool ENDS, int B> DQ_OWN_PAGES __global__ __launch_bounds__(32 << B) void rht_strided_long_kernel(StridedPass p)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    strided_rows<ENDS, 5, B>(p.x, pass_args<ENDS>(p), p.sbits, p.sign_mode, p.apply_scale, ends_of(p), blockIdx.x, lds);
}

// 256 (A = 4) or 1024 rows (A = 5) to THC's levels with drawn values
template <int A> DQ_OWN_PAGES __global__ __launch_bounds__(32 << A) void rht_strided_draw_kernel(StridedPass p)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    strided_rows<true, A, A, true>(p.x, pass_args<true>(p), p.sbits, p.sign_mode, p.apply_scale, ends_of(p), blockIdx.x, lds);
}

template <bool ENDS> DQ_OWN_PAGES __global__ __launch_bounds__(1024) void rht_first_kernel(FirstPass p)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    first_pass<ENDS>(p.x, pass_args<ENDS>(p), p.sign_mode, ends_of(p), blockIdx.x, lds, tile_threads(p.kt),
                     ENDS && p.end != kNoEnd && p.n >= kEarlyFrom && p.n <= kEarlyTo);
}

#if DQ_RHT_PART & DQ_RHT_TRANSFORM
// ---- several vectors per launch (launch_rht_slices) -------------------------------------------------------------

struct PassSet {
    TilePass p[kMaxEdenSlices];
    int count;
};

// The set, the kernel's only argument, where it lies: by name, in more than a few hundred places, the compiler copies all 2 KB
// of it to scratch in front of the kernel, and a copy of one pass costs 0.5 us of loads that wait for one another.
__device__ __forceinline__ const TilePass &pass_of_block()
{
    const PassSet &set = *(const PassSet *)(const __attribute__((address_space(4))) PassSet *)__builtin_amdgcn_kernarg_segment_ptr();
    int k = 0;
    for (int i = 1; i < set.count; i++)
        if (blockIdx.x >= set.p[i].first) k = i;
    return set.p[k];
}

__device__ __forceinline__ RhtPassArgs pass_args(const TilePass &p)
{
    RhtPassArgs a;
    a.sign = nullptr; a.sign_bits = 0; a.n = p.n; a.kt = p.kt; a.kb = p.kb; a.scale = p.scale; a.vec = 1; a.gen = p.ends.gen;
    return a;
}

// (the largest pass gives every workgroup its threads and LDS: smaller tiles leave some of both idle)
__global__ __launch_bounds__(1024) void rht_tile_passes_kernel(PassSet set)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const TilePass &p = pass_of_block();
    first_pass<true>(p.x, pass_args(p), p.sign_mode, p.ends, blockIdx.x - p.first, lds, blockDim.x, false); // (slices end at 2^22 elements)
}

__global__ __launch_bounds__(512) void rht_strided_passes_kernel(PassSet set)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const TilePass &p = pass_of_block();
    strided_pass<true>(p.x, pass_args(p), p.rbits, p.sbits, p.sign_mode, p.apply_scale, p.ends, blockIdx.x - p.first, lds);
}
#endif

// ---- blocks of 2^15: the tile in two halves -----------------------------------------------------------
//
// A 2^15 tile with its padding needs 135 KB of LDS: one workgroup per CU, whose load, butterfly and
// quantise phases cannot overlap with a neighbour's.  Here thread t owns chunk t of both halves of the
// block: the stages of strides 1..8 run on registers, the stages of strides 16 .. 2^13 run in LDS one half
// after the other (68 KB: two workgroups per CU), and the last stage (stride 2^14) pairs the thread's own
// two chunks.  In the inverse kernel and the plain transform the record windows (and the MEE table) share the
// LDS with the tile: they are used only before the first half enters it or after the second has left.  The
// forward kernel keeps its second half in the LDS through the pairing stage and the quantiser of the first
// (see rht_compress_split_kernel).  All of them ask for eight waves per SIMD (64 registers): two resident
// workgroups are worth more than anything the register file could hold instead.
constexpr int kSplitBits = 15, kHalfBits = 14, kSplitThreads = 1024;

// stages of strides 16 .. 2^13 of the half block whose chunk t the thread holds in v (in and out)
template <int HB = kHalfBits>
__device__ __forceinline__ void half_block_stages(float (&v)[16], float *lds, int tid)
{
    float *mine = lds + chunk_word(tid);
#pragma unroll
    for (int i = 0; i < 16; i++) mine[i] = v[i];
    fwht_lds_stages_after4(lds, HB, HB, tid, 1 << (HB - 4));
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = mine[i];
    __syncthreads(); // the half has left the LDS
}

// The forward kernel takes blocks of 2^(HB + 1) in two halves of 2^HB, one chunk of each half per thread: HB = 14 for
// blocks of 2^15 (1024 threads; a CU holds at most two such workgroups), HB = 13 for blocks of 2^14 (512 threads, up to
// four per CU; as one tile those blocks need 1024 threads of which half sit idle in both LDS passes), ... HB = 10 for
// blocks of 2^11 on one wave.
//
// LDS: the half tile, in which the second half is parked through the quantiser of the first, and the record windows of
// the waves behind it.  For HB = 14 the sum must leave room for two workgroups per CU (80 KB each).
// records per window: four (one run per wave) where two workgroups of 2^15-element blocks still fit a CU with the parked half,
// two for the wider codes (7 and 8 bits), whose runs then leave in two pieces
template <int NBITS, int HB> __host__ __device__ constexpr int split_window_rows()
{
    return HB < kHalfBits || (size_t)padded_tile_floats(HB) * sizeof(float) + ((1 << (HB - 4)) / 64) * window_bytes<NBITS>(4) <= 80 * 1024 ? 4 : 2;
}
template <int NBITS, int HB> __host__ __device__ constexpr size_t split_lds_bytes()
{
    return (size_t)padded_tile_floats(HB) * sizeof(float) + ((1 << (HB - 4)) / 64) * window_bytes<NBITS>(split_window_rows<NBITS, HB>());
}

// PAIR = false: the two halves are two whole blocks of 2^HB (no pairing stage): blocks of 2^10 on one wave.
template <int RDT, int NBITS, bool MEE, int HB, bool PAIR = true>
__global__ __launch_bounds__(1 << (HB - 4), 8) void rht_compress_split_kernel(
    const float *__restrict__ x, uint8_t *__restrict__ dst, const void *__restrict__ rnd, RhtTileArgs a, int rvec, RandKey key,
    MeeArg<NBITS, MEE> mp)
{
    typedef Rec<NBITS> RC;
    constexpr int kThreads = 1 << (HB - 4), kWaves = kThreads / 64;
    constexpr int kWinRows = split_window_rows<NBITS, HB>();
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t origin = (int64_t)blockIdx.x << (HB + 1);
    float va[16], vb[16];
    load_chunk(va, x, a, origin + tid * 16);
    load_chunk(vb, x, a, origin + (1 << HB) + tid * 16);
    butterflies<4>(va);
    butterflies<4>(vb);
    half_block_stages<HB>(va, lds, tid);
    // The second half stays in the LDS after its stages: the thread pairs its two chunks there, keeps the sums and
    // leaves the differences in its own slot until the sums are quantised.  With both halves in registers through the
    // quantiser the kernel needs more than its 64 registers, and what it spills travels to memory and back (measured
    // at 2^28 elements in blocks of 2^15: 757 MB written and 1.52 GB read for 153 MB of records and 1.11 GB of input).
    // The record windows then lie behind the tile instead of inside it.
    float *mine = lds + chunk_word(tid);
#pragma unroll
    for (int i = 0; i < 16; i++) mine[i] = vb[i];
    fwht_lds_stages_after4(lds, HB, HB, tid, kThreads); // ends with a barrier; own slot only from here on
    if constexpr (PAIR) {
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const float p = va[i], q = mine[i];
            va[i] = p + q;
            mine[i] = p - q;
        }
    }
    uint8_t *win_out = reinterpret_cast<uint8_t *>(lds + padded_tile_floats(HB)) + wave * window_bytes<NBITS>(kWinRows);
    // quantise: the wave's 64 chunks of a half are 4 superchunks, one run of records
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int64_t sc0 = (origin >> 8) + h * (kWaves * kRowsPerWave) + wave * kRowsPerWave;
        Raw16<DQ_F32> v;
        Raw16<RDT> r;
        if constexpr (RDT == DQ_PHILOX)
            r.generate(key, sc0 * 16 + lane);
        else
            r.load(rnd, (sc0 * 16 + lane) * 16, rvec);
#pragma unroll
        for (int i = 0; i < 16; i++) v.w[i] = __float_as_uint((h ? mine[i] : va[i]) * a.scale);
        encode_store_run<NBITS, MEE, kWinRows, false>(v, r, mp, dst + sc0 * RC::REC, kRowsPerWave, win_out, threadIdx.x & 63);
        wave_lds_sync(); // the window is reused for the other half
    }
}

// The inverse: a block of 2^HB elements per workgroup, or (PAIR) one of 2^(HB + 1) in two halves.  A thread decodes a chunk of each half,
// which goes through the LDS twice (chunk_into_tile, middle_stages); the highest four stages, that between the halves, scale and signs
// are done on the registers that the last trip fills, and stored from there: consecutive lanes hold consecutive elements, a store of a
// wave is two whole lines, and their 64 signs are two words of the wave.  Bound by memory: the vector ALU is half busy, the LDS 40 %.
// Four accesses to the LDS per element where tiles read back by chunks took eight, and 6 barriers instead of 13: 2^30 elements in
// blocks of 2^13, 5 bits, 1,143 -> 990 us (5.1 TB/s; plain instead of non-temporal stores 1,130).
template <int NBITS, bool MEE, int HB, bool PAIR>
__global__ __launch_bounds__(1 << (HB - 4), 8) void irht_decompress_kernel(const uint8_t *__restrict__ src, float *__restrict__ x, RhtTileArgs a,
                                                                       MeeArg<NBITS, MEE> mp)
{
    typedef Rec<NBITS> RC;
    constexpr int kThreads = 1 << (HB - 4), kWaves = kThreads / 64, kParts = PAIR ? 2 : 1;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int chunk = chunk_of<HB>(lane), row = chunk >> 4, j = chunk & 15;
    const int64_t origin = (int64_t)blockIdx.x << (HB + (PAIR ? 1 : 0));
    // the record windows and the MEE table use the LDS before the tile does
    uint8_t *win_in = reinterpret_cast<uint8_t *>(lds) + wave * RC::WIN;
    float *table = reinterpret_cast<float *>(reinterpret_cast<uint8_t *>(lds) + kWaves * RC::WIN);
    constexpr int kTotal = kRowsPerWave * RC::REC;
    const auto records = [&](int h) { return src + ((origin >> 8) + h * (kWaves * kRowsPerWave) + wave * kRowsPerWave) * RC::REC; };
    WinRegs wr[kParts];
#pragma unroll
    for (int h = 0; h < kParts; h++) wr[h] = window_fetch(records(h), kTotal, lane);
    if (MEE) {
        for (int k = tid; k < (1 << NBITS); k += kThreads) table[k] = f16_bits_to_f32(mp.levels()[k]);
        __syncthreads();
    }
    float v[kParts][16];
#pragma unroll
    for (int h = 0; h < kParts; h++) {
        const int mis = window_commit(win_in, wr[h], records(h), kTotal, lane);
        wave_lds_sync();
        const uint8_t *rec = win_in + mis + row * RC::REC;
        uint32_t cw[RC::WORDS], cq;
        chunk_read<NBITS>(rec + j * RC::CB, cw, cq);
        const uint32_t ub = (uint32_t)rec[16 * RC::CB] | ((uint32_t)rec[16 * RC::CB + 1] << 8);
        chunk_decode<NBITS, MEE, false>(cw, cq, ub, table, v[h]);
        wave_lds_sync(); // the window is reused for the other half
    }
    __syncthreads(); // windows and table are done with: the tile takes the LDS
#pragma unroll
    for (int h = 0; h < kParts; h++) {
        chunk_into_tile<HB>(v[h], lds, tid);
        __syncthreads();
        middle_stages<HB>(lds, tid, kThreads);
        __syncthreads();
        const float *q = lds + pad_idx(tid);
#pragma unroll
        for (int k = 0; k < 16; k++) v[h][k] = q[tuple_step<HB - 4>(k)];
        butterflies<4>(v[h]);
        if (h + 1 < kParts) __syncthreads(); // the half has left the LDS
    }
    if constexpr (PAIR) {
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const float p = v[0][k], q = v[1][k];
            v[0][k] = p + q;
            v[1][k] = p - q;
            asm volatile("" : "+v"(v[1][k])); // (formed behind the stores of the first half, the differences keep both operands alive)
        }
    }
    const int64_t first = origin + 64 * wave; // of the wave's 64 consecutive elements
    float *out = x + first + lane;
#pragma unroll
    for (int h = 0; h < kParts; h++) {
#pragma unroll
        for (int k = 0; k < 16; k++) v[h][k] *= a.scale;
        if (a.sign && a.sign_bits) {
            // (scalar loads, which the compiler makes of nothing it thinks the stores could change)
            typedef const __attribute__((address_space(4))) uint32_t *constant_words;
            const constant_words words = (constant_words)(static_cast<const uint32_t *>(a.sign) + (first >> 5));
#pragma unroll
            for (int k = 0; k < 16; k++) {
                const int at = ((h << HB) + (k << (HB - 4))) >> 5;
                const uint64_t mask = (uint64_t)words[at] | ((uint64_t)words[at + 1] << 32);
                asm("v_cndmask_b32_e64 %0, %0, -%0, %1" : "+v"(v[h][k]) : "s"(mask));
            }
        } else if (a.sign) {
            const float *sign = static_cast<const float *>(a.sign) + first + lane;
#pragma unroll
            for (int k = 0; k < 16; k++) v[h][k] *= sign[(h << HB) + (k << (HB - 4))];
        }
#pragma unroll
        for (int k = 0; k < 16; k++) __builtin_nontemporal_store(v[h][k], out + (h << HB) + (k << (HB - 4)));
    }
}

// the transform alone on blocks of 2^15, the tile in two halves as above
__global__ __launch_bounds__(kSplitThreads, 8) void rht_tile_split_kernel(float *__restrict__ x, RhtTileArgs a, int sign_mode,
                                                                      int apply_scale)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = threadIdx.x;
    const int64_t origin = (int64_t)blockIdx.x << kSplitBits;
    RhtTileArgs in = a;
    if (sign_mode != 1) in.sign = nullptr;
    float va[16], vb[16];
    load_chunk(va, x, in, origin + tid * 16);
    load_chunk(vb, x, in, origin + (1 << kHalfBits) + tid * 16);
    butterflies<4>(va);
    butterflies<4>(vb);
    half_block_stages(va, lds, tid);
    half_block_stages(vb, lds, tid);
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const float p = va[i], q = vb[i];
        va[i] = p + q;
        vb[i] = p - q;
    }
    // store one half after the other through the LDS, so that every store instruction covers 1 KiB contiguously
    float *mine = lds + chunk_word(tid);
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int i = 0; i < 16; i++) mine[i] = h ? vb[i] : va[i];
        __syncthreads();
        const int64_t half_origin = origin + ((int64_t)h << kHalfBits);
        if (a.vec) {
            for (int i = tid * 4; i < (1 << kHalfBits); i += kSplitThreads * 4) {
                const int q = pad_idx(i);
                float4 v = make_float4(lds[q], lds[q + 1], lds[q + 2], lds[q + 3]);
                if (apply_scale) { v.x *= a.scale; v.y *= a.scale; v.z *= a.scale; v.w *= a.scale; }
                if (sign_mode == 2) flip4(v, a, half_origin + i);
                *reinterpret_cast<float4 *>(x + half_origin + i) = v;
            }
        } else {
            for (int i = tid; i < (1 << kHalfBits); i += kSplitThreads) {
                float v = lds[pad_idx(i)];
                if (apply_scale) v *= a.scale;
                x[half_origin + i] = sign_mode == 2 ? flip1(v, a, half_origin + i) : v;
            }
        }
        __syncthreads();
    }
}

constexpr int kPrefTileBits = 13; // 32 KiB tiles: eight waves, one run each, several workgroups per CU

struct Geometry {
    RhtTileArgs a;
    unsigned grid, threads;
    size_t lds_floats;
};

Geometry geometry(const float *vec, const void *sign, int sign_bits, int64_t n, int64_t block, float scale)
{
    Geometry g;
    const int kb = ilog2(block);
    int kt = kb < kPrefTileBits ? kPrefTileBits : kb;
    // short vectors: smaller tiles until there are two workgroups per CU (a tile is at least one run of 1024)
    while (kt > kb && kt > 10 && (n >> kt) < 512) kt--;
    while (kt > kb && kt > 8 && ((int64_t)1 << kt) > n) kt--;
    g.a.sign = sign; g.a.sign_bits = sign_bits; g.a.n = n; g.a.kt = kt; g.a.kb = kb; g.a.scale = scale;
    g.a.vec = aligned16(vec) && (sign == nullptr || sign_bits || aligned16(sign)) ? 1 : 0;
    const int tile = 1 << kt;
    g.threads = (unsigned)tile_threads(kt);
    g.grid = (unsigned)((n + tile - 1) >> kt);
    g.lds_floats = (size_t)padded_tile_floats(kt);
    return g;
}

template <class K> hipError_t allow_lds(K kernel, size_t bytes)
{
    if (bytes <= 48 * 1024) return hipSuccess;
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

// Blocks of 2^10 .. 2^14 as whole tiles, one chunk per thread, or in two halves, two chunks per thread.  Up to 2^23 elements
// all chunks fit the GPU at once (256 CUs x 2048 threads x 16 elements): then the halves only leave threads idle, and a block
// takes twice as long through its workgroup.  Beyond, the halves keep more loads in flight per thread and their tiles leave
// room for more workgroups.  Compress + decompress at 4 bits, in halves -> whole: 2^20 elements in blocks of 2^12 12.4 -> 10.1
// us, 2^14 17.1 -> 14.9, 2^22 15.9 -> 14.5, 2^23 23.7 -> 21.6, 2^24 39.7 -> 37.1; 2^25 68.6 against 68.7 and, in blocks of
// 2^10, 64.6 against 69.5.
constexpr int64_t kWholeTiles = (int64_t)1 << 23;

template <int RDT, int NBITS, bool MEE>
hipError_t run_compress(const float *src, const void *sign, int sign_bits, uint8_t *dst, const void *rnd, int64_t n, int64_t block,
                        float scale, const MeeParams &mp, RandKey key, hipStream_t stream)
{
    const Geometry g = geometry(src, sign, sign_bits, n, block, scale);
    const bool halves = n > kWholeTiles || g.a.kb == kSplitBits;
    if (halves && g.a.kb == 10 && (n & 2047) == 0) {
        // blocks of 2^10, two per wave
        auto kernel = rht_compress_split_kernel<RDT, NBITS, MEE, 10, false>;
        const size_t lds = split_lds_bytes<NBITS, 10>();
        hipLaunchKernelGGL(kernel, dim3((unsigned)(n >> 11)), dim3(64), lds, stream, src, dst, rnd, g.a, aligned16(rnd) ? 1 : 0, key,
                           make_arg<NBITS, MEE>(mp));
        return hipGetLastError();
    }
    if (halves && g.a.kb >= kSplitBits - 4 && g.a.kb <= kSplitBits && (n & ((1 << g.a.kb) - 1)) == 0) {
        // blocks of 2^11 .. 2^15: two halves per workgroup
        auto launch = [&](auto kernel, size_t lds, int half_bits) -> hipError_t {
            hipError_t es = allow_lds(kernel, lds);
            if (es != hipSuccess) return es;
            hipLaunchKernelGGL(kernel, dim3((unsigned)(n >> (half_bits + 1))), dim3(1 << (half_bits - 4)), lds, stream, src, dst, rnd,
                               g.a, aligned16(rnd) ? 1 : 0, key, make_arg<NBITS, MEE>(mp));
            return hipGetLastError();
        };
        switch (g.a.kb) {
        case kSplitBits:
            return launch(rht_compress_split_kernel<RDT, NBITS, MEE, kHalfBits>, split_lds_bytes<NBITS, kHalfBits>(), kHalfBits);
        case kSplitBits - 1:
            return launch(rht_compress_split_kernel<RDT, NBITS, MEE, kHalfBits - 1>, split_lds_bytes<NBITS, kHalfBits - 1>(), kHalfBits - 1);
        case kSplitBits - 2:
            return launch(rht_compress_split_kernel<RDT, NBITS, MEE, kHalfBits - 2>, split_lds_bytes<NBITS, kHalfBits - 2>(), kHalfBits - 2);
        case kSplitBits - 3:
            return launch(rht_compress_split_kernel<RDT, NBITS, MEE, kHalfBits - 3>, split_lds_bytes<NBITS, kHalfBits - 3>(), kHalfBits - 3);
        default:
            return launch(rht_compress_split_kernel<RDT, NBITS, MEE, kHalfBits - 4>, split_lds_bytes<NBITS, kHalfBits - 4>(), kHalfBits - 4);
        }
    }
    if (g.a.kt >= kSplitBits) return hipErrorInvalidValue; // one run of records per wave needs tiles of at most 2^14
    const size_t windows = (size_t)(g.threads / 64) * Rec<NBITS>::WIN;
    const size_t lds = std::max(g.lds_floats * sizeof(float), windows);
    auto kernel = rht_compress_kernel<RDT, NBITS, MEE>;
    hipError_t e = allow_lds(kernel, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(g.grid), dim3(g.threads), lds, stream, src, dst, rnd, g.a, aligned16(rnd) ? 1 : 0, key,
                       make_arg<NBITS, MEE>(mp));
    return hipGetLastError();
}

// The inverse, whole blocks or halves: with halves a thread has twice the loads and stores on the way and a block half the waves that
// meet at its barriers, while the vector leaves twice the threads idle.  us, whole against halves, 5 bits (4 up to 2^23):
//   blocks of  2^11          2^12          2^13          2^14
//   2^21        5.3    6.0    4.5    5.6    5.0    6.0    6.3    6.8
//   2^23        8.6    9.8    8.6   10.8    8.8   10.2   10.4   10.4  (2^22 8.1 against 7.2)
//   2^25       25.9   29.5   27.0   30.0   28.0   28.0   35.4   28.6
//   2^26       53.4   54.8   53.2   58.3   57.0   57.0   65.0   60.0
//   2^28        251    216    252    251    280    248    314    270
//   2^30       1000    881   1014    992   1124    983   1315   1074
// Blocks of 2^10 are one wave each (2^30 882 us; two blocks per wave 909), blocks of 2^15 do not fit as a whole.  Quarters and eighths
// are slower at every size: 100 and 150 registers.
constexpr int64_t kWholeInverse = (int64_t)1 << 26, kWholeInverse14 = (int64_t)1 << 21;

template <int PRE, int NBITS, bool MEE>
hipError_t run_decompress(const uint8_t *src, const void *sign, int sign_bits, float *dst, int64_t n, int64_t block, float scale,
                          const MeeParams &mp, hipStream_t stream)
{
    const Geometry g = geometry(dst, sign, sign_bits, n, block, scale);
    if (g.a.kb >= 10 && g.a.kb <= kSplitBits && (n & (((int64_t)1 << g.a.kb) - 1)) == 0) {
        const auto launch = [&](auto kernel, int part_bits) -> hipError_t {
            const size_t tile = (size_t)padded_tile_floats(part_bits) * sizeof(float);
            const size_t windows = (size_t)((1 << (part_bits - 4)) / 64) * Rec<NBITS>::WIN + (MEE ? (sizeof(float) << NBITS) : 0);
            const size_t lds = std::max(tile, windows);
            hipError_t es = allow_lds(kernel, lds);
            if (es != hipSuccess) return es;
            hipLaunchKernelGGL(kernel, dim3((unsigned)(n >> g.a.kb)), dim3(1 << (part_bits - 4)), lds, stream, src, dst, g.a, make_arg<NBITS, MEE>(mp));
            return hipGetLastError();
        };
        const bool whole = n <= (g.a.kb == 14 ? kWholeInverse14 : kWholeInverse);
        switch (g.a.kb) {
        case 15: return launch(irht_decompress_kernel<NBITS, MEE, 14, true>, 14);
        case 14: return whole ? launch(irht_decompress_kernel<NBITS, MEE, 14, false>, 14) : launch(irht_decompress_kernel<NBITS, MEE, 13, true>, 13);
        case 13: return whole ? launch(irht_decompress_kernel<NBITS, MEE, 13, false>, 13) : launch(irht_decompress_kernel<NBITS, MEE, 12, true>, 12);
        case 12: return whole ? launch(irht_decompress_kernel<NBITS, MEE, 12, false>, 12) : launch(irht_decompress_kernel<NBITS, MEE, 11, true>, 11);
        case 11: return whole ? launch(irht_decompress_kernel<NBITS, MEE, 11, false>, 11) : launch(irht_decompress_kernel<NBITS, MEE, 10, true>, 10);
        default: return launch(irht_decompress_kernel<NBITS, MEE, 10, false>, 10);
        }
    }
    if (g.a.kt >= kSplitBits) return hipErrorInvalidValue;
    const size_t windows = (size_t)(g.threads / 64) * Rec<NBITS>::WIN + (MEE ? (sizeof(float) << NBITS) : 0);
    const size_t lds = std::max(g.lds_floats * sizeof(float), windows);
    auto kernel = irht_decompress_tile_kernel<NBITS, MEE>;
    hipError_t e = allow_lds(kernel, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(g.grid), dim3(g.threads), lds, stream, src, dst, g.a, make_arg<NBITS, MEE>(mp));
    return hipGetLastError();
}

} // namespace

// one entry point per rounding source, each in a translation unit of its own
hipError_t launch_rht_compress_philox(const float *src, const void *sign, int sign_bits, uint8_t *dst, int64_t n, int64_t block, float scale,
                                      int nbits, bool mee, const MeeParams &mp, RandKey key, hipStream_t stream);
hipError_t launch_rht_compress_bf16_pool(const float *src, const void *sign, int sign_bits, uint8_t *dst, const void *rnd, int64_t n,
                                         int64_t block, float scale, int nbits, bool mee, const MeeParams &mp, hipStream_t stream);
hipError_t launch_rht_compress_f32_pool(const float *src, const void *sign, int sign_bits, uint8_t *dst, const void *rnd, int64_t n,
                                        int64_t block, float scale, int nbits, bool mee, const MeeParams &mp, hipStream_t stream);

#if DQ_RHT_PART & DQ_RHT_COMPRESS_PHILOX
hipError_t launch_rht_compress_philox(const float *src, const void *sign, int sign_bits, uint8_t *dst, int64_t n, int64_t block, float scale,
                                      int nbits, bool mee, const MeeParams &mp, RandKey key, hipStream_t stream)
{
    DQ_NBITS_MEE(run_compress, DQ_PHILOX, src, sign, sign_bits, dst, nullptr, n, block, scale, mp, key, stream)
}
#endif

#if DQ_RHT_PART & DQ_RHT_COMPRESS_BF16
hipError_t launch_rht_compress_bf16_pool(const float *src, const void *sign, int sign_bits, uint8_t *dst, const void *rnd, int64_t n,
                                         int64_t block, float scale, int nbits, bool mee, const MeeParams &mp, hipStream_t stream)
{
    const RandKey key{0, 0};
    DQ_NBITS_MEE(run_compress, DQ_BF16, src, sign, sign_bits, dst, rnd, n, block, scale, mp, key, stream)
}
#endif

#if DQ_RHT_PART & DQ_RHT_COMPRESS_F32
hipError_t launch_rht_compress_f32_pool(const float *src, const void *sign, int sign_bits, uint8_t *dst, const void *rnd, int64_t n,
                                        int64_t block, float scale, int nbits, bool mee, const MeeParams &mp, hipStream_t stream)
{
    const RandKey key{0, 0};
    DQ_NBITS_MEE(run_compress, DQ_F32, src, sign, sign_bits, dst, rnd, n, block, scale, mp, key, stream)
}
#endif

#if DQ_RHT_PART & DQ_RHT_TRANSFORM
// rand_kind: DQ_F32 or DQ_BF16 pool, or DQ_PHILOX (rnd ignored)
hipError_t launch_rht_compress(const float *src, const void *sign, int sign_bits, uint8_t *dst, const void *rnd, int rand_kind, int64_t n,
                               int64_t block, float scale, int nbits, bool mee, const MeeParams &mp, uint64_t seed,
                               uint64_t step, hipStream_t stream)
{
    if (rand_kind == DQ_PHILOX)
        return launch_rht_compress_philox(src, sign, sign_bits, dst, n, block, scale, nbits, mee, mp, RandKey{seed, step}, stream);
    if (rand_kind == DQ_BF16) return launch_rht_compress_bf16_pool(src, sign, sign_bits, dst, rnd, n, block, scale, nbits, mee, mp, stream);
    return launch_rht_compress_f32_pool(src, sign, sign_bits, dst, rnd, n, block, scale, nbits, mee, mp, stream);
}

// the 4-bit AEE kernel with the in-kernel rounding stream and the first four stages on the matrix cores (measurement variant)
hipError_t launch_rht_compress_mfma16(const float *src, const void *sign, int sign_bits, uint8_t *dst, int64_t n, int64_t block,
                                      float scale, const MeeParams &mp, uint64_t seed, uint64_t step, hipStream_t stream)
{
    const Geometry g = geometry(src, sign, sign_bits, n, block, scale);
    if (g.a.kb < 4 || g.a.kb >= kSplitBits || g.a.kt >= kSplitBits || g.a.kt < 10 || !g.a.vec || (n & ((1 << g.a.kt) - 1)) != 0 || (g.threads & 63) != 0)
        return hipErrorInvalidValue;
    const size_t windows = (size_t)(g.threads / 64) * Rec<4>::WIN;
    const size_t lds = std::max(g.lds_floats * sizeof(float), windows);
    auto kernel = rht_compress_kernel<DQ_PHILOX, 4, false, true>;
    hipError_t e = allow_lds(kernel, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(g.grid), dim3(g.threads), lds, stream, src, dst, nullptr, g.a, 0, RandKey{seed, step},
                       make_arg<4, false>(mp));
    return hipGetLastError();
}

#endif // DQ_RHT_TRANSFORM (first part)

#if DQ_RHT_PART & DQ_RHT_DECOMPRESS
hipError_t launch_irht_decompress(const uint8_t *src, const void *sign, int sign_bits, float *dst, int64_t n, int64_t block, float scale,
                                  int nbits, bool mee, const MeeParams &mp, hipStream_t stream)
{
    DQ_NBITS_MEE(run_decompress, 0, src, sign, sign_bits, dst, n, block, scale, mp, stream)
}
#endif

#if DQ_RHT_PART & DQ_RHT_TRANSFORM

// stages [0, kb) of every aligned block of 2^kb elements, tiles of 2^kt contiguous elements (10 <= kt <= 15, kb <= kt);
// vec: 16-byte accesses to x (and to a float sign vector) are allowed; ends: needs vec, n a multiple of 32 and 16-byte
// aligned levels
hipError_t launch_rht_tile(float *x, const void *sign, int sign_bits, int64_t n, int kt, int kb, float scale, int apply_scale,
                           int sign_mode, int vec, const TransformEnds &ends, hipStream_t stream)
{
    if (kt < 10 || kt > 15 || kb > kt || kb < 0) return hipErrorInvalidValue;
    const bool plain = ends.plain();
    if (!plain && (!vec || (n & 31) != 0)) return hipErrorInvalidValue;
    RhtPassArgs a;
    a.sign = sign; a.sign_bits = sign_bits; a.n = n; a.kt = kt; a.kb = kb; a.scale = scale; a.vec = vec; a.gen = ends.gen;
    const bool diagonal = sign || ends.gen.bits != 0;
    const RhtTileArgs &plain_args = a;
    const int tile = 1 << kt;
    if (plain && kt == kSplitBits && kb == kSplitBits && (n & (tile - 1)) == 0) {
        // whole blocks of 2^15: half the LDS, two workgroups per CU
        const size_t half_lds = (size_t)padded_tile_floats(kHalfBits) * sizeof(float);
        hipError_t es = allow_lds(rht_tile_split_kernel, half_lds);
        if (es != hipSuccess) return es;
        hipLaunchKernelGGL(rht_tile_split_kernel, dim3((unsigned)(n >> kSplitBits)), dim3(kSplitThreads), half_lds, stream, x, plain_args,
                           sign ? sign_mode : 0, apply_scale);
        return hipGetLastError();
    }
    const unsigned threads = (unsigned)tile_threads(kt);
    const size_t lds = ((size_t)padded_tile_floats(kt) + (ends.in_planes ? 256 : 0)) * sizeof(float);
    const dim3 grid((unsigned)((n + tile - 1) >> kt));
    if (sign_mode != 2 && !apply_scale && kb == kt && kt <= 14 && vec && (n & (tile - 1)) == 0 && ends.plain_out()) {
        const int mode = diagonal ? sign_mode : 0;
        const FirstPass pass = first_of(x, a, mode, ends);
        const auto launch = [&](auto kernel) -> hipError_t {
            const hipError_t e = allow_lds(kernel, lds);
            return e == hipSuccess ? launch_with(kernel, grid, dim3(threads), stream, pass, lds) : e;
        };
        return plain ? launch(rht_first_kernel<false>) : launch(rht_first_kernel<true>);
    }
    if (plain) {
        hipError_t e = allow_lds(rht_tile_kernel<false>, lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(rht_tile_kernel<false>, grid, dim3(threads), lds, stream, x, plain_args, sign ? sign_mode : 0, apply_scale, ends);
    } else {
        hipError_t e = allow_lds(rht_tile_kernel<true>, lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(rht_tile_kernel<true>, grid, dim3(threads), lds, stream, x, a, diagonal ? sign_mode : 0, apply_scale, ends);
    }
    return hipGetLastError();
}

// stages of the index bits [sbits, sbits + rbits) of x[0 .. n), n a multiple of 2^(sbits + rbits); 4 <= rbits <= 10, sbits >= 5
hipError_t launch_rht_strided(float *x, const void *sign, int sign_bits, int64_t n, int rbits, int sbits, float scale,
                              int apply_scale, int sign_mode, int vec, const TransformEnds &ends, hipStream_t stream)
{
    if (rbits < 4 || rbits > 10 || sbits < 5 || (n & (((int64_t)1 << (sbits + rbits)) - 1)) != 0) return hipErrorInvalidValue;
    const bool plain = ends.plain_out() && ends.gen.bits == 0;
    if (!plain && !vec) return hipErrorInvalidValue;
    const bool draws = ends.out_levels && ends.draw.bits >= 0;
    if (draws && ((rbits != 8 && rbits != 10) || sign_mode == 2 || ends.post_scale || ends.sums)) return hipErrorInvalidValue;
    RhtPassArgs a;
    a.sign = sign; a.sign_bits = sign_bits; a.n = n; a.kt = rbits + 5; a.kb = 0; a.scale = scale; a.vec = vec; a.gen = ends.gen;
    const dim3 grid((unsigned)(n >> (rbits + 5))), block((unsigned)strided_threads(rbits));
    const size_t lds = strided_lds_bytes(rbits);
    if (ends.out_levels && (ends.out_dst || ends.post_scale || ends.sums)) return hipErrorInvalidValue; // (they share a place)
    const StridedPass pass = strided_of(x, a, rbits, sbits, sign || ends.gen.bits != 0 ? sign_mode : 0, apply_scale, ends);
    const auto launch = [&](auto kernel) -> hipError_t {
        const hipError_t e = allow_lds(kernel, lds);
        return e == hipSuccess ? launch_with(kernel, grid, block, stream, pass, lds) : e;
    };
    if (plain) {
        if (rbits == 10) return launch(rht_strided_long_kernel<false, 5>);
        if (rbits == 9) return launch(rht_strided_long_kernel<false, 4>);
        return launch(rht_strided_kernel<false>);
    }
    if (draws) return rbits == 10 ? launch(rht_strided_draw_kernel<5>) : launch(rht_strided_draw_kernel<4>);
    if (rbits == 10) return launch(rht_strided_long_kernel<true, 5>);
    if (rbits == 9) return launch(rht_strided_long_kernel<true, 4>);
    return launch(rht_strided_kernel<true>);
}

// every x 16-byte aligned, n a multiple of 2^kt and 10 <= kt <= 14
hipError_t launch_rht_tile_passes(const TilePass *passes, int count, hipStream_t stream)
{
    PassSet set;
    set.count = count;
    unsigned blocks = 0;
    int most = 10;
    for (int k = 0; k < count; k++) {
        if (passes[k].kt < 10 || passes[k].kt > 14 || passes[k].kb != passes[k].kt || passes[k].sign_mode == 2 || passes[k].apply_scale || !passes[k].ends.plain_out() || (passes[k].n & ((1 << passes[k].kt) - 1)) != 0 || !aligned16(passes[k].x))
            return hipErrorInvalidValue;
        set.p[k] = passes[k];
        set.p[k].first = blocks;
        blocks += (unsigned)(passes[k].n >> passes[k].kt);
        most = std::max(most, passes[k].kt);
    }
    const size_t lds = ((size_t)padded_tile_floats(most) + 256) * sizeof(float);
    const hipError_t e = allow_lds(rht_tile_passes_kernel, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(rht_tile_passes_kernel, dim3(blocks), dim3(1u << (most - 4)), lds, stream, set);
    return hipGetLastError();
}

// every x 16-byte aligned, n a multiple of 2^(sbits + rbits), 4 <= rbits <= 8
hipError_t launch_rht_strided_passes(const TilePass *passes, int count, hipStream_t stream)
{
    PassSet set;
    set.count = count;
    unsigned blocks = 0;
    int most = 4;
    for (int k = 0; k < count; k++) {
        if (passes[k].rbits < 4 || passes[k].rbits > 8 || passes[k].sbits < 5 || (passes[k].n & (((int64_t)1 << (passes[k].sbits + passes[k].rbits)) - 1)) != 0 ||
            !aligned16(passes[k].x))
            return hipErrorInvalidValue;
        set.p[k] = passes[k];
        set.p[k].first = blocks;
        blocks += (unsigned)(passes[k].n >> (passes[k].rbits + 5));
        most = std::max(most, passes[k].rbits);
    }
    const size_t lds = strided_lds_bytes(most);
    const hipError_t e = allow_lds(rht_strided_passes_kernel, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(rht_strided_passes_kernel, dim3(blocks), dim3((unsigned)strided_threads(most)), lds, stream, set);
    return hipGetLastError();
}

#endif // DQ_RHT_TRANSFORM

} // namespace dq
