// Quantise and dequantise a chunk of 16 elements in registers, with the bit width as a value instead of a template
// parameter: what the kernels need that run compress -> decompress (or a whole chain of ring steps) without a packed
// stream in between.  Without the packing there is nothing in a chunk's arithmetic that depends on the width but a
// dozen constants, so one body serves the three widths of the dynamic mix, also where they differ inside a wave.
//
// The levels are those of chunk_encode_* followed by chunk_decode (dq_hier16_tiles.cuh), operation by operation; a code
// travels as the float level it decodes to instead of a bit field.
//
// The kernels on it are bound by the vector ALU.  Additions, products, fused multiply-adds, bitwise operations and right shifts on vector
// registers and constants issue a wave in 1.2 ns, everything else -- conversions, comparisons, minima, left shifts, double precision,
// and all of them with a scalar operand -- in 2.2.  So elements stay binary32 numbers in the precision of their type (round_element), the
// largest and the least of a lane's values come two to an instruction, and the scale byte from an estimate (chunk_ratio).  Kernels, us:
// one rank, nine 25 MB buckets 46.9 -> 43.1 (MEE 64 -> 60.3), ring of 8 x 1,000,003 14.4 -> 12.6 (MEE 16.0 -> 14.6), of 8 x 33,000,001 in
// MEE 265 -> 255; 8 x 124,439,808 in AEE, which memory bounds, 723 -> 725.
#pragma once

#include "dq_hier16_tiles.cuh"

namespace dq {

// 8, 4 and 2 bits, in this order everywhere
struct WidthConst {
    double inv_c, inv_l2b;     // MEE
    float inv_top;             // of R (AEE) or chunk_max_mee (MEE)
    float r;                   // R = 2^(bits - 1) - 1
    float bias, two_delta;     // of the level estimate: 1 + kDelta, 2 kDelta
    float c, cmm, l2b;         // MEE
};

struct WidthSet {
    WidthConst w[3];
};

// one width's constants in registers; table: its level zero among the floats in LDS (MEE)
template <bool MEE> struct WidthRegs {
    double inv_c, inv_l2b;
    float inv_top, r, bias, two_delta, c, cmm, l2b;
    const float *table;
};

template <bool MEE> __device__ __forceinline__ WidthRegs<MEE> width_regs(const WidthSet &s, int cls, const float *levels)
{
    WidthRegs<MEE> x;
    const auto pick = [cls](auto a, auto b, auto c) { return cls == 0 ? a : (cls == 1 ? b : c); };
    x.inv_top = pick(s.w[0].inv_top, s.w[1].inv_top, s.w[2].inv_top);
    x.r = pick(s.w[0].r, s.w[1].r, s.w[2].r);
    x.bias = pick(s.w[0].bias, s.w[1].bias, s.w[2].bias);
    x.two_delta = pick(s.w[0].two_delta, s.w[1].two_delta, s.w[2].two_delta);
    if (MEE) {
        x.inv_c = pick(s.w[0].inv_c, s.w[1].inv_c, s.w[2].inv_c);
        x.inv_l2b = pick(s.w[0].inv_l2b, s.w[1].inv_l2b, s.w[2].inv_l2b);
        x.c = pick(s.w[0].c, s.w[1].c, s.w[2].c);
        x.cmm = pick(s.w[0].cmm, s.w[1].cmm, s.w[2].cmm);
        x.l2b = pick(s.w[0].l2b, s.w[1].l2b, s.w[2].l2b);
        x.table = levels + pick(kLevels[0] + 127, kLevels[1] + 7, kLevels[2] + 1);
    } else {
        x.inv_c = x.inv_l2b = 0.0;
        x.c = x.cmm = x.l2b = 0.0f;
        x.table = nullptr;
    }
    return x;
}

// the three level tables into LDS (kLevelCount floats): the loads of every lane leave together
__device__ __forceinline__ void levels_to_lds(float *levels, int lane)
{
    const uint32_t *pairs = reinterpret_cast<const uint32_t *>(kMeeLevelsOfWidths.at);
    uint32_t p[3];
#pragma unroll
    for (int k = 0; k < 3; k++) p[k] = lane + 64 * k < kLevelCount / 2 ? pairs[lane + 64 * k] : 0u;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const int at = lane + 64 * k;
        if (at < kLevelCount / 2) {
            levels[2 * at] = f16_bits_to_f32(p[k] & 0xffffu);
            levels[2 * at + 1] = f16_bits_to_f32(p[k] >> 16);
        }
    }
}

// largest magnitude of N values; NaN if one of them is not a number (v_maximum3_f32: two values per instruction)
template <int N> __device__ __forceinline__ float abs_maximum(const float (&x)[N])
{
    float m = __builtin_fabsf(x[0]);
#pragma unroll
    for (int i = 1; i + 1 < N; i += 2)
        m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(x[i])), __builtin_fabsf(x[i + 1]));
    return N % 2 ? m : __builtin_elementwise_maximum(m, __builtin_fabsf(x[N - 1]));
}

// the least of N numbers
template <int N> __device__ __forceinline__ float minimum(const float (&x)[N])
{
    float m = x[0];
#pragma unroll
    for (int i = 1; i + 1 < N; i += 2) m = __builtin_elementwise_minimum(__builtin_elementwise_minimum(m, x[i]), x[i + 1]);
    return N % 2 ? m : __builtin_elementwise_minimum(m, x[N - 1]);
}

// A copy of a lane's random words about which the compiler knows nothing: for a rare path that takes its values from them again, instead
// of keeping all of them in registers for it.
template <class RR> __device__ __forceinline__ RR forgotten(const RR &r)
{
    static_assert(sizeof(RR) % 4 == 0, "words");
    union {
        RR r;
        uint32_t w[sizeof(RR) / 4];
    } u = {r};
#pragma unroll
    for (size_t k = 0; k < sizeof(RR) / 4; k++) asm volatile("" : "+v"(u.w[k]));
    return u.r;
}

// The binary32 quotient a / b by a constant, y its rounded reciprocal: a product and one correction, the correctly rounded quotient for b =
// 255, the greatest levels and the chunk maxima of the MEE lattices (every significand of a tried: tests/test_exact_division.py).
// Where a is so small that the remainder is not exact, a / b disappears in the sum with 1e-7.  (Two operations where the product with a
// reciprocal in double takes three, two of them conversions.)
__device__ __forceinline__ float divide_by_constant(float a, float b, float y)
{
    const float q = a * y;
    return __builtin_fmaf(__builtin_fmaf(-q, b, a), y, q);
}

// ceil(fl(fl(s / g) * 255)) between 1 and 255, for 1e-7 <= s <= g <= 2^101.  The estimate with the hardware's reciprocal (1 ulp) errs by
// less than 255 (2^-22 + 2^-23) + 2^-17 < 2^-13 = e, so floor(estimate + e) + 1 is the ceiling where no integer lies within e of the
// estimate; above 254 it is 255 whatever the ratio, which settles the row's largest chunk (s = g).
__device__ __forceinline__ float chunk_ratio(float s, float g)
{
    constexpr float e = 0x1p-13f;
    const float above = __builtin_fminf(__builtin_fmaf(s * __builtin_amdgcn_rcpf(g), 255.0f, e), 254.75f);
    const float down = __builtin_floorf(above);
    float q = down + 1.0f;
    const bool doubt = above - down < 2.0f * e;
    if (__builtin_amdgcn_ballot_w64(doubt) != 0) {
        asm volatile(""); // (a branch of the wave that the compiler keeps)
        if (doubt) q = __builtin_amdgcn_fmed3f(__builtin_ceilf(div_by(s, recip_f64(g)) * 255.0f), 1.0f, 255.0f);
    }
    return q;
}

// t in the precision of the element type.  A bfloat16 behind a zero is its own binary32 pattern: one conversion, where a pair of
// bfloat16 takes two more instructions to be floats again.
template <int DT> __device__ __forceinline__ float round_element(float t)
{
    if constexpr (DT == DQ_F32)
        return t;
    else
        return __uint_as_float(f32x2_to_bf16x2(0.0f, t));
}

// the quantiser with every guard of the reference (chunk_encode_guarded): lev[i] = level of element i, returns the
// chunk's step (chunk_decode's sc)
template <bool MEE, int N, class RR>
__device__ __forceinline__ float quantize_guarded(const float (&v)[N], const RR &rnd, const WidthRegs<MEE> &w, float (&lev)[N])
{
    float a = __builtin_fabsf(v[0]);
#pragma unroll
    for (int i = 1; i < N; i++) a = __builtin_fmaxf(a, __builtin_fabsf(v[i]));
    a = chunk_max<N>(a);
    const float s = pos_scale(MEE ? a / pos_scale(w.cmm) + 1e-7f : a / w.r + 1e-7f);
    const float g = pos_scale(superchunk_max<N>(s));
    const uint32_t unit_bits = f32_to_bf16_bits(pos_scale(g / 255.0f));
    const float unit = pos_scale(bf16_bits_to_f32(unit_bits));
    float ratio = pos_scale(s) / pos_scale(g) * 255.0f;
    if (!__builtin_isfinite(ratio)) ratio = ratio > 0.0f ? 255.0f : 1.0f;
    const int qi = min(max(sat_u16(__builtin_ceilf(ratio)), 1), 255);
    const float d = pos_scale(pos_scale((float)qi * unit));
    const int top = (int)w.r;
#pragma unroll
    for (int i = 0; i < N; i++) {
        float x = v[i] / d;
        if (MEE) x = mee_inverse_guarded(x, w.c, w.l2b);
        const int level = clamp_code(sr_guarded(x, rnd.get(i)), top) - top;
        lev[i] = MEE ? w.table[level] : (float)level;
    }
    return nonneg_scale((float)qi * nonneg_scale(bf16_bits_to_f32(unit_bits)));
}

// chunk_encode_fast + estimate_codes: elements finite and <= 2^100, random values in [0, 1].  The estimate is that of
// L - r + 1 instead of L - r + R + 1 -- its floor is the signed level -- against the same guard: the constant 1 + kDelta
// minus r is as exact (1 and 20 bits of fraction), and the fused multiply-add rounds a number of less magnitude.
// The guard: the estimate's distance from its floor, the least of the lane's first (v_minimum3_f32, two per instruction), and where any lane of
// the wave is in doubt the elements that are.
template <bool MEE, int N, class RR>
__device__ __forceinline__ float quantize_fast(const float (&v)[N], const RR &rnd, float amax, const WidthRegs<MEE> &w, float (&lev)[N])
{
    const float s = divide_by_constant(amax, MEE ? w.cmm : w.r, w.inv_top) + 1e-7f;
    const float g = superchunk_max_pos<N>(s);
    const float d = chunk_ratio(s, g) * round_element<DQ_BF16>(divide_by_constant(g, 255.0f, 1.0f / 255.0f));
    const float rd = __builtin_amdgcn_rcpf(d);
    const float rc = MEE ? (float)w.inv_c : 0.0f, rl2b = MEE ? (float)w.inv_l2b : 0.0f;
    uint32_t top_bit = 0x80000000u;
    if (MEE) asm("" : "+v"(top_bit));
    float above[N];
#pragma unroll
    for (int i = 0; i < N; i++) {
        const float off = below(rnd, i, w.bias);
        float t;
        if (MEE)
            t = __builtin_fmaf(__builtin_amdgcn_logf(__builtin_fmaf(__builtin_fabsf(v[i] * rd), rc, 1.0f)),
                               __uint_as_float(__builtin_amdgcn_bitop3_b32(__float_as_uint(v[i]), top_bit, __float_as_uint(rl2b), 0x6A)), off); // (v & top_bit) ^ rl2b
        else
            t = __builtin_fmaf(v[i], rd, off);
        // (floor and not t minus its fraction: in -2^-25 < t < 0 the fraction rounds to 1 - 2^-24 and the difference is not -1)
        const float fl = __builtin_floorf(t);
        above[i] = t - fl;
        lev[i] = __builtin_amdgcn_fmed3f(fl, -w.r, w.r);
    }
    if (__builtin_amdgcn_ballot_w64(minimum(above) < w.two_delta) != 0) {
        const RR again = forgotten(rnd);
        const double yd = recip_f64(d);
#pragma unroll
        for (int i = 0; i < N; i++) {
            const bool doubt = above[i] < w.two_delta;
            if (__builtin_amdgcn_ballot_w64(doubt) != 0) {
                const float sv = (float)exact_code_fast<MEE>(v[i], again.get(i), d, yd, w);
                if (doubt) lev[i] = __builtin_amdgcn_fmed3f(sv, -w.r, w.r);
            }
        }
    }
    if (MEE) {
#pragma unroll
        for (int i = 0; i < N; i++) lev[i] = w.table[(int)lev[i]];
    }
    return d; // (positive and finite, as its unit is: chunk_decode's guards are for records from elsewhere)
}

// levels of the lane's elements and step of their chunk; every lane of the wave must call
template <bool MEE, int N, class RR>
__device__ __forceinline__ float quantize_chunk(const float (&v)[N], const RR &rnd, const WidthRegs<MEE> &w, float (&lev)[N])
{
    // (the pattern of a NaN is above that of infinity)
    const uint32_t amax = chunk_max<N>(__float_as_uint(abs_maximum(v)));
    const bool lane_fast = amax <= kFastMaxBits && rnd.unit_interval();
    if (__builtin_amdgcn_ballot_w64(!lane_fast) == 0) return quantize_fast<MEE>(v, rnd, __uint_as_float(amax), w, lev);
    return quantize_guarded<MEE>(v, rnd, w, lev);
}

// mp: the MEE parameters of 8, 4 and 2 bits
inline WidthSet make_width_set(const MeeParams *mp, bool mee)
{
    static const int bits[3] = {8, 4, 2};
    WidthSet s;
    __builtin_memset(&s, 0, sizeof(s));
    for (int k = 0; k < 3; k++) {
        WidthConst &w = s.w[k];
        const int top = (1 << (bits[k] - 1)) - 1;
        const float delta = estimate_delta(bits[k], mee); // (kDelta of estimate_codes)
        w.r = (float)top;
        w.bias = 1.0f + delta;
        w.two_delta = 2.0f * delta;
        w.c = mp[k].c; w.cmm = mp[k].cmm; w.l2b = mp[k].l2b;
        w.inv_top = 1.0f / (mee ? mp[k].cmm : (float)top);
        w.inv_c = 1.0 / (double)mp[k].c;
        w.inv_l2b = 1.0 / (double)mp[k].l2b;
    }
    return s;
}

// ---- a lane's chunk at the ragged end of a vector ------------------------------------------------------

// Elements of a vector of n at and behind e (at most `most`, at least 0), where only the ragged end of the vector or an
// unaligned buffer looks at it: written as comparisons of e + i with n -- sixteen of 64 bits per chunk -- the compiler moves
// them out of that branch, in front of every tile (about 60 of the 270 vector instructions of a wave of ranks_stats_kernel).
__device__ __forceinline__ int left_here(int64_t n, int64_t e, int most)
{
    asm volatile("" : "+s"(n));
    return (int)max((int64_t)0, min((int64_t)most, n - e));
}

// Every element is loaded, those beyond the end from the last one's address, and then masked: sixteen loads in flight
// together.  (Each behind its own comparison they went one by one, and the one ragged wave of a launch outlasted the others:
// 4 of 26 us on 8 x 1,000,003 elements.)
template <int DT, class RV> __device__ __forceinline__ void load_chunk_guarded(RV &v, const void *src, int64_t e0, int64_t n)
{
    typedef typename ElemIO<DT>::storage elem;
    constexpr int N = RV::kCount;
    const int left = left_here(n, e0, N), last = max(left - 1, 0);
    const elem *p = static_cast<const elem *>(src) + min(e0, n - 1);
    elem x[N];
#pragma unroll
    for (int i = 0; i < N; i++) x[i] = p[min(i, last)];
    v.zero();
#pragma unroll
    for (int i = 0; i < N; i++) {
        if (DT == DQ_F32)
            v.w[i] = i < left ? __builtin_bit_cast(uint32_t, (float)x[i]) : 0u;
        else
            v.w[i >> 1] |= (i < left ? (uint32_t)x[i] : 0u) << (16 * (i & 1));
    }
}

// the lane's elements from e0 on, zero at and beyond n; ragged: the wave's tile reaches beyond n (uniform)
template <int DT, class RV>
__device__ __forceinline__ void load_chunk(RV &v, const void *src, int64_t e0, int64_t n, bool vec, bool ragged)
{
    if (!ragged)
        v.load(src, e0, vec);
    else
        load_chunk_guarded<DT>(v, src, e0, n);
}

// zeros at and beyond element n of the vector, and the precision of the element type
template <int DT, int N> __device__ __forceinline__ void finish_centered(float (&t)[N], int64_t e0, int64_t n, bool ragged)
{
    if (ragged) {
        const int left = left_here(n, e0, N);
#pragma unroll
        for (int i = 0; i < N; i++) {
            // (In place: as a selection the tiles that are not ragged copy every element.  The comparison that writes the mask may come
            // directly before, and the two wait states between the two are the compiler's only for its own instructions.)
            const uint64_t inside = __builtin_amdgcn_ballot_w64(i < left);
            asm volatile("s_nop 1\n\tv_cndmask_b32_e64 %0, 0, %0, %1" : "+v"(t[i]) : "s"(inside));
        }
    }
#pragma unroll
    for (int i = 0; i < N; i++) t[i] = round_element<DT>(t[i]);
}

// t = T(v / world - mean), zero at and beyond element n of the vector (center_chunk without its own loads).  For 16-bit elements every
// power of two that a ring has ranks is fuse16's (and the general quotient is right for the others).
template <int DT, class RV>
__device__ __forceinline__ void center_loaded(float (&t)[RV::kCount], const RV &v, const WorldDiv &wd, float mean, int64_t e0, int64_t n, bool ragged)
{
    constexpr int N = RV::kCount;
    float inv = wd.inv;
    asm("" : "+v"(inv)); // (an instruction with a scalar operand takes nearly twice the time of one without)
    if (DT != DQ_F32 && wd.fuse16) {
#pragma unroll
        for (int i = 0; i < N; i++) t[i] = __builtin_fmaf(v.get(i), inv, -mean);
    } else if (DT == DQ_F32 && wd.pow2) {
#pragma unroll
        for (int i = 0; i < N; i++) t[i] = v.get(i) * inv - mean;
    } else {
#pragma unroll
        for (int i = 0; i < N; i++) t[i] = v.get(i);
        wd.divide(t);
#pragma unroll
        for (int i = 0; i < N; i++) t[i] -= mean;
    }
    finish_centered<DT>(t, e0, n, ragged);
}

// ---- statistics of a tile of four superchunks -----------------------------------------------------------

template <int CTRL> __device__ __forceinline__ float dpp_row_shift(float v)
{
    // lanes without a source inside the row receive 0; they only feed partial sums that are never read again
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}

template <int DT> struct StatsTile {
    static constexpr int ESZ = DT == DQ_F32 ? 4 : 2;
    static constexpr int RS = 256 * ESZ + 16 * ESZ; // padded row stride: the four rows use disjoint banks
    static constexpr int BYTES = 4 * RS;
};

// Sum and sum of squares of v / world over each superchunk of the wave's tile in the reference's reduction order
// (csrc/cuda_hadamard.cu:1286-1292: strides 128 ... 1), from the lane's chunk: the elements go through LDS once so that
// lane (row r, column j) holds elements j + 16 k of superchunk r -- strides 128 .. 16 are then additions in the lane,
// strides 8 .. 1 row shifts.  lds: StatsTile<DT>::BYTES, 16-byte aligned, owned by this wave.  sum and sq are complete in
// the lanes j == 0.
template <int DT> __device__ __forceinline__ void staged_tile_sums(const WorldDiv &wd, const uint8_t *lds, int lane, float &sum, float &sq);

template <int DT>
__device__ __forceinline__ void tile_sums(const Raw16<DT> &v, const WorldDiv &wd, uint8_t *lds, int lane, float &sum, float &sq)
{
    typedef StatsTile<DT> ST;
    const int row = lane >> 4, j = lane & 15;
#pragma unroll
    for (int k = 0; k < Raw16<DT>::kSlots; k++)
        *reinterpret_cast<uint4 *>(lds + row * ST::RS + j * 16 * ST::ESZ + 16 * k) = v.slot(k);
    wave_lds_sync();
    staged_tile_sums<DT>(wd, lds, lane, sum, sq);
}

// strides 64 .. 1 of the sums and the squares
__device__ __forceinline__ void fold_tile_sums(float (&a)[8], float (&b)[8], float &sum, float &sq)
{
#pragma unroll
    for (int k = 0; k < 4; k++) {
        a[k] += a[k + 4];
        b[k] += b[k + 4];
    }
    sum = (a[0] + a[2]) + (a[1] + a[3]);
    sq = (b[0] + b[2]) + (b[1] + b[3]);
    sum += dpp_row_shift<0x108>(sum);
    sq += dpp_row_shift<0x108>(sq);
    sum += dpp_row_shift<0x104>(sum);
    sq += dpp_row_shift<0x104>(sq);
    sum += dpp_row_shift<0x102>(sum);
    sq += dpp_row_shift<0x102>(sq);
    sum += dpp_row_shift<0x101>(sum);
    sq += dpp_row_shift<0x101>(sq);
}

// of the tile in LDS
template <int DT> __device__ __forceinline__ void staged_tile_sums(const WorldDiv &wd, const uint8_t *lds, int lane, float &sum, float &sq)
{
    typedef StatsTile<DT> ST;
    const int row = lane >> 4, j = lane & 15;
    const uint8_t *mine = lds + row * ST::RS + j * ST::ESZ;
    float t[16];
#pragma unroll
    for (int k = 0; k < 16; k++) {
        if (DT == DQ_F32)
            t[k] = *reinterpret_cast<const float *>(mine + 16 * k * ST::ESZ);
        else
            t[k] = bf16_bits_to_f32(*reinterpret_cast<const uint16_t *>(mine + 16 * k * ST::ESZ));
    }
    if (wd.pow2) {
        if (wd.inv != 1.0f) {
#pragma unroll
            for (int k = 0; k < 16; k++) t[k] = t[k] * wd.inv;
        }
    } else {
        wd.divide(t);
    }
    float a[8], b[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        a[k] = t[k] + t[k + 8];
        b[k] = t[k] * t[k] + t[k + 8] * t[k + 8];
    }
    fold_tile_sums(a, b, sum, sq);
}

// The same where the lane has its elements as numbers, already divided by world, and needs them as such again: they go through the LDS in
// binary32, which spares the kernel of one rank sixteen conversions and a second division.  The 16-byte pieces of a lane change
// places by its number, so that eight lanes writing theirs touch 32 different banks.
constexpr int kFloatRow = 256 + 16, kFloatTileBytes = 4 * kFloatRow * (int)sizeof(float);

__device__ __forceinline__ void float_tile_sums(const float (&t)[16], float *lds, int lane, float &sum, float &sq)
{
    const int row = lane >> 4, j = lane & 15;
    float *mine = lds + row * kFloatRow + j * 16;
#pragma unroll
    for (int p = 0; p < 4; p++)
        *reinterpret_cast<float4 *>(mine + 4 * (p ^ ((j >> 1) & 3))) = make_float4(t[4 * p], t[4 * p + 1], t[4 * p + 2], t[4 * p + 3]);
    wave_lds_sync();
    // element j of lane k's sixteen
    float x[16];
#pragma unroll
    for (int k = 0; k < 16; k++) x[k] = lds[row * kFloatRow + 16 * k + (j ^ (4 * ((k >> 1) & 3)))];
    float a[8], b[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        a[k] = x[k] + x[k + 8];
        b[k] = x[k] * x[k] + x[k + 8] * x[k + 8];
    }
    fold_tile_sums(a, b, sum, sq);
}

// the mean the reference divides out: sum / 256 exactly, or by the count of a ragged last superchunk
__device__ __forceinline__ float superchunk_mean(float sum, int64_t first, int64_t n, bool ragged)
{
    if (!ragged) return sum * 0.00390625f;
    const int valid = left_here(n, first, 256);
    return valid >= 256 ? sum * 0.00390625f : sum / (float)valid;
}

} // namespace dq
