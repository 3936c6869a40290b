// EDEN's compress and decompress (srrcomp.py:293-361) of slices of at most 2^14 elements: one workgroup does the whole slice
// -- the load in the caller's type with the padding, every rotation, the sums, the bins and their planes, the scale -- and
// one launch all short slices of a vector.
//
// Such a slice is all latency: as launches of its own it took eight to ten of about 3.4 us each, every one of them a few
// workgroups.  A thread holds a chunk of sixteen consecutive elements, as in the tile passes of dq_rht_scaling_impl.cuh, and
// the chunk is what the quantiser wants of it too; LDS is only for the stages beyond the chunk and for the sums, whose
// association is that of dq_eden.hip.  The bits are those of the kernels there.
#define DQ_RHT_PART 0
#include "dq_eden.cuh"
#include "dq_rht_scaling_impl.cuh"

namespace dq {

namespace {

constexpr int kShortThreads = kEdenShort / 16;

// (one slice travels alone: an eighth of the arguments)
template <int MOST> struct ShortSet {
    dq_eden_slice_t s[MOST];
    float inv[MOST], sqrt_n[MOST]; // 1 / sqrt(n) and sqrt(n) as torch takes them
    int dtype;
    int threads; // of a workgroup
};

// the diagonal of one rotation (sign_seed of dq_hadamard.hip in 32-bit arithmetic: only low words are used)
__device__ __forceinline__ RhtPassArgs diagonal(int kb, int64_t seed)
{
    RhtPassArgs a;
    a.sign = nullptr;
    a.sign_bits = 0;
    a.gen.bits = kb - 3;
    a.gen.ss = ((uint32_t)seed * 1664525u + 1013904223u) * 8121u + 28411u;
    return a;
}

// all stages of the slice of 2^kb elements whose chunk tid is v, times scale
__device__ __forceinline__ void transform_chunk(float (&v)[16], int kb, float scale, float *lds, int tid, int nthreads)
{
    const bool mine = tid < (1 << kb) / 16;
    float *own = lds + chunk_word(tid);
    chunk_stages(v, kb);
    if (mine) {
#pragma unroll
        for (int i = 0; i < 16; i++) own[i] = v[i];
    }
    fwht_lds_stages_after4(lds, kb, kb, tid, nthreads);
    if (mine) {
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = own[i] * scale;
    }
}

// the fold of the one, two or four tiles' sums, each in the first of its tile's slots
__device__ __forceinline__ double fold_tiles(const double *sums, int n)
{
    if (n <= kEdenTile) return sums[0];
    if (n <= 2 * kEdenTile) return sums[0] + sums[kEdenThreads];
    return (sums[0] + sums[2 * kEdenThreads]) + (sums[kEdenThreads] + sums[3 * kEdenThreads]);
}

template <int NBITS, int MOST> __global__ __launch_bounds__(kShortThreads) void eden_short_compress_kernel(ShortSet<MOST> set)
{
    constexpr int L = 1 << NBITS;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    __shared__ double sums[kShortThreads];
    __shared__ float tree[L], cen[L];
    const int tid = threadIdx.x, nthreads = set.threads;
    const dq_eden_slice_t &s = set.s[blockIdx.x];
    const int n = (int)s.n, kb = 31 - __builtin_clz((unsigned)n);
    const bool mine = tid < n / 16;
    float v[16];
    TransformEnds e;
    e.in_src = s.vec;
    e.in_dtype = set.dtype;
    e.in_count = s.count;
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = 0.0f;
    if (mine) load_source(v, e, tid * 16);
    eden_tables<NBITS>(s.boundaries, s.centroids, tree, cen, tid, nthreads);
    for (int i = 0; i < s.rotations; i++) {
        if (mine) flip16(v, diagonal(kb, s.seed + i), tid * 16);
        transform_chunk(v, kb, set.inv[blockIdx.x], lds, tid, nthreads);
    }
    if (mine) {
#pragma unroll
        for (int i = 0; i < 16; i++) lds[chunk_word(tid) + i] = v[i];
    }
    __syncthreads();
    // tile g = threads 256 g .. 256 g + 255 (nthreads is a multiple of 256)
    const int t = tid & (kEdenThreads - 1), g = tid / kEdenThreads;
    float sum;
    if (sums_by_rows(n)) { // (n is then 16 nthreads: a piece of 32 columns per half of a wave, 32 of them)
        static_assert(kRowSumsFrom == kEdenShort, "the longest slice here");
        float w[16];
#pragma unroll
        for (int k = 0; k < 16; k++) w[k] = lds[pad_idx(k * kShortThreads + tid)];
        const double piece = sum_columns_f64(halve_squares(w));
        if ((tid & 31) == 0) sums[tid >> 5] = piece;
        __syncthreads();
        // (every wave the same)
        sum = (float)first_lane_f64(halve_row_f64(add_across_f64<16>(sums[tid & 31])));
    } else {
        double acc = 0.0;
#pragma unroll
        for (int k = 0; k < kEdenPerThread; k++) {
            const int i = g * kEdenTile + t + kEdenThreads * k;
            if (i < n) {
                const double x = (double)lds[pad_idx(i)];
                acc += x * x;
            }
        }
        fold256(acc, sums + g * kEdenThreads, t);
        sum = (float)fold_tiles(sums, n);
    }
    const float norm = __builtin_sqrtf(sum);
    __syncthreads();
    uint8_t *half = mine ? reinterpret_cast<uint8_t *>(s.packed) + 2 * tid : nullptr;
    const double dots = eden_bins_of<NBITS, kEdenPerThread>(v, norm, set.sqrt_n[blockIdx.x], tree, cen, half, n >> 5);
    fold256(mine ? dots : 0.0, sums + g * kEdenThreads, t);
    if (tid == 0) {
        const float d = (float)fold_tiles(sums, n);
        s.result[0] = sum;
        s.result[1] = d;
        s.result[2] = (norm * norm) / d;
        s.result[3] = norm;
    }
}

template <int MOST> __global__ __launch_bounds__(kShortThreads) void eden_short_decompress_kernel(ShortSet<MOST> set)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    __shared__ float cen[256];
    const int tid = threadIdx.x, nthreads = set.threads;
    const dq_eden_slice_t &s = set.s[blockIdx.x];
    const int n = (int)s.n, kb = 31 - __builtin_clz((unsigned)n);
    const bool mine = tid < n / 16;
    for (int k = tid; k < (1 << s.nbits); k += nthreads) cen[k] = s.centroids[k];
    __syncthreads();
    float v[16];
    TransformEnds e;
    e.in_planes = s.packed;
    e.in_nbits = s.nbits;
    e.out_dst = s.vec;
    e.out_dtype = set.dtype;
    e.out_count = s.count;
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = 0.0f;
    if (mine) load_planes(v, e, cen, tid * 16, n >> 5);
    for (int i = s.rotations - 1; i >= 0; i--) {
        transform_chunk(v, kb, set.inv[blockIdx.x], lds, tid, nthreads);
        if (mine) flip16(v, diagonal(kb, s.seed + i), tid * 16);
    }
    if (!mine) return;
    const float scale = *s.result;
#pragma unroll
    for (int k = 0; k < 4; k++)
        store_destination(e, make_float4(v[4 * k] * scale, v[4 * k + 1] * scale, v[4 * k + 2] * scale, v[4 * k + 3] * scale), tid * 16 + 4 * k);
}

// threads: a multiple of 256 that gives every chunk of the longest slice one
template <int MOST>
hipError_t short_set(const dq_eden_slice_t *slices, int count, int dtype, ShortSet<MOST> &set, unsigned *threads, size_t *lds)
{
    int64_t most = 32;
    if (count < 1 || count > kMaxEdenSlices) return hipErrorInvalidValue;
    for (int k = 0; k < count; k++) {
        if (slices[k].n > kEdenShort) return hipErrorInvalidValue;
        most = std::max(most, slices[k].n);
        set.s[k] = slices[k];
        set.sqrt_n[k] = (float)sqrt((double)slices[k].n);
        set.inv[k] = 1.0f / set.sqrt_n[k];
    }
    set.dtype = dtype;
    *threads = set.threads = (unsigned)((most / 16 + kEdenThreads - 1) / kEdenThreads * kEdenThreads);
    *lds = (size_t)padded_tile_floats(ilog2(most)) * sizeof(float);
    return hipSuccess;
}

template <int MOST> hipError_t short_compress(const dq_eden_slice_t *slices, int count, int dtype, hipStream_t stream)
{
    ShortSet<MOST> set;
    unsigned threads;
    size_t lds;
    const hipError_t e = short_set(slices, count, dtype, set, &threads, &lds);
    if (e != hipSuccess) return e;
    const auto go = [&](auto kernel) {
        const hipError_t allowed = allow_lds(kernel, lds);
        return allowed == hipSuccess ? launch_with(kernel, dim3((unsigned)count), dim3(threads), stream, set, lds) : allowed;
    };
    switch (slices[0].nbits) {
    case 1: return go(eden_short_compress_kernel<1, MOST>);
    case 2: return go(eden_short_compress_kernel<2, MOST>);
    case 3: return go(eden_short_compress_kernel<3, MOST>);
    case 4: return go(eden_short_compress_kernel<4, MOST>);
    case 5: return go(eden_short_compress_kernel<5, MOST>);
    case 6: return go(eden_short_compress_kernel<6, MOST>);
    case 7: return go(eden_short_compress_kernel<7, MOST>);
    default: return go(eden_short_compress_kernel<8, MOST>);
    }
}

template <int MOST> hipError_t short_decompress(const dq_eden_slice_t *slices, int count, int dtype, hipStream_t stream)
{
    ShortSet<MOST> set;
    unsigned threads;
    size_t lds;
    hipError_t e = short_set(slices, count, dtype, set, &threads, &lds);
    if (e == hipSuccess) e = allow_lds(eden_short_decompress_kernel<MOST>, lds);
    return e == hipSuccess ? launch_with(eden_short_decompress_kernel<MOST>, dim3((unsigned)count), dim3(threads), stream, set, lds) : e;
}

} // namespace

hipError_t launch_eden_short_compress(const dq_eden_slice_t *slices, int count, int dtype, hipStream_t stream)
{
    return count == 1 ? short_compress<1>(slices, count, dtype, stream) : short_compress<kMaxEdenSlices>(slices, count, dtype, stream);
}

hipError_t launch_eden_short_decompress(const dq_eden_slice_t *slices, int count, int dtype, hipStream_t stream)
{
    return count == 1 ? short_decompress<1>(slices, count, dtype, stream) : short_decompress<kMaxEdenSlices>(slices, count, dtype, stream);
}

} // namespace dq
