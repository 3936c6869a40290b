// The consumers of the rotated vector: EDEN's Lloyd-Max quantiser with its bit-plane packer
// (cuda_kernels/src/srrcomp/srrcomp.py:293-361) and THC's uniform stochastic quantiser
// (testbed_evaluation/new_comm_hooks/thc_hooks.py:149-181), which the reference runs as chains of
// torch element-wise ops and reductions around eden_utils.Hadamard.
//
// EDEN quantise, three launches, no host synchronisation:
//   sumsq   n = 2^k >= 2^14: in the order of dq_sums.cuh; workgroup b adds the pieces b + i n/4096, i < 8 -> work[b].
//           Any other n: tile b = elements [4096 b, 4096 b + 4096): thread t adds v^2 of elements t + 256 k (k ascending)
//           in double, the 256 sums are halved (stride 128 .. 1) -> work[b]
//   bins    every workgroup folds work[] the same way -> sumsq (double); norm = sqrtf((float)sumsq);
//           x = (v * (float)sqrt(n)) / norm; bin = number of boundaries b with !(b >= x) (torch.bucketize, right=False: NaN -> last bin);
//           bit plane p of 32 consecutive bins -> packed[p * n/32 + w]; the products centroid[bin] * v are
//           summed in double, thread t adding elements 16 t + k of the tile (k ascending), then halved -> work[tiles + b]
//   scale   dot = fold(work[tiles ..]); scale = (norm * norm) / (float)dot
// Beyond 1024 partial sums (2^22 elements) the fold of sumsq is a launch of its own (eden_norm_kernel): in every workgroup it
// would read more than the workgroup's own elements; the products then go to work[b].
// In compress a rotation of more than one pass leaves the partial sums itself, one per workgroup of its strided pass: no sumsq
// launch, and at most 1024 of them up to 2^25 elements.  Both directions at 4 bits: 2^20 elements 34.0 -> 30.1 us, 500,000
// 31.9 -> 29.2, 12,000,000 136.6 -> 128.4.
// (scale inside bins, by the workgroup that finishes last: its release of the other XCDs' sums costs more than the launch --
// bins 5.7 -> 10.8 us at 2^20 elements, against 1.8 us for scale.)
// The sums are in double with a fixed association, so the result does not depend on the launch geometry -- nor on which launch
// adds the squares, nor on the slices that travel with this one -- and the CPU restatement reproduces it bit for bit.
#include <mutex>
#include <vector>

#include "dq_eden.cuh"
#include "dq_launch.h"

namespace dq {

namespace {

// Several slices in one launch: slice k owns the workgroups from first[k] on, one per tile.  A single slice travels alone: 96 bytes of
// arguments instead of 568, which take the host and the GPU 1 us longer a launch (launch_with).
template <int MOST> struct QuantizeSet {
    QuantizeSlice s[MOST];
    unsigned first[MOST];
    int count;
    bool fold;
    const float *boundaries, *centroids;
    __device__ __forceinline__ int slice_of_block() const
    {
        int k = 0;
        if constexpr (MOST > 1) {
            for (int i = 1; i < count; i++)
                if (blockIdx.x >= first[i]) k = i;
        }
        return k;
    }
};

// A whole tile's loads leave together; behind a comparison each they wait for one another (6.9 -> 3.2 us at 2^20 elements).
template <int MOST> __global__ __launch_bounds__(kEdenThreads) void eden_sumsq_kernel(QuantizeSet<MOST> set)
{
    __shared__ double lds[kEdenThreads];
    const int which = set.slice_of_block();
    const QuantizeSlice &s = set.s[which];
    const int64_t tile = blockIdx.x - set.first[which], base = tile * kEdenTile;
    float v[kEdenPerThread];
    if (sums_by_rows(s.n)) {
        const int piece = threadIdx.x >> 5;
        const float *vec = s.vec + (tile + piece * (s.n / kEdenTile)) * 32 + (threadIdx.x & 31);
#pragma unroll
        for (int k = 0; k < kEdenPerThread; k++) v[k] = vec[k * (s.n / kEdenPerThread)];
        const double sum = sum_columns_f64(halve_squares(v));
        if ((threadIdx.x & 31) == 0) lds[piece] = sum;
        __syncthreads();
        if (threadIdx.x < 64) {
            const double total = halve_row_f64(threadIdx.x < kEdenThreads / 32 ? lds[threadIdx.x] : 0.0);
            if (threadIdx.x == 0) s.work[tile] = total;
        }
        return;
    }
    const float *vec = s.vec + base + threadIdx.x;
    const int left = (int)min((int64_t)kEdenTile, s.n - base);
    if (left == kEdenTile) {
#pragma unroll
        for (int k = 0; k < kEdenPerThread; k++) v[k] = vec[kEdenThreads * k];
    } else {
#pragma unroll
        for (int k = 0; k < kEdenPerThread; k++) v[k] = (int)threadIdx.x + kEdenThreads * k < left ? vec[kEdenThreads * k] : 0.0f;
    }
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < kEdenPerThread; k++) acc = __builtin_fma((double)v[k], (double)v[k], acc); // (the square is exact)
    const double total = fold256(acc, lds, threadIdx.x);
    if (threadIdx.x == 0) s.work[tile] = total;
}

// folds work[0 .. count): thread t adds entries t + 256 k (k ascending), then the halving tree
__device__ __forceinline__ double fold_array(const double *work, int64_t count, double *lds, double acc)
{
    if (threadIdx.x < kEdenThreads) { // (of a workgroup with more)
        for (int64_t i = threadIdx.x + kEdenThreads; i < count; i += kEdenThreads) acc += work[i];
        lds[threadIdx.x] = acc;
    }
    return fold256_of(lds, threadIdx.x);
}
// (the thread's first entry may be asked for earlier)
__device__ __forceinline__ double first_of_array(const double *work, int64_t count)
{
    return threadIdx.x < kEdenThreads && threadIdx.x < count ? work[threadIdx.x] : 0.0;
}
__device__ __forceinline__ double fold_array(const double *work, int64_t count, double *lds)
{
    return fold_array(work, count, lds, first_of_array(work, count));
}
// the sums of squares of n elements, at most kEdenFoldTiles of them: by rows it is the halving tree all the way (as the fold above
// is for up to two entries a thread)
__device__ __forceinline__ double fold_sums(const double *sums, int64_t count, int64_t n, double *lds, double acc)
{
    static_assert(kEdenFoldTiles == 4 * kEdenThreads, "four entries a thread at most");
    if (count == kEdenFoldTiles && sums_by_rows(n)) {
        if (threadIdx.x < kEdenThreads) {
            const double *mine = sums + threadIdx.x;
            lds[threadIdx.x] = (acc + mine[2 * kEdenThreads]) + (mine[kEdenThreads] + mine[3 * kEdenThreads]);
        }
        return fold256_of(lds, threadIdx.x);
    }
    return fold_array(sums, count, lds, acc);
}

// result[0] = (float)sumsq, result[3] = norm
// By rows a thread halves its entries t + 256 k in place, sixteen at a time (nobody else reads them): compress of 2^26 elements,
// 32,768 sums, 396 us with one chain of additions per thread, 371 so.
__global__ __launch_bounds__(kEdenThreads) void eden_norm_kernel(double *sums, int64_t count, int64_t n, float *__restrict__ result)
{
    __shared__ double lds[kEdenThreads];
    if (sums_by_rows(n)) {
        double *mine = sums + threadIdx.x;
        int64_t left = count / kEdenThreads;
        double x[16];
        while (left > 16) {
            left /= 16;
            for (int64_t k = 0; k < left; k++) {
#pragma unroll
                for (int i = 0; i < 16; i++) x[i] = mine[(k + i * left) * kEdenThreads];
                mine[k * kEdenThreads] = halve(x);
            }
        }
#pragma unroll
        for (int i = 0; i < 16; i++) x[i] = i < left ? mine[i * kEdenThreads] : 0.0;
        lds[threadIdx.x] = halve(x);
    }
    const double sumsq = sums_by_rows(n) ? fold256_of(lds, threadIdx.x) : fold_array(sums, count, lds);
    if (threadIdx.x == 0) {
        const float s = (float)sumsq;
        result[0] = s;
        result[3] = __builtin_sqrtf(s);
    }
}

// A thread owns PER = 8 or 16 consecutive elements, two or four 16-byte loads, so that it builds its byte or half word of every
// bit plane in registers; the additions are the same in the same order.
// FOLD: the norm is not in result[3] yet; the workgroup folds the partial sums the way eden_norm_kernel does (the same
// association: the same bits), workgroup 0 leaves result[0] and result[3] as that kernel would, and the
// products go to a region of their own (other workgroups are still reading the sums).
template <int NBITS, bool FOLD, int PER, int MOST>
__global__ __launch_bounds__(kEdenTile / PER) void eden_bins_kernel(QuantizeSet<MOST> set)
{
    constexpr int L = 1 << NBITS;
    __shared__ double lds[kEdenThreads];
    __shared__ float tree[L], cen[L];
    const int which = FOLD ? set.slice_of_block() : 0;
    const QuantizeSlice &s = set.s[which];
    const int64_t tile = blockIdx.x - (FOLD ? set.first[which] : 0u);
    const int64_t tiles = eden_tiles(s.n);
    // n is a multiple of 32: the thread's elements are all inside the vector or all outside
    const int64_t first = tile * kEdenTile + (int64_t)threadIdx.x * PER;
    const bool in = first < s.n;
    float v[PER];
    if (in) {
        const float *vec = s.vec;
        if ((reinterpret_cast<uintptr_t>(vec) & 15) == 0) { // uniform over the grid
#pragma unroll
            for (int q = 0; q < PER / 4; q++) {
                const float4 f = *reinterpret_cast<const float4 *>(vec + first + 4 * q);
                v[4 * q] = f.x; v[4 * q + 1] = f.y; v[4 * q + 2] = f.z; v[4 * q + 3] = f.w;
            }
        } else {
#pragma unroll
            for (int k = 0; k < PER; k++) v[k] = vec[first + k];
        }
    } else {
#pragma unroll
        for (int k = 0; k < PER; k++) v[k] = 0.0f;
    }
    const double part = FOLD ? first_of_array(s.sums, s.sum_count) : 0.0;
    eden_tables<NBITS>(set.boundaries, set.centroids, tree, cen, threadIdx.x, kEdenTile / PER);
    __syncthreads();
    float norm;
    if constexpr (FOLD) {
        const float sum = (float)fold_sums(s.sums, s.sum_count, s.n, lds, part);
        norm = __builtin_sqrtf(sum);
        if (tile == 0 && threadIdx.x == 0) {
            s.result[0] = sum;
            s.result[3] = norm;
        }
    } else {
        norm = s.result[3];
    }
    // plane p, word (first >> 5), half (first >> 4) & 1; threads past the end hold zeros and drop their sum
    uint8_t *piece = in ? reinterpret_cast<uint8_t *>(s.packed) + (first >> 3) : nullptr;
    const double acc = eden_bins_of<NBITS, PER>(v, norm, s.sqrt_n, tree, cen, piece, s.n >> 5);
    if (PER == 16 || (threadIdx.x & 1)) lds[threadIdx.x / (16 / PER)] = in ? acc : 0.0;
    const double total = fold256_of(lds, threadIdx.x);
    if (threadIdx.x == 0) s.work[(FOLD && s.sums == s.work ? tiles : 0) + tile] = total;
}

// one workgroup per slice: result[1] = (float)dot, result[2] = scale
template <int MOST> __global__ __launch_bounds__(kEdenThreads) void eden_scale_kernel(QuantizeSet<MOST> set)
{
    __shared__ double lds[kEdenThreads];
    const QuantizeSlice &s = set.s[blockIdx.x];
    const int64_t tiles = eden_tiles(s.n);
    const double dot = fold_array(s.work + (set.fold && s.sums == s.work ? tiles : 0), tiles, lds);
    if (threadIdx.x == 0) {
        const float d = (float)dot;
        const float norm = s.result[3];
        s.result[1] = d;
        s.result[2] = (norm * norm) / d;
    }
}

// sixteen consecutive elements per thread: its half word of every bit plane, transposed back into sixteen bins;
// the centroids leave through a per-wave LDS tile so that the lanes store contiguous 16-byte pieces
template <int NBITS>
__global__ __launch_bounds__(256) void eden_dequantize_kernel(const uint32_t *__restrict__ packed, int64_t n,
                                                              const float *__restrict__ centroids, float *__restrict__ out)
{
    constexpr int L = 1 << NBITS;
    __shared__ float cen[L];
    __shared__ __attribute__((aligned(16))) uint4 tiles[4][256];
    for (int k = threadIdx.x; k < L; k += 256) cen[k] = centroids[k];
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t first = g * 16, wave_first = (g - lane) * 16;
    if (wave_first >= n) return; // the whole wave
    const int64_t words = n >> 5;
    uint64_t lo = 0, hi = 0;
    if (first < n) { // n is a multiple of 32
        const uint16_t *half = reinterpret_cast<const uint16_t *>(packed) + g;
#pragma unroll
        for (int p = 0; p < NBITS; p++) {
            const uint32_t h = half[(int64_t)p * words * 2];
            lo |= (uint64_t)(h & 0xffu) << (8 * p);
            hi |= (uint64_t)(h >> 8) << (8 * p);
        }
    }
    lo = transpose8x8(lo);
    hi = transpose8x8(hi);
    uint32_t w[16];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        w[k] = __float_as_uint(cen[(lo >> (8 * k)) & 0xffu]);
        w[8 + k] = __float_as_uint(cen[(hi >> (8 * k)) & 0xffu]);
    }
    store_wave_words16(tiles[wave], w, reinterpret_cast<uint4 *>(out + wave_first), lane,
                       (int)min((int64_t)256, (n - wave_first) >> 2));
}

// ---- THC ------------------------------------------------------------------------------------------

// levels stored as bf16; VEC: four elements per thread through 16-byte loads and one 8-byte store
template <bool VEC>
__global__ __launch_bounds__(256) void thc_quantize_kernel(const float *__restrict__ rotated, const float *__restrict__ uniform,
                                                           uint16_t *__restrict__ out, int64_t begin, int64_t n,
                                                           const float *__restrict__ lo_p, const float *__restrict__ delta_p,
                                                           float top)
{
    const float lo = *lo_p, delta = *delta_p;
    if (VEC) {
        const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
        if (i + 4 > n) return;
        const float4 v = *reinterpret_cast<const float4 *>(rotated + i);
        const float4 u = *reinterpret_cast<const float4 *>(uniform + i);
        uint2 o;
        o.x = f32x2_to_bf16x2(thc_level(v.x, u.x, lo, delta, top), thc_level(v.y, u.y, lo, delta, top));
        o.y = f32x2_to_bf16x2(thc_level(v.z, u.z, lo, delta, top), thc_level(v.w, u.w, lo, delta, top));
        *reinterpret_cast<uint2 *>(out + i) = o;
    } else {
        const int64_t i = begin + (int64_t)blockIdx.x * 256 + threadIdx.x;
        if (i >= n) return;
        out[i] = (uint16_t)f32_to_bf16_bits(thc_level(rotated[i], uniform[i], lo, delta, top));
    }
}

// v = float(level sum) * step + lo, two roundings
template <bool VEC>
__global__ __launch_bounds__(256) void thc_dequantize_kernel(const uint16_t *__restrict__ levels, float *__restrict__ out,
                                                             int64_t begin, int64_t n, const float *__restrict__ step_p,
                                                             const float *__restrict__ lo_p)
{
    const float step = *step_p, lo = *lo_p;
    if (VEC) {
        const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
        if (i + 4 > n) return;
        const uint2 l = *reinterpret_cast<const uint2 *>(levels + i);
        float4 o;
        float p0 = bf16_bits_to_f32(l.x & 0xffffu) * step, p1 = bf16_bits_to_f32(l.x >> 16) * step;
        float p2 = bf16_bits_to_f32(l.y & 0xffffu) * step, p3 = bf16_bits_to_f32(l.y >> 16) * step;
        o.x = p0 + lo; o.y = p1 + lo; o.z = p2 + lo; o.w = p3 + lo;
        stream_store(reinterpret_cast<float4 *>(out + i), o);
    } else {
        const int64_t i = begin + (int64_t)blockIdx.x * 256 + threadIdx.x;
        if (i >= n) return;
        const float prod = bf16_bits_to_f32(levels[i]) * step;
        out[i] = prod + lo;
    }
}

} // namespace

int64_t eden_work_doubles(int64_t n)
{
    const int64_t tiles = eden_tiles(n);
    return tiles <= kEdenFoldTiles ? 2 * tiles : tiles;
}

// Up to so many tiles the bins kernel has eight elements per thread, for twice the waves; beyond, the second table and fold per
// element is what counts.  Sixteen -> eight, us, 4 bits: 2^18 elements 5.2 -> 4.8, 2^20 5.6 -> 5.0 (8 bits 6.8 -> 5.7), 2^22
// 9.3 -> 9.2, 2^23 13.7 -> 13.4, 2^24 22.8 -> 23.4, 2^25 37.8 -> 42.5, 2^26 63.0 -> 72.9.
constexpr int64_t kFewTiles = 2048;

template <int MOST>
static hipError_t quantize_slices(const QuantizeSlice *slices, int count, const float *boundaries, const float *centroids, int nbits,
                                  hipStream_t stream)
{
    QuantizeSet<MOST> set;
    static_assert(MOST > 1 || sizeof(set) <= 128, "beyond, a launch takes 0.8 us longer (launch_with)");
    set.count = count;
    set.boundaries = boundaries;
    set.centroids = centroids;
    int64_t blocks = 0;
    bool have_sums = true;
    for (int k = 0; k < count; k++) have_sums = have_sums && slices[k].sums;
    for (int k = 0; k < count; k++) {
        set.s[k] = slices[k];
        set.s[k].sqrt_n = (float)sqrt((double)slices[k].n);
        if (!have_sums) {
            set.s[k].sums = slices[k].work;
            set.s[k].sum_count = eden_tiles(slices[k].n);
        }
        set.first[k] = (unsigned)blocks;
        blocks += eden_tiles(slices[k].n);
    }
    const bool fold = set.fold = count > 1 || set.s[0].sum_count <= kEdenFoldTiles;
    const bool few = fold && blocks <= kFewTiles;
    const dim3 grid((unsigned)blocks), block(kEdenThreads);
    hipError_t e = hipSuccess;
    if (!have_sums) e = launch_with(eden_sumsq_kernel<MOST>, grid, block, stream, set);
    if (e == hipSuccess && !fold) {
        hipLaunchKernelGGL(eden_norm_kernel, dim3(1), block, 0, stream, set.s[0].sums, set.s[0].sum_count, set.s[0].n, slices[0].result);
        e = hipGetLastError();
    }
    if (e != hipSuccess) return e;
#define DQ_EDEN_BINS(B)                                                                                       \
    do {                                                                                                      \
        if (few)                                                                                              \
            e = launch_with(eden_bins_kernel<B, true, 8, MOST>, grid, dim3(kEdenTile / 8), stream, set);      \
        else if (fold)                                                                                        \
            e = launch_with(eden_bins_kernel<B, true, 16, MOST>, grid, block, stream, set);                   \
        else if constexpr (MOST == 1)                                                                         \
            e = launch_with(eden_bins_kernel<B, false, 16, MOST>, grid, block, stream, set);                  \
    } while (0)
    switch (nbits) {
    case 1: DQ_EDEN_BINS(1); break;
    case 2: DQ_EDEN_BINS(2); break;
    case 3: DQ_EDEN_BINS(3); break;
    case 4: DQ_EDEN_BINS(4); break;
    case 5: DQ_EDEN_BINS(5); break;
    case 6: DQ_EDEN_BINS(6); break;
    case 7: DQ_EDEN_BINS(7); break;
    default: DQ_EDEN_BINS(8); break;
    }
#undef DQ_EDEN_BINS
    return e == hipSuccess ? launch_with(eden_scale_kernel<MOST>, dim3((unsigned)count), block, stream, set) : e;
}

// slices of at most kEdenFoldTiles tiles, or one of any length; bits of an NBITS-wide code for all of them
hipError_t launch_eden_quantize_slices(const QuantizeSlice *slices, int count, const float *boundaries, const float *centroids,
                                       int nbits, hipStream_t stream)
{
    return count == 1 ? quantize_slices<1>(slices, count, boundaries, centroids, nbits, stream)
                      : quantize_slices<kMaxEdenSlices>(slices, count, boundaries, centroids, nbits, stream);
}

hipError_t launch_eden_quantize(const float *vec, int64_t n, const float *boundaries, const float *centroids, int nbits,
                                uint32_t *packed, float *result, double *work, hipStream_t stream)
{
    const QuantizeSlice s{vec, n, packed, result, work};
    return launch_eden_quantize_slices(&s, 1, boundaries, centroids, nbits, stream);
}

} // namespace dq

// ---- EDEN quantise without any allocation ------------------------------------------------------
// The per-tile partial sums of launch_eden_quantize live in this array instead of a caller's buffer.
// Every device the library runs on holds its own copy for the life of the process (512 KiB).  The
// array's name is only a host-side handle: its device address comes from hipGetSymbolAddress, once
// per device, and that pointer is what the kernels receive.
static constexpr int64_t kEdenStaticMaxTiles = 65536; // 2^28 elements of 4096-element tiles
static __device__ __align__(256) double eden_static_scratch[kEdenStaticMaxTiles];

namespace dq {

int64_t eden_static_max_n() { return kEdenStaticMaxTiles * (int64_t)kEdenTile; }

namespace {
constexpr int kMaxDevices = 64;
std::mutex static_lock;
double *static_scratch_of[kMaxDevices]; // device address of eden_static_scratch, per device
} // namespace

// Resolves the address of the static array on `device` (which the caller has made current), once per device.  Called
// by the library's first call on a device, so that the entry point below has nothing left to look up when it runs
// (e.g. under stream capture).
hipError_t eden_static_prepare(int device)
{
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> g(static_lock);
    if (!static_scratch_of[device]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(eden_static_scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        static_scratch_of[device] = static_cast<double *>(p);
    }
    return hipSuccess;
}

hipError_t launch_eden_quantize_static(const float *vec, int64_t n, const float *boundaries, const float *centroids,
                                       int nbits, uint32_t *packed, float *result, int device, hipStream_t stream)
{
    if (eden_tiles(n) > kEdenStaticMaxTiles) return hipErrorInvalidValue;
    const hipError_t e = eden_static_prepare(device);
    if (e != hipSuccess) return e;
    double *scratch;
    {
        std::lock_guard<std::mutex> g(static_lock);
        scratch = static_scratch_of[device];
    }
    // every word of scratch that a kernel reads has been written by an earlier kernel of this same
    // call (sumsq -> norm or bins, bins -> scale), so nothing has to be cleared between calls; the array
    // holds the two regions of a short vector (2 * 1024 doubles) as it holds the one of a long vector
    return launch_eden_quantize(vec, n, boundaries, centroids, nbits, packed, result, scratch, stream);
}

hipError_t launch_eden_dequantize(const uint32_t *packed, int64_t n, const float *centroids, int nbits, float *out,
                                  hipStream_t stream)
{
    // n is a multiple of 32 and out 16-byte aligned: a thread's sixteen elements are half a word of every plane
    dim3 grid((unsigned)((n / 16 + 255) / 256)), block(256);
    switch (nbits) {
#define DQ_EDEN_CASE(B)                                                                                      \
    case B: hipLaunchKernelGGL(eden_dequantize_kernel<B>, grid, block, 0, stream, packed, n, centroids, out); break;
        DQ_EDEN_CASE(1) DQ_EDEN_CASE(2) DQ_EDEN_CASE(3) DQ_EDEN_CASE(4) DQ_EDEN_CASE(5) DQ_EDEN_CASE(6) DQ_EDEN_CASE(7)
    default: hipLaunchKernelGGL(eden_dequantize_kernel<8>, grid, block, 0, stream, packed, n, centroids, out); break;
#undef DQ_EDEN_CASE
    }
    return hipGetLastError();
}

hipError_t launch_thc_quantize(const float *rotated, const float *uniform, void *out, int64_t n, const float *lo,
                               const float *delta, int levels, hipStream_t stream)
{
    uint16_t *o = static_cast<uint16_t *>(out);
    const float top = (float)(levels - 1);
    const bool aligned = ((reinterpret_cast<uintptr_t>(rotated) | reinterpret_cast<uintptr_t>(uniform)) & 15) == 0 &&
                         (reinterpret_cast<uintptr_t>(out) & 7) == 0;
    int64_t done = 0;
    if (aligned && n >= 4) {
        done = n / 4 * 4;
        hipLaunchKernelGGL(thc_quantize_kernel<true>, dim3((unsigned)((done / 4 + 255) / 256)), dim3(256), 0, stream, rotated,
                           uniform, o, (int64_t)0, done, lo, delta, top);
    }
    if (done < n)
        hipLaunchKernelGGL(thc_quantize_kernel<false>, dim3((unsigned)((n - done + 255) / 256)), dim3(256), 0, stream, rotated,
                           uniform, o, done, n, lo, delta, top);
    return hipGetLastError();
}

hipError_t launch_thc_dequantize(const void *levels, float *out, int64_t n, const float *step, const float *lo,
                                 hipStream_t stream)
{
    const uint16_t *l = static_cast<const uint16_t *>(levels);
    const bool aligned = (reinterpret_cast<uintptr_t>(levels) & 7) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    int64_t done = 0;
    if (aligned && n >= 4) {
        done = n / 4 * 4;
        hipLaunchKernelGGL(thc_dequantize_kernel<true>, dim3((unsigned)((done / 4 + 255) / 256)), dim3(256), 0, stream, l, out,
                           (int64_t)0, done, step, lo);
    }
    if (done < n)
        hipLaunchKernelGGL(thc_dequantize_kernel<false>, dim3((unsigned)((n - done + 255) / 256)), dim3(256), 0, stream, l, out,
                           done, n, step, lo);
    return hipGetLastError();
}

// ---- the slices of EDEN's compress / decompress in one call ----------------------------------------------
//
// The reference (and the element-wise sequence this replaced) copies a slice to float32, copies it again or pads it, and
// writes the diagonal to memory before every rotation.  Here the first pass of the first rotation reads the caller's vector
// in its own type with the padding's zeros, the diagonal is drawn in the pass that applies it, and the last pass of the last
// inverse rotation multiplies by the scale and stores the caller's type.
//
// A launch costs about 3.4 us whatever it does, and a vector has up to five slices, each half as long as the one before or
// less: the time of a vector of less than a few million elements was its launches.  So the slices travel together:
//   up to 2^13 elements   one workgroup per slice does all of it, all slices in one launch (dq_eden_short.hip); 2^14 as well
//                         where no longer slice travels with the next kind's launches anyway
//   up to 2^22            one launch per pass for all slices: tiles, strided pass, bins, scale; tiles, strided pass
//   beyond                one after the other: their launches fill the GPU, and their diagonal is read from memory
// Slices that are not plain powers of one rotation (only a caller's own dictionary asks for that) go one by one as well.
// Both directions at 4 bits, fp32: 2^20 elements (one slice) 94 -> 38 -> 28-32 us, 20,000 (two) 165 -> 20, 115,387 (four) 364 -> 135 -> 43,
// 419,364 (three) 266 -> 115 -> 29, 6,000,000 (two) 186 -> 62: at first, (with one native call per slice,) now together.

namespace {

// Longer vectors read the diagonal from memory, one bit per element, written by a launch of its own (about 4 us): drawing it
// costs 25 instruction slots per element, 2.7 us at 2^22 elements.
constexpr int64_t kEdenDrawnSigns = (int64_t)1 << 22;

// no rotation at all, which a slice of the C call may ask for (Eden's own have one or two): the slice padded and converted /
// scaled and converted
__global__ __launch_bounds__(256) void eden_pad_kernel(const void *__restrict__ src, int dtype, int64_t count, int64_t n,
                                                       float *__restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float v = 0.0f;
    if (i < count)
        v = dtype == DQ_F32 ? ElemIO<DQ_F32>::load(src, i) : (dtype == DQ_BF16 ? ElemIO<DQ_BF16>::load(src, i) : ElemIO<DQ_F16>::load(src, i));
    out[i] = v;
}

// out = T(scale * vec), elements below count
__global__ __launch_bounds__(256) void eden_finish_kernel(const float *__restrict__ vec, const float *__restrict__ scale,
                                                          void *__restrict__ out, int dtype, int64_t count)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    const float v = *scale * vec[i];
    if (dtype == DQ_F32)
        ElemIO<DQ_F32>::store(out, i, v);
    else if (dtype == DQ_BF16)
        ElemIO<DQ_BF16>::store(out, i, v);
    else
        ElemIO<DQ_F16>::store(out, i, v);
}

struct SliceScratch {
    float *vec;
    double *work;
    uint32_t *signs;
    // the last pass's sums of squares take the place of the signs, which the first pass has read: n / 64 doubles' room, at
    // most one for every 512 elements
    double *sums() const { return reinterpret_cast<double *>(signs); }
};

int64_t round_up(int64_t v) { return (v + 255) & ~(int64_t)255; }

// (short slices need none; their share is taken all the same, it is small)
SliceScratch slice_scratch(char *c, int64_t n)
{
    SliceScratch s;
    s.vec = reinterpret_cast<float *>(c);
    s.work = reinterpret_cast<double *>(c + round_up(4 * n));
    s.signs = reinterpret_cast<uint32_t *>(c + round_up(4 * n) + round_up(8 * eden_work_doubles(n)));
    return s;
}

float inv_sqrt_of(int64_t n) { return 1.0f / (float)sqrt((double)n); } // as torch divides by a host scalar on the device

// one rotation of a slice of at least 1024 elements
hipError_t rotate(const SliceScratch &s, int64_t n, int64_t seed, int inverse, TransformEnds ends, hipStream_t stream)
{
    const void *sign = nullptr;
    if (n <= kEdenDrawnSigns) {
        ends.gen = sign_seed(n, seed);
    } else {
        const hipError_t e = launch_rand_diag_bits(s.signs, n, seed, stream);
        if (e != hipSuccess) return e;
        sign = s.signs;
    }
    return launch_rht_ends(s.vec, sign, sign != nullptr, n, n, inv_sqrt_of(n), inverse, ends, stream);
}

TransformEnds compress_ends(const dq_eden_slice_t &s, int dtype)
{
    TransformEnds ends;
    ends.in_src = s.vec;
    ends.in_dtype = dtype;
    ends.in_count = s.count;
    return ends;
}

// the first (planes) and last (destination) ends of an inverse
TransformEnds decompress_ends(const dq_eden_slice_t &s, int dtype, bool planes, bool destination)
{
    TransformEnds ends;
    if (planes) {
        ends.in_planes = s.packed;
        ends.in_centroids = s.centroids;
        ends.in_nbits = s.nbits;
    }
    if (destination) {
        ends.post_scale = s.result;
        ends.out_dst = s.vec;
        ends.out_dtype = dtype;
        ends.out_count = s.count;
    }
    return ends;
}

// a slice by itself, n > kEdenShort / 2
hipError_t compress_one(const dq_eden_slice_t &x, int dtype, const SliceScratch &s, hipStream_t stream)
{
    hipError_t e = hipSuccess;
    if (x.rotations == 0) {
        hipLaunchKernelGGL(eden_pad_kernel, dim3((unsigned)((x.n + 255) / 256)), dim3(256), 0, stream, x.vec, dtype, x.count, x.n, s.vec);
        e = hipGetLastError();
    }
    QuantizeSlice q{s.vec, x.n, x.packed, x.result, s.work};
    for (int i = 0; e == hipSuccess && i < x.rotations; i++) {
        TransformEnds ends = i == 0 ? compress_ends(x, dtype) : TransformEnds();
        if (i == x.rotations - 1) {
            q.sum_count = rht_sum_count(x.n);
            if (q.sum_count) q.sums = ends.sums = s.sums();
        }
        e = rotate(s, x.n, x.seed + i, 0, ends, stream);
    }
    return e == hipSuccess ? launch_eden_quantize_slices(&q, 1, x.boundaries, x.centroids, x.nbits, stream) : e;
}

hipError_t decompress_one(const dq_eden_slice_t &x, int dtype, const SliceScratch &s, hipStream_t stream)
{
    hipError_t e = hipSuccess;
    if (x.rotations == 0) {
        e = launch_eden_dequantize(x.packed, x.n, x.centroids, x.nbits, s.vec, stream);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(eden_finish_kernel, dim3((unsigned)((x.count + 255) / 256)), dim3(256), 0, stream, s.vec, x.result, x.vec, dtype, x.count);
        return hipGetLastError();
    }
    for (int i = 0; e == hipSuccess && i < x.rotations; i++)
        e = rotate(s, x.n, x.seed + x.rotations - 1 - i, 1, decompress_ends(x, dtype, i == 0, i == x.rotations - 1), stream);
    return e;
}

bool travels_together(const dq_eden_slice_t &x) { return x.n <= kEdenDrawnSigns && x.rotations == 1; }

// the slices of one kind, kMaxEdenSlices at a time
template <class Mine, class Launch>
hipError_t in_groups(const dq_eden_slice_t *slices, char *const *scratch, int count, Mine mine, Launch launch)
{
    dq_eden_slice_t group[kMaxEdenSlices];
    SliceScratch room[kMaxEdenSlices];
    int have = 0;
    for (int k = 0; k <= count; k++) {
        if (k < count && mine(slices[k])) {
            group[have] = slices[k];
            room[have++] = slice_scratch(scratch[k], slices[k].n);
        }
        if (have == kMaxEdenSlices || (k == count && have > 0)) {
            const hipError_t e = launch(group, room, have);
            if (e != hipSuccess) return e;
            have = 0;
        }
    }
    return hipSuccess;
}

} // namespace

int64_t eden_slice_bytes(int64_t n) { return round_up(4 * n) + round_up(8 * eden_work_doubles(n)) + round_up(n / 8); }

// compress: slices share nbits, boundaries and centroids
hipError_t launch_eden_slices(const dq_eden_slice_t *slices, int count, int dtype, bool decompress, void *scratch, hipStream_t stream)
{
    std::vector<char *> at(count);
    char *c = static_cast<char *>(scratch);
    for (int k = 0; k < count; k++) {
        at[k] = c;
        c += eden_slice_bytes(slices[k].n);
    }
    bool longer = false;
    for (int k = 0; k < count; k++) longer = longer || (slices[k].n > kEdenShort && travels_together(slices[k]));
    const auto is_short = [longer](const dq_eden_slice_t &x) { return x.n <= (longer ? kEdenShort / 2 : kEdenShort); };
    hipError_t e = in_groups(slices, at.data(), count, [&](const dq_eden_slice_t &x) { return !is_short(x) && travels_together(x); },
                             [&](const dq_eden_slice_t *group, const SliceScratch *room, int have) {
        TransformSlice t[kMaxEdenSlices];
        QuantizeSlice q[kMaxEdenSlices];
        for (int k = 0; k < have; k++) {
            t[k].x = room[k].vec;
            t[k].n = group[k].n;
            t[k].scale = inv_sqrt_of(group[k].n);
            t[k].ends = decompress ? decompress_ends(group[k], dtype, true, true) : compress_ends(group[k], dtype);
            t[k].ends.gen = sign_seed(group[k].n, group[k].seed);
            if (!decompress) t[k].ends.sums = room[k].sums();
        }
        const hipError_t r = launch_rht_slices(t, have, decompress ? 1 : 0, stream);
        if (r != hipSuccess || decompress) return r;
        for (int k = 0; k < have; k++)
            q[k] = QuantizeSlice{room[k].vec, group[k].n, group[k].packed, group[k].result, room[k].work, room[k].sums(), t[k].sum_count};
        return launch_eden_quantize_slices(q, have, group[0].boundaries, group[0].centroids, group[0].nbits, stream);
    });
    if (e == hipSuccess)
        e = in_groups(slices, at.data(), count, is_short,
                      [&](const dq_eden_slice_t *group, const SliceScratch *, int have) {
            return decompress ? launch_eden_short_decompress(group, have, dtype, stream) : launch_eden_short_compress(group, have, dtype, stream);
        });
    for (int k = 0; e == hipSuccess && k < count; k++) {
        if (is_short(slices[k]) || travels_together(slices[k])) continue;
        const SliceScratch s = slice_scratch(at[k], slices[k].n);
        e = decompress ? decompress_one(slices[k], dtype, s, stream) : compress_one(slices[k], dtype, s, stream);
    }
    return e;
}

} // namespace dq
