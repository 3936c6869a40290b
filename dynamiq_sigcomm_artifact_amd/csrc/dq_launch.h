// Host-side launcher declarations shared by the translation units of
// libdynamiq_eden.so.  Each launcher enqueues on `stream` and returns the
// launch status; argument validation happens in the C ABI layer (dq_api.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "dq_device.cuh"

namespace dq {

// A kernel whose only argument is `args`.  Short calls wait for the host, and the runtime copies a kernel's arguments one by one to
// where the GPU reads them: a decoder call of eight arguments and 104 bytes takes 3.8 us, with one argument of 56 bytes 2.9 (and 576
// bytes 1.1 us more than 64).  In a stream, not in a graph, the GPU takes 0.7 us longer where they are more than 128 bytes.  The host's
// part of an eight-rank ring of 65,792 elements, 17 calls, 68 -> 55 us.
template <class K, class A> inline hipError_t launch_with(K *kernel, dim3 grid, dim3 block, hipStream_t stream, const A &args, size_t lds = 0)
{
    static_assert(std::is_same<K, void(A)>::value, "the kernel takes these arguments");
    void *list[] = {const_cast<A *>(&args)};
    const hipError_t e = hipLaunchKernel(reinterpret_cast<const void *>(kernel), grid, block, list, lds, stream);
    if (e != hipSuccess) (void)hipGetLastError();
    return e;
}

// scaling quantisation, catch-all kernels (dq_scaling_generic.hip)
hipError_t launch_generic_compress(const void *src, uint8_t *dst, const void *rnd, int64_t n,
                                   int nbits, int C, int dtype, int strategy, const MeeParams &mp,
                                   hipStream_t stream);
hipError_t launch_generic_decompress(const uint8_t *src, void *dst, int64_t n, int nbits, int C,
                                     int dtype, int strategy, const MeeParams &mp, int add,
                                     hipStream_t stream);

// the same without a row list, for vectors of few superchunks (dq_scaling_hier16_short.hip); recv != null: the fused ring step
hipError_t launch_hier16_short_compress(const void *src, const uint8_t *recv, uint8_t *dst, const void *rnd, int64_t nsc, int nbits,
                                        int dtype, bool mee, const MeeParams &mp, const RandKey *philox, hipStream_t stream);
hipError_t launch_hier16_short_decompress(const uint8_t *src, void *dst, int64_t nsc, int nbits, int dtype, bool mee, const MeeParams &mp,
                                          hipStream_t stream);

// scaling quantisation, vectorised chunk-16 hierarchical kernels
// (dq_scaling_hier16.hip); dtype BF16 or F32, element pointers 16-byte aligned
hipError_t launch_hier16_compress(const void *src, uint8_t *dst, const void *rnd, int64_t n,
                                  int nbits, int dtype, bool mee, const MeeParams &mp,
                                  hipStream_t stream);
hipError_t launch_hier16_decompress(const uint8_t *src, void *dst, int64_t n, int nbits, int dtype,
                                    bool mee, const MeeParams &mp, int add, hipStream_t stream);
// compress (recv == null) or the fused ring step with the uniform values drawn in the kernel
hipError_t launch_hier16_compress_philox(const void *src, const uint8_t *recv, uint8_t *dst, int64_t n,
                                         int nbits, int dtype, bool mee, const MeeParams &mp,
                                         uint64_t seed, uint64_t step, hipStream_t stream);
hipError_t launch_hier16_dec_comp(const uint8_t *recv, const void *inp, uint8_t *send,
                                  const void *rnd, int64_t n, int nbits, int dtype, bool mee,
                                  const MeeParams &mp, hipStream_t stream);

// vectorised chunk-16 kernels for the remaining shapes (dq_scaling_tile16.hip): binary16 elements
// with any strategy, bf16 / fp32 elements with the flat strategies 0 / 1
hipError_t launch_tile16_compress(const void *src, uint8_t *dst, const void *rnd, int64_t n, int nbits,
                                  int dtype, int strategy, const MeeParams &mp, hipStream_t stream,
                                  const RandKey *philox = nullptr);
// the in-kernel random stream (dq_device.cuh: chunk_uniform_words) written out as a tensor
hipError_t launch_philox_uniform(void *out, int64_t n, int dtype, uint64_t seed, uint64_t step,
                                 hipStream_t stream);
hipError_t launch_tile16_decompress(const uint8_t *src, void *dst, int64_t n, int nbits, int dtype,
                                    int strategy, const MeeParams &mp, int add, hipStream_t stream);

// the same kernels over a list of superchunk indices: record k <-> superchunk rows[k] of the
// element buffer; recv != null makes compress the fused decode-accumulate-recompress step;
// stats != null adds the destination superchunk's mean after decoding; elements >= limit are
// not written
hipError_t launch_hier16_compress_rows(const void *src, const uint8_t *recv, const int32_t *rows,
                                       uint8_t *dst, const void *rnd, int64_t nrows, int nbits,
                                       int dtype, bool mee, const MeeParams &mp, hipStream_t stream);
hipError_t launch_hier16_decompress_rows(const uint8_t *src, void *dst, const int32_t *rows,
                                         const void *stats, int64_t limit, int64_t nrows, int nbits,
                                         int dtype, bool mee, const MeeParams &mp, int add,
                                         hipStream_t stream);

// stable partition of superchunk indices by bit width (dq_grouping.hip)
int64_t group_plan_work_ints(int64_t nsc);
hipError_t launch_group_plan(const int64_t *qbits, int64_t nsc, int32_t *order, int32_t *work,
                             hipStream_t stream);
// the same with the widths computed from the norm column of the bf16 stats and the offset u
// fixed-proportion groups (stable descending sort of the bf16 norms); nsc <= 65535, stats 4-byte aligned
hipError_t launch_group_plan_sorted(const void *stats, int64_t nsc, int64_t top, int64_t bottom, int64_t *qbits_out,
                                    int32_t *order, int32_t *work, hipStream_t stream);
int64_t group_plan_sorted_large_work_ints(int64_t nsc);
hipError_t launch_group_plan_sorted_large(const void *stats, int64_t nsc, int64_t top, int64_t bottom, int64_t *qbits_out,
                                          int32_t *order, int32_t *work, int64_t work_ints, hipStream_t stream);
hipError_t launch_group_plan_stats(const void *stats, float u, const double *u_dev, int64_t nsc, int64_t *qbits_out,
                                   int32_t *order, int32_t *work, uint32_t *hist, hipStream_t stream);

// the offset u of the bit-width rule from a histogram of the norm patterns (dq_bitrate.hip)
int64_t bitrate_hist_ints();
hipError_t launch_norm_histogram(const void *stats, int64_t nsc, uint32_t *hist, hipStream_t stream);
hipError_t launch_bitrate_search(uint32_t *hist, int mode, double prev_u, const double *prev_u_dev, double target, double *out,
                                 hipStream_t stream);

// all bit-width groups of a planned bucket in one launch (dq_scaling_mixed.hip); mp: the MEE
// parameters of 8, 4 and 2 bits in this order; step_dev (nullable, device memory): a value the kernel adds to
// philox->step when it runs, so that a recorded launch can draw fresh rounding randomness on every replay
int64_t mixed_stream_bytes(int64_t nsc, int world);
hipError_t launch_mixed_compress(const void *src, const float *center_mean, int center_world, int64_t n_valid,
                                 const int32_t *order, const int32_t *counts, int ring_chunk, int ring_world,
                                 const uint8_t *recv, uint8_t *dst, const void *rnd, const RandKey *philox,
                                 int64_t nsc, int dtype, bool mee, const MeeParams *mp, hipStream_t stream,
                                 const uint64_t *step_dev = nullptr);
hipError_t launch_mixed_decompress(const uint8_t *src, void *dst, const int32_t *order, const int32_t *counts,
                                   int ring_chunk, int ring_world, const void *stats, int64_t limit, int64_t nsc,
                                   int dtype, bool mee, const MeeParams *mp, hipStream_t stream);

// the all-reduce of buckets whose ranks share this GPU's memory, without a packed stream (dq_single_pass.hip)
constexpr int kMaxBuckets = 32;   // per launch of the one-rank kernel (their descriptors are kernel arguments)
constexpr int kMaxRanks = 16;     // simulated ranks, likewise
constexpr int kMaxPoolRanks = 8;  // simulated ranks with random pools: three tables of ranks x steps travel with the launch
typedef dq_roundtrip_t RoundtripDesc;
// *step_dev + step_more is added to every bucket's step, and *step_dev left there, when step_dev is set
hipError_t launch_roundtrip(const RoundtripDesc *desc, int count, int world, float u, const double *u_dev, uint64_t seed,
                            uint64_t *step_dev, uint64_t step_more, uint32_t *hist, int dtype, bool mee, const MeeParams *mp,
                            hipStream_t stream);
// total: bf16 pairs [nsc], mean: float [world][nsc]; tile_widths (may be null): a word per four superchunks, how many of them u
// (or *u_dev) gives 8 bits, and 4 bits in the upper half (added up as words: at most 65,535 superchunks, see ring_plans_itself)
hipError_t launch_ranks_stats(const void *const *src, int world, int64_t n, void *total, float *mean, int dtype,
                              uint32_t *tile_widths, float u, const double *u_dev, hipStream_t stream);
// a ring that finds its groups from the words of launch_ranks_stats (in the place of a plan and its lists)
bool ring_plans_itself(int64_t n, int world, int dtype);
struct RingDesc {
    const void *const *src;
    void *const *out;
    int world;
    int64_t n;
    const void *total;
    const float *mean;
    const int32_t *order, *counts;
    uint64_t seed;                               // rank r draws from seed + r, step s of the ring from step s
    const uint32_t *tile_widths;                     // null, or what launch_ranks_stats left there: the ring does without order
    int32_t *work;                               // (with tile_widths) and writes the group sizes to work[0..3]
    float u;
    const double *u_dev;
    bool pooled;                                 // or the random values come from pools:
    const void *pool[3][kMaxPoolRanks];          // by width (8, 4, 2 bits) and rank
    int32_t first[3][kMaxPoolRanks][kMaxPoolRanks]; // first row of 16 values, by width, rank and step
};
hipError_t launch_ring(const RingDesc &d, int dtype, bool mee, const MeeParams *mp, hipStream_t stream);
int host_width_threshold(float u, int target);

// superchunk mean-centring (dq_superchunk.hip)
// residual == nullptr: statistics only; mean_out (nullable) receives the binary32 means
hipError_t launch_mean_center(const void *src, void *residual, void *stats, float *mean_out, int64_t n,
                              int world_size, int dtype, hipStream_t stream);
hipError_t launch_add_mean_copy(const void *residual, void *dst, const void *stats, int64_t n,
                                int dtype, hipStream_t stream);

// Walsh-Hadamard (dq_hadamard.hip)
struct TransformEnds;
hipError_t launch_hadamard(float *vec, int64_t n, hipStream_t stream);
// sign: float +-1 values, or (sign_packed) the bit vector of launch_pack_signs; may be null
hipError_t launch_rht_blocked(float *vec, const void *sign, bool sign_packed, int64_t n, int64_t block, float scale,
                              int inverse, hipStream_t stream);
// EDEN's dequantiser folded into the first pass of the inverse transform, EDEN's scale (device scalar, may be null)
// into the last
hipError_t launch_eden_dequantize_irht(const uint32_t *packed, const float *centroids, int nbits, const void *sign,
                                       bool sign_packed, float *out, int64_t n, int64_t block, float scale,
                                       const float *post_scale, hipStream_t stream);
// rht_blocked with quantisers, a source or a destination of another type at its ends; x (fp32 [n], 16-byte aligned) is
// where the passes meet and where the result goes unless ends.out_* say otherwise; n a multiple of 1024, block >= 1024
hipError_t launch_rht_ends(float *x, const void *sign, bool sign_packed, int64_t n, int64_t block, float scale, int inverse,
                           const TransformEnds &ends, hipStream_t stream);
hipError_t launch_rand_diag(float *out, int64_t size, int64_t seed, hipStream_t stream);
// the same diagonal as packed bits (set where the value is -1); size a multiple of 256
hipError_t launch_rand_diag_bits(uint32_t *bits, int64_t size, int64_t seed, hipStream_t stream);
// THC's quantiser folded into the last pass of the forward transform / the first pass of the inverse one
hipError_t launch_thc_rht_quantize(float *vec, const void *sign, bool sign_packed, const float *uniform, void *levels_out,
                                   int64_t n, int64_t block, float scale, const float *lo, const float *delta, int levels,
                                   hipStream_t stream);
hipError_t launch_thc_dequantize_irht(const void *levels_in, const void *sign, bool sign_packed, float *out, int64_t n,
                                      int64_t block, float scale, const float *step, const float *lo, hipStream_t stream);

// blocked randomized Hadamard transform fused with the hierarchical chunk-16 quantiser (dq_rht_scaling_impl.cuh and the translation units that include it);
// rand_kind: DQ_F32 or DQ_BF16 pool, or 3 for the in-kernel stream (rnd ignored)
hipError_t launch_pack_signs(const float *sign, uint32_t *bits, int64_t n, hipStream_t stream);
// sign: fp32 +-1 values, or with sign_bits one bit per element (launch_pack_signs); may be null
hipError_t launch_rht_compress(const float *src, const void *sign, int sign_bits, uint8_t *dst, const void *rnd, int rand_kind,
                               int64_t n, int64_t block, float scale, int nbits, bool mee, const MeeParams &mp,
                               uint64_t seed, uint64_t step, hipStream_t stream);
hipError_t launch_rht_compress_mfma16(const float *src, const void *sign, int sign_bits, uint8_t *dst, int64_t n, int64_t block,
                                      float scale, const MeeParams &mp, uint64_t seed, uint64_t step, hipStream_t stream);
hipError_t launch_irht_decompress(const uint8_t *src, const void *sign, int sign_bits, float *dst, int64_t n, int64_t block,
                                  float scale, int nbits, bool mee, const MeeParams &mp, hipStream_t stream);
// THC's grid (thc_hooks.py:143-147) where it is not a pair of device scalars: numbers from the host, or worked out from the
// norm on the device with the operations of torch's float32 scalars in their order -- top = (t * norm) * inv_sqrt, lowest
// level -top, spacing ((top + top) * inv_levels) + 1e-23, step of an aggregate spacing * inv_clients, the inv_* being
// float32 reciprocals of host numbers
struct ThcGrid {
    enum { POINTERS, HOST, NORM };
    int kind = POINTERS;
    float lo = 0.0f, spacing = 0.0f, step = 0.0f;
    const float *norm = nullptr;
    float t = 0.0f, inv_sqrt = 0.0f, inv_levels = 0.0f, inv_clients = 0.0f;
};
// the diagonal of rand_diag(size, seed), drawn where it is applied; size = 8 * 2^bits >= 1024
struct SignSeed {
    int bits = 0; // 0: none
    uint32_t ss = 0;
};
SignSeed sign_seed(int64_t size, int64_t seed);

// Uniform values drawn where they are compared (dq_uniform_stream_t); bits: log2 of the stream's threads, negative: none
constexpr int64_t kDrawsFrom = (int64_t)1 << 19, kDrawsTo = (int64_t)1 << 25; // transforms that may
struct UniformDraw {
    int bits = -1;
    uint64_t seed = 0, counter = 0;
};

// Quantisers folded into the two ends of a transform (all null: the plain transform).  `in_*` replace the load of the
// first pass, `out_*` / `post_scale` act on the store of the last one.
// What a first pass looks at, and what a strided one does: a kernel gets the one or the other (FirstPass and StridedPass of
// dq_rht_scaling_impl.cuh).
struct InEnds {
    // the first pass loads in_count elements of in_dtype from in_src, zeros behind them, instead of x
    const void *in_src = nullptr;
    int in_dtype = 0;
    int64_t in_count = 0;
    // THC: the pass loads float(level) * *in_step + *in_lo instead of x
    const uint16_t *in_levels = nullptr;
    const float *in_step = nullptr, *in_lo = nullptr;
    // EDEN: the pass loads centroids[bin] from the bit planes of the bins
    const uint32_t *in_planes = nullptr;
    const float *in_centroids = nullptr;
    int in_nbits = 0;
    bool plain_in() const { return !in_src && !in_levels && !in_planes; }
};
struct OutEnds {
    // a strided pass over the whole vector that draws THC's uniform values finds zeros from here on and does not read them (a
    // multiple of its row stride; negative: it reads everything)
    int64_t zeros_from = -1;
    // the last pass stores its first out_count elements as out_dtype to out_dst, and nothing to x
    void *out_dst = nullptr;
    int out_dtype = 0;
    int64_t out_count = 0;
    // THC: the pass stores thc_level(value, uniform) as bf16 instead of the value
    uint16_t *out_levels = nullptr;
    const float *uniform = nullptr, *out_lo = nullptr, *out_delta = nullptr;
    float out_top = 0.0f;
    UniformDraw draw; // instead of uniform: transforms of 2^19 .. 2^25 elements
    // EDEN: the last pass multiplies by *post_scale
    const float *post_scale = nullptr;
    // EDEN: a strided last pass over the whole vector also leaves, in double, the sum of the squares of the values that its
    // workgroup w stores in sums[w] (rht_sum_count of them, in the order of dq_sums.cuh)
    double *sums = nullptr;
    bool plain_out() const { return !out_dst && !out_levels && !post_scale && !sums; }
};
struct TransformEnds : InEnds, OutEnds {
    // THC with the grid worked out in the kernels instead of in_step / in_lo / out_lo / out_delta
    ThcGrid grid;
    // the diagonal drawn in the kernels instead of a sign vector
    SignSeed gen;
    bool plain() const { return plain_in() && plain_out() && gen.bits == 0; }
};
// workgroups of the last pass of a whole-vector transform by launch_rht_ends; 0: that pass knows no sums
int64_t rht_sum_count(int64_t n);

hipError_t launch_rht_tile(float *x, const void *sign, int sign_bits, int64_t n, int kt, int kb, float scale, int apply_scale,
                           int sign_mode, int vec, const TransformEnds &ends, hipStream_t stream);
hipError_t launch_rht_strided(float *x, const void *sign, int sign_bits, int64_t n, int rbits, int sbits, float scale,
                              int apply_scale, int sign_mode, int vec, const TransformEnds &ends, hipStream_t stream);

// whole-vector transforms of 2^14 to 2^22 elements, at most kMaxEdenSlices of them, in one launch per pass; scale and the
// diagonal of ends.gen as in launch_rht_ends
constexpr int kMaxEdenSlices = 8;
struct TransformSlice {
    float *x;
    int64_t n;
    float scale;
    TransformEnds ends;
    int64_t sum_count = 0; // set by the call: how many of ends.sums it leaves
};
hipError_t launch_rht_slices(TransformSlice *slices, int count, int inverse, hipStream_t stream);
// the two launches behind it: pass k owns the workgroups from `first` on
struct TilePass {
    float *x;
    int64_t n;
    float scale;
    int kt, kb;          // tile pass: tile bits, stages [0, kb)
    int rbits, sbits;    // strided pass: stages [sbits, sbits + rbits)
    int sign_mode, apply_scale;
    unsigned first;
    TransformEnds ends;
};
hipError_t launch_rht_tile_passes(const TilePass *passes, int count, hipStream_t stream);
hipError_t launch_rht_strided_passes(const TilePass *passes, int count, hipStream_t stream);

// EDEN Lloyd-Max quantiser + packer, THC uniform quantiser (dq_eden.hip)
struct QuantizeSlice {
    const float *vec;
    int64_t n;
    uint32_t *packed;
    float *result;
    double *work;
    double *sums = nullptr; // partial sums of the squares, if some pass has left them already
    int64_t sum_count = 0;
    float sqrt_n = 0.0f;
};
int64_t eden_work_doubles(int64_t n);
hipError_t launch_eden_quantize(const float *vec, int64_t n, const float *boundaries, const float *centroids,
                                int nbits, uint32_t *packed, float *result, double *work,
                                hipStream_t stream);
// *overlap = 1 when kernels enqueued on a and b run side by side, 0 when the two streams take turns (they share a
// hardware queue, or are the same stream).  Synchronises with both streams: a set-up call, not for stream capture.
hipError_t probe_streams_overlap(hipStream_t a, hipStream_t b, int *overlap);
// `stream` waits for the work enqueued on `after` so far (pooled event, no allocation after the first 64 calls per device)
hipError_t stream_order_after(hipStream_t stream, hipStream_t after, int device);
// a kernel with the access pattern of the chunk-16 codec on `tiles` tiles and no arithmetic (dq_io_floor.hip); direction 0
// reads a and b and writes run, direction 1 reads run (and b) and writes a
bool tile_io_floor_shape_ok(int a_bytes, int b_bytes, int run_bytes);
hipError_t launch_tile_io_floor(int direction, void *a, int a_bytes, const void *b, int b_bytes, void *run, int run_bytes, int64_t tiles,
                                hipStream_t stream);

// the same launches with the partial sums in the library's own static device array (no allocation anywhere);
// `device` must be current
int64_t eden_static_max_n();
hipError_t eden_static_prepare(int device);
hipError_t launch_eden_quantize_static(const float *vec, int64_t n, const float *boundaries, const float *centroids,
                                       int nbits, uint32_t *packed, float *result, int device,
                                       hipStream_t stream);
hipError_t launch_eden_dequantize(const uint32_t *packed, int64_t n, const float *centroids, int nbits,
                                  float *out, hipStream_t stream);
// the slices of EDEN's compress / decompress (srrcomp.py:293-361); scratch: eden_slice_bytes of every slice, one after the
// other, 256-byte aligned.  compress: all slices of the same nbits, boundaries and centroids
int64_t eden_slice_bytes(int64_t n);
hipError_t launch_eden_slices(const dq_eden_slice_t *slices, int count, int dtype, bool decompress, void *scratch, hipStream_t stream);
// slices of at most kEdenShort elements, at most kMaxEdenSlices of them, one workgroup each (dq_eden_short.hip)
constexpr int kEdenShort = 1 << 14;
hipError_t launch_eden_short_compress(const dq_eden_slice_t *slices, int count, int dtype, hipStream_t stream);
hipError_t launch_eden_short_decompress(const dq_eden_slice_t *slices, int count, int dtype, hipStream_t stream);
hipError_t launch_thc_quantize(const float *rotated, const float *uniform, void *out, int64_t n,
                               const float *lo, const float *delta, int levels, hipStream_t stream);
hipError_t launch_thc_dequantize(const void *levels, float *out, int64_t n, const float *step,
                                 const float *lo, hipStream_t stream);

// EDEN bit-plane packing and THC rounding (dq_packing.hip)
hipError_t launch_bins_to_bits(const int32_t *bins, int64_t nbins, uint32_t *arr, int nbits,
                               hipStream_t stream);
hipError_t launch_bits_to_bins(int32_t *bins, int64_t nbins, const uint32_t *arr, int nbits,
                               hipStream_t stream);
hipError_t launch_quantization(float *vec, int64_t n, float div_factor, float tensor_max,
                               uint64_t seed, hipStream_t stream);

} // namespace dq
