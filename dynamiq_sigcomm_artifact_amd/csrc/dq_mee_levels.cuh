// The MEE level tables (csrc/cuda_hadamard.cu:873-899), worked out by the compiler: they hold for every call, so they lie in the code
// object's constant data, where the second launch finds them in the L2.  As kernel arguments, 512 bytes for 8 bits, the host wrote them
// anew for every launch (1.1 us of it) and the GPU fetched them from there: compress, ring step and decompress of 65,536 bf16 elements at 8 bits
// 13.0 -> 9.7 us, of 2^20 fp32 14.2 -> 11.4; 2^28 at 4 bits unchanged.
#pragma once

#include <stdint.h>

#include "dq_device.cuh"

namespace dq {

constexpr float mee_eps(int nbits) { return nbits <= 2 ? 0.23f : (nbits <= 5 ? 0.18f : 0.1f); }

// the nearest binary16, for normal numbers of it
constexpr uint16_t normal_f16_bits(float f)
{
    const uint32_t u = __builtin_bit_cast(uint32_t, f), a = u & 0x7fffffffu;
    return (uint16_t)(((u >> 16) & 0x8000u) | ((a + 0xfffu + ((a >> 13) & 1u) - 0x38000000u) >> 13));
}

// binary16 levels of the codes 0 .. 2^nbits - 1 (the last one, which no code has, is 0); binary32 arithmetic, one rounding per operation
constexpr void mee_fill(uint16_t *levels, int nbits)
{
    const float eps = mee_eps(nbits);
    const float two_eps = 2.0f * eps;
    const float two_eps2 = two_eps * eps;
    const float base = 1.0f + two_eps2;
    const float eps2 = eps * eps;
    const float one_plus_eps2 = 1.0f + eps2;
    const int anchor = (1 << (nbits - 1)) - 1;
    for (int k = 0; k < 1 << nbits; k++) levels[k] = 0;
    float power = 1.0f;
    for (int j = 1; j <= anchor; j++) {
        power = power * base;
        const float num = power - 1.0f;
        const float quo = num / two_eps2;
        const float rep = quo * one_plus_eps2;
        levels[anchor + j] = normal_f16_bits(rep);
        levels[anchor - j] = normal_f16_bits(-rep);
    }
}

template <int NBITS> struct MeeLevels {
    alignas(4) uint16_t at[1 << NBITS];
    constexpr MeeLevels() : at() { mee_fill(at, NBITS); }
};
template <int NBITS> __device__ constexpr MeeLevels<NBITS> kMeeLevels;

// the tables of 8, 4 and 2 bits end to end
constexpr int kLevels[3] = {0, 256, 272}; // where each width's begins
constexpr int kLevelCount = 276;
struct MeeLevelsOfWidths {
    alignas(4) uint16_t at[kLevelCount];
    constexpr MeeLevelsOfWidths() : at()
    {
        mee_fill(at + kLevels[0], 8);
        mee_fill(at + kLevels[1], 4);
        mee_fill(at + kLevels[2], 2);
    }
};
__device__ constexpr MeeLevelsOfWidths kMeeLevelsOfWidths;

} // namespace dq
