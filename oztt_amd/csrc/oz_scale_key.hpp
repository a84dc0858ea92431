// The 32-bit key of an element's magnitude that the normalization reduces (the BF16 code of |x|, see
// oz_scale.hip), and the delta and range flags of a maximum's key.
#pragma once
#include "oz_internal.hpp"

namespace {

constexpr uint32_t KEY_NAN = 0xFFFFFFFFu;  // Inf/NaN: dominates every other key
constexpr uint32_t KEY_TINY = 1u;          // nonzero maximum below 2^-126 (loses to any normal value)

// Key of |x| for the rounding mode (the BF16 code for normal in-range magnitudes; 0x7F80 above range).
// Branch-free: the in-range code is computed for every input, then the special cases replace it in
// increasing priority (above range, below range, Inf/NaN), so a wave never splits over its elements.
template <int CEIL>
__device__ __forceinline__ uint32_t bf16_key(double x) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(x);
    const uint32_t h = (uint32_t)(u >> 32) & 0x7FFFFFFFu, l = (uint32_t)u;
    const int32_t E = (int32_t)(h >> 20);
    const int32_t e8 = E - 896;
    uint32_t v = ((uint32_t)e8 << 7) | ((h >> 13) & 0x7Fu);
    const bool dropped = (h & 0x1FFFu) || l;
    if (CEIL == 1) v += dropped ? 1u : 0u;
    if (CEIL == 2) v += (dropped || !(v & 0x7Fu)) ? 1u : 0u;
    v = e8 >= 255 ? 0x7F80u : v;
    v = e8 <= 0 ? ((h | l) ? KEY_TINY : 0u) : v;
    return E == 0x7FF ? KEY_NAN : v;
}

// The delta and the flag bits of a maximum's key (the conversion of key_to_delta_kernel).
__device__ __forceinline__ int32_t key_delta(uint32_t key, int shift, uint32_t& bad) {
    int32_t e = 0;
    bad = 0;
    if (key == KEY_NAN)
        bad = 4u;
    else if (key == KEY_TINY)
        bad = 2u;
    else if (key >= 0x7F80u)
        bad = 1u;
    else if (key != 0u) {
        const uint32_t E = (key >> 7) & 0xFFu, m = key & 0x7Fu;
        e = (int32_t)E - 127 + (m ? 1 : 0);
    }
    return shift - e;
}

}  // namespace
