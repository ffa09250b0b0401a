// level_digits.h -- the sixteen OIL4 levels (src/block_codec.cpp:18-23) as two signed byte digits, and codes to digits.
// 10000 times a level is an integer n = 256 a + b of at most 15 bits; level q < 8 is minus level 15 - q.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace oilhip {

// 10000 times the levels 0.1260, 0.3976, 0.6508, 0.9275, 1.2392, 1.5995, 2.0522, 2.7178
constexpr int kLevelTimes1e4[8] = {1260, 3976, 6508, 9275, 12392, 15995, 20522, 27178};
constexpr int low_digit(int n) { return ((n + 128) & 255) - 128; }
// the digits a (high) or b of four magnitudes, one byte each
constexpr uint32_t digit_table(bool high, int first) {
    uint32_t t = 0;
    for (int i = 0; i < 4; ++i) {
        const int n = kLevelTimes1e4[first + i], b = low_digit(n), a = (n - b) / 256;
        t |= (uint32_t)((high ? a : b) & 255) << (8 * i);
    }
    return t;
}
constexpr bool digits_fit() {
    for (int n : kLevelTimes1e4) {
        const int b = low_digit(n), a = (n - b) / 256;
        if (a <= 0 || a > 127 || b == 0 || b == -128) return false;
    }
    return true;
}
static_assert(digits_fit(), "the byte-wise negation needs digits other than 0 and -128");

// four codes (low nibbles of the bytes of w) -> their digits, by byte permutes over tables held in registers; the sign is applied to
// four bytes at once, (x ^ m) + (m & 1), and carries nowhere because no digit is 0
__device__ __forceinline__ void level_digits(uint32_t w, uint32_t& a, uint32_t& b) {
    const uint32_t m = __builtin_amdgcn_perm(0u, 0u, (~w & 0x08080808u) | 0x05050505u);   // 0xFF where the code is below 8 (selector 13), else 0
    const uint32_t at = (w ^ m) & 0x07070707u, one = m & 0x01010101u;                     // magnitude: code - 8, or 7 - code
    a = (__builtin_amdgcn_perm(digit_table(true, 4), digit_table(true, 0), at) ^ m) + one;
    b = (__builtin_amdgcn_perm(digit_table(false, 4), digit_table(false, 0), at) ^ m) + one;
}

}  // namespace oilhip
