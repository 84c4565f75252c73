// f32 values to halves and back on the host, and whether it has the instructions. Plain C++, without the runtime.
#pragma once

#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <atomic>

#if !defined(__HIP_DEVICE_COMPILE__)
#include <immintrin.h>
#endif

namespace itak {

// n bytes of f32 values from n / 2 bytes of halves, and back: false where some value is no f16's (a NaN
// counts as none: its payload would have to survive two conversions on either side).
#if !defined(__HIP_DEVICE_COMPILE__)
// (Streaming stores are no faster here: the pages are fresh, and the kernel has just cleared them.)
inline __attribute__((target("avx,f16c"))) void widen_halves(unsigned char *out, const unsigned char *in, uint64_t n) {
    uint64_t at = 0;
    for (; at + 32 <= n; at += 32)
        _mm256_storeu_ps(reinterpret_cast<float *>(out + at),
                         _mm256_cvtph_ps(_mm_loadu_si128(reinterpret_cast<const __m128i *>(in + at / 2))));
    for (; at < n; at += 4) {
        uint16_t h;
        memcpy(&h, in + at / 2, 2);
        const float f = _mm_cvtss_f32(_mm_cvtph_ps(_mm_cvtsi32_si128(h)));
        memcpy(out + at, &f, 4);
    }
}
inline __attribute__((target("avx,f16c"))) bool narrow_floats(unsigned char *out, const unsigned char *in, uint64_t n) {
    __m256 differ = _mm256_setzero_ps(), unordered = _mm256_setzero_ps();
    uint64_t at = 0;
    for (; at + 32 <= n; at += 32) {
        const __m256 f = _mm256_loadu_ps(reinterpret_cast<const float *>(in + at));
        const __m128i h = _mm256_cvtps_ph(f, _MM_FROUND_TO_NEAREST_INT);
        _mm_storeu_si128(reinterpret_cast<__m128i *>(out + at / 2), h);
        // (Bits, not values: a thread that takes subnormal f32 values as zero, as torch.set_flush_denormal asks for, would
        // find them equal to the zeros they become.)
        differ = _mm256_or_ps(differ, _mm256_xor_ps(f, _mm256_cvtph_ps(h)));
        unordered = _mm256_or_ps(unordered, _mm256_cmp_ps(f, f, _CMP_UNORD_Q));
    }
    const __m256i bits = _mm256_castps_si256(differ);
    bool exact = _mm256_testz_si256(bits, bits) && _mm256_movemask_ps(unordered) == 0;
    for (; at < n; at += 4) {
        float f;
        memcpy(&f, in + at, 4);
        const uint16_t h = uint16_t(_mm_cvtsi128_si32(_mm_cvtps_ph(_mm_set_ss(f), _MM_FROUND_TO_NEAREST_INT)));
        memcpy(out + at / 2, &h, 2);
        const float back = _mm_cvtss_f32(_mm_cvtph_ps(_mm_cvtsi32_si128(h)));
        exact = exact && f == f && memcmp(&f, &back, 4) == 0;
    }
    return exact;
}
inline bool has_f16c() {
    __builtin_cpu_init();
    return __builtin_cpu_supports("avx") && __builtin_cpu_supports("f16c");
}
#else
inline void widen_halves(unsigned char *, const unsigned char *, uint64_t) {}
inline bool narrow_floats(unsigned char *, const unsigned char *, uint64_t) { return false; }
inline bool has_f16c() { return false; }
#endif

// A chunk's n bytes of f32 values as halves at `out`, piece by piece while every value is an f16's and no other thread
// has met one that is none; otherwise false, with `worth_it` down, and `out` holds nothing. Rows that an f32 cache wrote
// fail on their first values: a piece is a few us, the chunk that was narrowed to its end before it was looked at 300, beside
// the 350 of the copy that follows (4.1 / 8.2 MB of such rows loaded in 384 / 516 us, now 296 / 436; 321 / 436 before rows
// crossed the link as halves).
constexpr uint64_t kNarrowPiece = 32 << 10;
inline bool narrow_chunk(unsigned char *out, const unsigned char *in, uint64_t n, std::atomic<bool> &worth_it) {
    for (uint64_t at = 0; at < n; at += kNarrowPiece) {
        if (!worth_it.load(std::memory_order_relaxed)) return false;
        if (narrow_floats(out + at / 2, in + at, std::min(kNarrowPiece, n - at))) continue;
        worth_it.store(false, std::memory_order_relaxed);
        return false;
    }
    return true;
}

}  // namespace itak
