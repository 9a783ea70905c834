// Eight terms of a left-to-right sum at a time.  Host and device.
#pragma once
#include <cstdint>

#include "wm_expf.h"  // WM_HD

namespace wm {

// v[j] = f.map(a[i + j], i + j) for the terms i .. i+7 of n (i a multiple of
// 8, a 32-byte aligned), zeros from n on.  n may be any uint32_t: i + 8 can
// be 2^32.
template <typename F>
WM_HD inline void terms_get8(const F &f, const float *a, uint32_t i, uint32_t n, float (&v)[8]) {
    if (n >= 8 && i <= n - 8) {
        const float *p = static_cast<const float *>(__builtin_assume_aligned(a + i, 32));
        float r[8];
        for (int j = 0; j < 8; j++) r[j] = p[j];
        for (int j = 0; j < 8; j++) v[j] = f.map(r[j], i + j);
    } else {
        for (uint32_t j = 0; j < 8; j++) v[j] = i + j < n ? f.map(a[i + j], i + j) : 0.0f;
    }
}

}  // namespace wm
