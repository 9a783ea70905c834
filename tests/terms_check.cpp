// terms_get8 (csrc/wm_terms.h) at the ends of its range: prints one line per
// case, "ok" or what differs.
#include <sys/mman.h>

#include <cstdio>

#include "wm_terms.h"

struct plain {
    float map(float x, uint32_t) const { return x; }
};

int main() {
    // 2^32 floats, of which only the pages touched exist
    const size_t n_max = size_t(1) << 32;
    void *m = mmap(nullptr, n_max * 4, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) {
        perror("mmap");
        return 2;
    }
    float *a = static_cast<float *>(m);
    for (size_t i = 0; i < 64; i++) a[i] = 1.0f + i;
    for (size_t i = n_max - 64; i < n_max; i++) a[i] = 1.0f + (i - (n_max - 64));
    const uint32_t last = 0xfffffff8u;  // the last multiple of 8
    const uint32_t cases[][2] = {{0, 1},   {0, 7},    {0, 8},           {8, 8},           {8, 15},          {8, 16},
                                 {16, 17}, {16, 8},   {24, 3},          {last, last + 1}, {last, last + 3}, {last, last + 7},
                                 {last, last}, {last - 8, last}, {last - 8, last - 1}, {last - 8, last + 7}};
    int bad = 0;
    for (const auto &c : cases) {
        float v[8];
        wm::terms_get8(plain{}, a, c[0], c[1], v);
        for (uint32_t j = 0; j < 8; j++) {
            const uint64_t k = (uint64_t)c[0] + j;
            const float want = k < c[1] ? a[k] : 0.0f;
            if (v[j] != want) {
                printf("i %u n %u term %u: %g, not %g\n", c[0], c[1], j, v[j], want);
                bad = 1;
            }
        }
        printf("i %u n %u done\n", c[0], c[1]);
    }
    return bad;
}
