// ray_sums.h -- the position of a sample further along a ray, as the march's running sum gives it.
#pragma once
#include <cstdint>

namespace spr {

// p after n additions of d, each rounded (p = p + d), in one step: while the sums stay in
// one binade each addition moves p by the same multiple of its ulp, ties included (a tie
// rounds to the even neighbour, so the sum after it starts even and rounds the same way
// from then on: the step is taken from the third addition, whose two predecessors started
// on the binade's own grid).  Valid only when `same`: the first sum and the result lie in
// one binade, the result inside it (a sum a little below 2^e would round to 2^e on this
// binade's grid and not on the finer one below).  n >= 3; past 2^24, where n - 3 is rounded,
// sums that stay in one binade of 2^23 ulps do not move at all and q is c.
__device__ __forceinline__ float sum_ahead(float p, float d, float n, bool& same) {
    const float a = p + d, b = a + d, c = b + d;
    const float q = fmaf(n - 3.0f, c - b, c);
    same = (__float_as_uint(a) ^ __float_as_uint(q)) < 0x00800000u &&
           (__float_as_uint(q) & 0x007FFFFFu) != 0u;
    return q;
}

// p after n additions of d, binade by binade
__device__ __forceinline__ float sum_n(float p, float d, uint32_t n) {
    while (n >= 6u) {
        bool same;
        float q = sum_ahead(p, d, (float)n, same);
        if (same) return q;
        // as many additions as surely stay in the first sum's binade, else three by hand
        const float a = p + d, b = a + d, c = b + d;
        const float lo = __uint_as_float(__float_as_uint(a) & 0xFF800000u);  // its signed 2^e
        const float lim = (c > b) == (a > 0.0f) ? 2.0f * lo : lo;
        const float m = floorf((lim - c) * __builtin_amdgcn_rcpf(c - b)) - 1.0f;
        q = sum_ahead(p, d, m + 3.0f, same);
        const bool far = m >= 1.0f && m + 3.0f < (float)n && same;
        p = far ? q : c;
        n -= far ? (uint32_t)m + 3u : 3u;
    }
    for (; n > 0u; --n) p = p + d;
    return p;
}

}  // namespace spr
