// Where the lines of a launch start.  (Plain C++ as well, so that it can be
// checked without a GPU.)
#pragma once
#include <cstdint>

#if defined(__HIP__)
#define JT_HD __host__ __device__ __forceinline__
#else
#define JT_HD inline
#endif

namespace jt {

// l / n0 for 0 <= l < nlines as a multiply by mag = floor(2^64 / n0) + 1; mag 0
// where the quotient is always 0.  Straight code: a 64-bit division takes over
// a hundred instructions, and a branch around it puts the kernel arguments
// behind it a second, late load.
struct LineDiv {
    int64_t n0;
    uint64_t mag;
    JT_HD LineDiv(int64_t nlines, int64_t d) : n0(d), mag(nlines <= d ? 0 : ~uint64_t(0) / d + 1) {}
    JT_HD int64_t operator()(int64_t l) const {
#if defined(__HIP_DEVICE_COMPILE__)
        return (int64_t)__umul64hi((uint64_t)l, mag);
#else
        return (int64_t)(((unsigned __int128)(uint64_t)l * mag) >> 64);
#endif
    }
    // Whether every l < nlines divides right: mag * n0 = 2^64 + e with e < n0,
    // so the product is l / n0 + l * e / (n0 * 2^64), right while l * e < 2^64.
    // Only the middle axis of the largest volumes that a plan accepts (such as
    // 2 x 2 x 3087000000) goes beyond: a four-step transform or a Bluestein
    // convolution has under 2^32 columns and rows in all (2^40 points, factors
    // above 300).
    JT_HD bool exact(int64_t nlines) const {
        const uint64_t e = mag * (uint64_t)n0;
        return e == 0 || (uint64_t)nlines <= ~uint64_t(0) / e;
    }
};

// Lines l in [0, nlines) start at (l % n0)*s0 + (l / n0)*s1 (complex units);
// element k of a line sits es further per step.  (n0 = 1 is the same as
// n0 = nlines with s0 = s1.)
struct LineMap {
    int64_t nlines, s0, s1, es;
    LineDiv div;
    JT_HD LineMap(int64_t nl, int64_t n0, int64_t s0_, int64_t s1_, int64_t es_)
        : nlines(nl), s0(n0 == 1 ? s1_ : s0_), s1(s1_), es(es_), div(nl, n0 == 1 ? nl : n0) {}
    JT_HD int64_t base(int64_t l) const {
        const int64_t q = div(l);
        return (l - q * div.n0) * s0 + q * s1;
    }
};

// Calls f(offset, map) for maps that together are the lines of lm, each with
// an exact division: lm itself, or its groups of n0 lines one by one.  (As a
// host check: a shift that makes every quotient exact costs the FP64
// runtime-radix kernels 2-5%, 3000 points 19.1 -> 19.8 us for two calls.)
template <class F>
inline void exact_maps(const LineMap& lm, F f) {
    if (lm.div.exact(lm.nlines)) {
        f(int64_t(0), lm);
        return;
    }
    const int64_t n0 = lm.div.n0;
    for (int64_t l = 0; l < lm.nlines; l += n0) {
        const int64_t left = lm.nlines - l, nl = left < n0 ? left : n0;
        f(l / n0 * lm.s1, LineMap(nl, nl, lm.s0, 0, lm.es));
    }
}

}  // namespace jt
