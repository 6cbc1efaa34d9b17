// Real transforms of lengths without a fused half-length plan (odd n, even n
// whose half has a large prime factor).  In a DCT, DST or DHT two real lines
// travel as the real and imaginary part of one n-point complex transform,
//   Z = DFT(v_a + i v_b),  V_a = (Z_k + conj Z_{n-k})/2,
//                          V_b = (Z_k - conj Z_{n-k})/2i,
// in one launch while n (or its Bluestein convolution) fits a workgroup's
// LDS.  DCT and DST take Makhoul's order v_j = x_2j, v_{n-1-j} = x_{2j+1} and
// C_k = Re(q_k V_k), C_{n-k} = -Im(q_k V_k) with q_k = exp(-i pi k/2n).
// It replaces a mirrored 2n-point complex transform of every line: a quarter
// of the points (DST 999 x 1000 FP64, both directions: 203 -> 97 us; DST
// 381 x 1099 FP32 333 -> 64 with one-launch Bluestein).
// Two such lines share their rounding errors and their NaNs, which is right
// where several lines exist only as an axis of a 2D or 3D transform, whose
// other axes mix them all.  The lines of a batch of packed real transforms are
// signals of their own: they travel one by one, with zero imaginary parts.
#pragma once
#include "jt_fft1d.hpp"

namespace jt {

enum { R2R_DCT = 1, R2R_DST = 2, R2R_DHT = 3, R2R_PACKED = 4 };

// Lines of n reals, element k of line l at data[m.base(l) + k*m.es].
//   f0, g: factor of element 0 of the spectrum side, overall factor.
// I: the type of an index along a line.
template <typename T, int KIND, bool FWD, bool CONV, typename I = int>
struct IOPair {
    static constexpr bool pre_lds = true, post_lds = true, store_loads = false, conv = CONV;
    static constexpr bool makhoul = KIND == R2R_DCT || KIND == R2R_DST;
    static constexpr bool paired = KIND != R2R_PACKED;
    static const char* tag() {
        return KIND == R2R_DHT ? "dht,pair" : KIND == R2R_PACKED ? (FWD ? "r2c,odd" : "c2r,odd")
               : KIND == R2R_DCT ? (FWD ? "dct2,pair" : "dct3,pair") : (FWD ? "dst2,pair" : "dst3,pair");
    }
    std::string desc() const { return ",n=" + std::to_string(n) + ",es=" + std::to_string(m.es); }
    T* data;
    const cpx<T>* q;  // DCT, DST: exp(-i pi k / 2n), k in [0, n]
    Chirp<T> c;       // CONV
    LineMap m;
    int64_t nlines;  // transforms: pairs, or single lines
    I n;
    int len;  // points of the LDS line: n, or the convolution's m
    T f0, g;
    bool xcd;
    struct At {
        int64_t a, b;
        bool two;  // the last pair of an odd number of lines has one
    };
    __device__ __forceinline__ At base(int64_t p) const {
        if constexpr (!paired) {
            const int64_t o = m.base(p);
            return At{o, o, false};
        }
        const int64_t a = m.base(2 * p);
        const bool two = 2 * p + 1 < m.nlines;
        return At{a, two ? m.base(2 * p + 1) : a, two};
    }
    __device__ __forceinline__ cpx<T> rd(At at, I i) const {
        if constexpr (!paired) return cpx<T>{data[at.a + i * m.es], T(0)};
        const cpx<T> v{data[at.a + i * m.es], data[at.b + i * m.es]};
        return cpx<T>{v.x, at.two ? v.y : T(0)};
    }
    __device__ __forceinline__ void wr(At at, I i, T a, T b) const {
        data[at.a + i * m.es] = a;
        if constexpr (paired) {
            if (at.two) data[at.b + i * m.es] = b;
        }
    }
    // the line's element that is v_j
    __device__ __forceinline__ I vidx(I j) const {
        if constexpr (makhoul) return 2 * j < n ? 2 * j : 2 * (n - 1 - j) + 1;
        else return j;
    }
    // spectrum index (the DST reverses the DCT's)
    __device__ __forceinline__ I sidx(I k) const { return KIND == R2R_DST ? n - 1 - k : k; }

    // z_k of the signals (FWD), or Z_k of the spectra
    __device__ __forceinline__ cpx<T> in(At at, I k) const {
        if constexpr (FWD) {
            const I i = vidx(k);
            cpx<T> v = rd(at, i);
            if (KIND == R2R_DST && (i & 1)) v = cpx<T>{-v.x, -v.y};
            return v;
        } else if constexpr (KIND == R2R_PACKED) {
            const I h = 2 * k <= n ? k : n - k;
            const bool real = h == 0 || 2 * h == n;
            const I ir = 2 * h == n ? 1 : 2 * h, ii = real ? 0 : (2 * h + 1 == n ? 1 : 2 * h + 1);
            const cpx<T> r = rd(at, ir);
            cpx<T> s = rd(at, ii);
            if (real) s = cpx<T>{T(0), T(0)};
            if (h != k) s = cpx<T>{-s.x, -s.y};
            return cpx<T>{r.x - s.y, r.y + s.x};  // X_a + i X_b
        } else {
            cpx<T> u = rd(at, sidx(k)), w = rd(at, sidx(k ? n - k : 0));
            if (k == 0) {
                u = cpx<T>{u.x * f0, u.y * f0};
                w = cpx<T>{T(0), T(0)};
            }
            // half conj(q_k) (u - i w) of both lines, summed as A + i B
            u = cpx<T>{u.x * T(0.5), u.y * T(0.5)};
            w = cpx<T>{w.x * T(0.5), w.y * T(0.5)};
            return cmulc(cpx<T>{u.x + w.y, u.y - w.x}, q[k]);
        }
    }
    __device__ cpx<T> load(At, int, int) const { return cpx<T>{T(0), T(0)}; }
    __device__ void store(At, int, int, cpx<T>) const {}
    __device__ __forceinline__ cpx<T> spec(At, int k, int rm) const { return c.spec(k + rm); }

    // inverse: z_k = n (v_a + i v_b) back into the lines
    __device__ __forceinline__ void join(At at, I k, cpx<T> z) const {
        const I i = vidx(k);
        const T s = KIND == R2R_DST && (i & 1) ? -g : g;
        wr(at, i, z.x * s, z.y * s);
    }
    // forward: the outputs that Z_k and Z_{n-k} (k <= n/2; Z_0 twice for k = 0) give
    __device__ __forceinline__ void split(At at, I k, cpx<T> A, cpx<T> B, cpx<T> qk) const {
        if constexpr (!paired) {
            // Z_k = conj Z_{n-k} up to rounding, which their mean lowers by a
            // quarter (halved first: the sum may be beyond the type's range)
            const T h = T(0.5) * g;
            wr(at, 2 * k == n ? 1 : 2 * k, A.x * h + B.x * h, T(0));
            if (k > 0 && 2 * k != n) wr(at, 2 * k + 1 == n ? 1 : 2 * k + 1, A.y * h - B.y * h, T(0));
            return;
        }
        const cpx<T> Ah{A.x * T(0.5), A.y * T(0.5)}, Bc{B.x * T(0.5), B.y * T(-0.5)};
        const cpx<T> s = cadd(Ah, Bc), d = csub(Ah, Bc);
        cpx<T> a{s.x * g, s.y * g}, b{d.y * g, -d.x * g};  // g V_a, g V_b
        if constexpr (makhoul) {
            a = cmul(qk, a);
            b = cmul(qk, b);
            const T f = k == 0 ? f0 : T(1);
            wr(at, sidx(k), a.x * f, b.x * f);
            if (k > 0 && 2 * k != n) wr(at, sidx(n - k), -a.y, -b.y);
        } else {
            wr(at, k, a.x - a.y, b.x - b.y);
            if (k > 0 && 2 * k != n) wr(at, n - k, a.x + a.y, b.x + b.y);
        }
    }
    // Both hooks take a few points at a time: all loads of a batch before its
    // first LDS write or store (a wait for a load also waits for older
    // stores).  Loading the points into the first stage's registers instead
    // spilled: up to six loads make one point.
    template <int CN, int CTL>
    __device__ void pre(int64_t, At at, T* re, T* im, int t, int nt) const {
        constexpr int IT = 4;
        for (int k0 = t; k0 < len; k0 += IT * nt) {
            cpx<T> z[IT];
#pragma unroll
            for (int u = 0; u < IT; u++) {
                const int k = k0 + u * nt;
                if constexpr (CONV) z[u] = c.premul(k, [&](int64_t kk) { return in(at, (I)kk); });
                else if (k < len) z[u] = in(at, k);
            }
#pragma unroll
            for (int u = 0; u < IT; u++) {
                const int k = k0 + u * nt;
                if (k < len) {
                    re[gpos(k)] = z[u].x;
                    im[gpos(k)] = z[u].y;
                }
            }
        }
    }
    template <int CN, int CTL>
    __device__ void post(int64_t, At at, const T* re, const T* im, int t, int nt) const {
        constexpr int IT = 2;
        const int per = FWD ? n / 2 + 1 : n;
        for (int k0 = t; k0 < per; k0 += IT * nt) {
            cpx<T> qk[IT], ca[IT], cb[IT];
#pragma unroll
            for (int u = 0; u < IT; u++) {
                const int k = k0 + u * nt;
                if (k >= per) continue;
                if constexpr (FWD && makhoul) qk[u] = q[k];
                if constexpr (CONV) {
                    ca[u] = c.at(k);
                    if constexpr (FWD) cb[u] = c.at(k ? n - k : 0);
                }
            }
#pragma unroll
            for (int u = 0; u < IT; u++) {
                const int k = k0 + u * nt;
                if (k >= per) continue;
                cpx<T> A{re[gpos(k)], im[gpos(k)]};
                if constexpr (CONV) A = cmul(cpx<T>{A.x, -A.y}, ca[u]);
                if constexpr (FWD) {
                    const int kk = k ? n - k : 0;
                    cpx<T> B{re[gpos(kk)], im[gpos(kk)]};
                    if constexpr (CONV) B = cmul(cpx<T>{B.x, -B.y}, cb[u]);
                    split(at, k, A, B, qk[u]);
                } else {
                    join(at, k, A);
                }
            }
        }
    }
};

// The same steps around a transform of several launches, through a workspace
// of one n-point line per transform.
template <typename T, class IO>
__global__ void pair_in(IO io, cpx<T>* __restrict__ y) {
    const int64_t n = io.n, tot = io.nlines * n;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < tot; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t p = i / n;
        y[i] = io.in(io.base(p), i - p * n);
    }
}
template <typename T, class IO, bool FWD>
__global__ void pair_out(IO io, const cpx<T>* __restrict__ y) {
    const int64_t n = io.n, per = FWD ? n / 2 + 1 : n, tot = io.nlines * per;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < tot; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t p = i / per;
        const int64_t k = i - p * per;
        const cpx<T>* z = y + p * n;
        if constexpr (FWD) {
            cpx<T> qk{T(1), T(0)};
            if constexpr (IO::makhoul) qk = io.q[k];
            io.split(io.base(p), k, z[k], z[k ? n - k : 0], qk);
        } else {
            io.join(io.base(p), k, z[k]);
        }
    }
}

template <typename T>
bool pair_one_launch(const Fft1D<T>& p) { return p.kind == K_GEN || p.blue_single(); }

// Runs the lines lm through the n-point plan p; ws holds n points per
// transform (a pair of lines, or a line if packed) plus p's workspace for
// them, unless p is one launch.
template <typename T, int KIND, bool FWD>
void pair_lines(const Fft1D<T>& p, T* data, const cpx<T>* q, LineMap lm, T f0, T g, cpx<T>* ws, hipStream_t st) {
    const int64_t count = KIND == R2R_PACKED ? lm.nlines : (lm.nlines + 1) / 2;
    constexpr int D = FWD ? -1 : 1;
    const bool col = lm.es != 1;
    if (p.kind == K_GEN) {
        go_gen<T, D>(p, IOPair<T, KIND, FWD, false>{data, q, {}, lm, count, (int)p.n, (int)p.n, f0, g, col}, col, st);
        return;
    }
    if (p.blue_single()) {
        const Chirp<T> c{p.chirp.template as<cpx<T>>(), p.bspec.template as<cpx<T>>(), p.n, T(D)};
        go_gen<T, -1>(*p.pm, IOPair<T, KIND, FWD, true>{data, q, c, lm, count, (int)p.n, (int)p.m, f0, g, col}, col, st);
        return;
    }
    need_ws(ws);
    using IO = IOPair<T, KIND, FWD, false, int64_t>;
    const IO io{data, q, {}, lm, count, p.n, 0, f0, g, false};
    { JT_PROF(st, "pair_in");
    hipLaunchKernelGGL((pair_in<T, IO>), ew_grid(count * p.n), dim3(256), 0, st, io, ws);
    }
    JT_HIP(hipGetLastError());
    c2c_contig<T, D>(p, ws, ws, count, T(1), ws + count * p.n, st);
    { JT_PROF(st, "pair_out");
    hipLaunchKernelGGL((pair_out<T, IO, FWD>), ew_grid(count * (FWD ? p.n / 2 + 1 : p.n)), dim3(256), 0, st, io, ws);
    }
    JT_HIP(hipGetLastError());
}

// Instantiated in jt_pair_f64.hip and jt_pair_f32.hip.
#define JT_PAIR_INST1(X, T, K, F)                                                                                \
    X template void pair_lines<T, K, F>(const Fft1D<T>&, T*, const cpx<T>*, LineMap, T, T, cpx<T>*, hipStream_t);
#define JT_PAIR_INST(X, T)              \
    JT_PAIR_INST1(X, T, R2R_DCT, true)   \
    JT_PAIR_INST1(X, T, R2R_DCT, false)  \
    JT_PAIR_INST1(X, T, R2R_DST, true)   \
    JT_PAIR_INST1(X, T, R2R_DST, false)  \
    JT_PAIR_INST1(X, T, R2R_DHT, true)   \
    JT_PAIR_INST1(X, T, R2R_PACKED, true) \
    JT_PAIR_INST1(X, T, R2R_PACKED, false)
JT_PAIR_INST(extern, float)
JT_PAIR_INST(extern, double)

}  // namespace jt
