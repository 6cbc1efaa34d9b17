// DCT-II/III, DST-II/III and DHT (1D/2D/3D) on the complex engine.
//
// Reference semantics (dct/DoubleDCT_1D.java:169-434, dst/DoubleDST_1D.java:
// 96-318, dht/DoubleDHT_1D.java:94-268, DHT_2D/3D yTransform):
//   DCT forward  C_k = sum_j x_j cos(pi (2j+1) k / 2n); returned as C_k for
//                power-of-two n, 2 C_k otherwise; scale -> orthonormal.
//   DCT inverse  power of two: a_0 + sum_{k>=1} a_k cos(pi k (2m+1)/2n);
//                otherwise (1/n)(a_0/2 + sum_{k>=1} ...); scale -> orthonormal.
//   DST          negate odd inputs, DCT-II, reverse (inverse mirrors it).
//   DHT          H_k = Re X_k - Im X_k; inverse = forward (x 1/n if scale).
//
// Even n with a single-kernel n/2 plan runs fused in one Stockham launch per
// axis: the pre hook gathers the line with Makhoul's even/odd permutation
// (v_j = x_2j, v_{n-1-j} = x_{2j+1}) into n/2 complex points, the post hook
// applies the real-FFT split and the exp(-i pi k/2n) twiddle and stores the
// n results (with the DST's sign/reverse maps folded into the index maps).
// Odd n, and even n whose Bluestein convolution fits LDS, run two lines as one
// n-point complex transform (jt_pair.hpp); other even n the same steps as the
// fused form, around an n/2-point transform of several launches.
#pragma once
#include "jt_multid.hpp"

namespace jt {

// ---------------------------------------------------------------------------
// scale conventions
// ---------------------------------------------------------------------------
struct R2RScale {
    double f0;    // extra factor on element 0 (forward: applied to output 0;
                  // inverse: applied to input 0)
    double g;     // overall factor
};

// Forward DCT-II from the unnormalised C_k.
inline R2RScale dct2_scale(int64_t n, bool scale) {
    if (scale) return {1.0 / std::sqrt(2.0), std::sqrt(2.0 / (double)n)};
    return {1.0, is_pow2(n) ? 1.0 : 2.0};
}
// Inverse DCT-III as g * y(a') with y(a) = a_0/2 + sum_{k>=1} a_k cos(.) and
// a'_0 = f0 a_0.
inline R2RScale dct3_scale(int64_t n, bool scale) {
    if (scale) return {std::sqrt(2.0), std::sqrt(2.0 / (double)n)};
    if (is_pow2(n)) return {2.0, 1.0};
    return {1.0, 1.0 / (double)n};
}

// ---------------------------------------------------------------------------
// the split between the n/2-point complex transform Z and the outputs at k,
// n-k, N-k and N+k (N = n/2, 0 < k <= N/2); w = exp(-2 pi i k/n), qa = q_k,
// qb = q_{N-k}, q_k = exp(-i pi k/2n)
// ---------------------------------------------------------------------------
template <int KIND, typename T>
__device__ __forceinline__ void half_fwd(cpx<T> A, cpx<T> B, cpx<T> w, cpx<T> qa, cpx<T> qb, T* y) {
    // A = Z_k, B = conj Z_{N-k}; halved before they are summed, so that V_k up
    // to the type's largest value does not overflow on the way
    A = cpx<T>{A.x * T(0.5), A.y * T(0.5)};
    B = cpx<T>{B.x * T(0.5), B.y * T(0.5)};
    const cpx<T> fe = cadd(A, B), d = csub(A, B);
    const cpx<T> fo = {d.y, -d.x};
    const cpx<T> wf = cmul(w, fo);
    const cpx<T> Vk = {fe.x + wf.x, fe.y + wf.y};
    const cpx<T> Vc = {fe.x - wf.x, -(fe.y - wf.y)};  // V_{N-k}
    if constexpr (KIND == R2R_DHT) {
        y[0] = Vk.x - Vk.y;
        y[1] = Vk.x + Vk.y;
        y[2] = Vc.x - Vc.y;
        y[3] = Vc.x + Vc.y;
    } else {
        const cpx<T> a = cmul(qa, Vk), c = cmul(qb, Vc);
        y[0] = a.x;
        y[1] = -a.y;
        y[2] = c.x;
        y[3] = -c.y;
    }
}
// DCT-III: Z_k and Z_{N-k} from V_k = conj(q_k)(a_k - i a_{n-k}) and V_{N-k}
template <typename T>
__device__ __forceinline__ void half_inv(cpx<T> qa, cpx<T> qb, cpx<T> w, T ak, T ank, T akk, T ankk, cpx<T>& Zk,
                                         cpx<T>& Zkk) {
    const cpx<T> Vk = cmulc(cpx<T>{ak, -ank}, qa);
    const cpx<T> Vc = cmulc(cpx<T>{akk, -ankk}, qb);
    const cpx<T> Xc = {Vc.x, -Vc.y};  // conj V_{N-k}
    const cpx<T> E = cadd(Vk, Xc), D = csub(Vk, Xc);
    const cpx<T> O = cmul(D, cpx<T>{w.x, -w.y});
    Zk = cpx<T>{E.x - O.y, E.y + O.x};
    Zkk = cpx<T>{E.x + O.y, O.x - E.y};
}

// ---------------------------------------------------------------------------
// fused IO policy.  Real data: element k of line l at data[base(l) + k*es].
// Bound: HBM, as long as a batch's loads are in flight together.  The inverse
// hook used to select per load (a_n = 0, a'_0 = f0 a_0), which put a wait
// behind every load, and to write one element at a time from LDS: the three
// DCT-III passes of 512^3 FP64 took 727, 775 and 743 us (2.9 TB/s); without
// the selections, four elements at a time, 495, 502 and 582 (3.7-4.3).
// N = n/2 complex points per line.  q[k] = exp(-i pi k / 2n), k in [0, n];
// rtw[k] = exp(-2 pi i k / n), k in [0, n/4 + 1].
// ---------------------------------------------------------------------------
template <typename T, int KIND, bool FWD>
struct IOR2R {
    static constexpr bool pre_lds = true, post_lds = true, store_loads = false, conv = false;
    // lines of reals: a column group's row segment is W * sizeof(T) bytes
    static constexpr bool real_lines = true;
    static const char* tag() {
        return KIND == R2R_DHT ? "dht" : (KIND == R2R_DCT ? (FWD ? "dct2" : "dct3") : (FWD ? "dst2" : "dst3"));
    }
    std::string desc() const { return ",es=" + std::to_string(m.es); }
    T* data;
    const cpx<T>* q;
    const cpx<T>* rtw;
    LineMap m;  // real units
    int64_t nlines;
    int n, N;
    T f0, g;
    bool xcd;
    __device__ __forceinline__ int64_t base(int64_t l) const { return m.base(l); }
    __device__ cpx<T> load(int64_t, int, int) const { return cpx<T>{T(0), T(0)}; }
    __device__ void store(int64_t, int, int, cpx<T>) const {}

    __device__ __forceinline__ T rd(int64_t b, int k) const { return data[b + (int64_t)k * m.es]; }
    __device__ __forceinline__ void wr(int64_t b, int k, T v) const { data[b + (int64_t)k * m.es] = v; }

    // inverse input a_k (DST reads reversed); a'_0 = f0 a_0 is the caller's
    __device__ __forceinline__ T ain(int64_t b, int k) const { return rd(b, KIND == R2R_DST ? n - 1 - k : k); }

    // Four consecutive elements i, .., i+3 of the line at a time: contiguous
    // lines hold them in two aligned pairs (n is even and the data
    // pair-aligned).
    __device__ __forceinline__ void rd4(int64_t b, int i, T* x) const {
        if (m.es == 1) {
            const cpx<T>* p = reinterpret_cast<const cpx<T>*>(data + b + i);
            const cpx<T> lo = p[0], hi = p[1];
            x[0] = lo.x; x[1] = lo.y; x[2] = hi.x; x[3] = hi.y;
        } else {
#pragma unroll
            for (int u = 0; u < 4; u++) x[u] = rd(b, i + u);
        }
    }
    __device__ __forceinline__ void wr4(int64_t b, int i, const T* x) const {
        if (m.es == 1) {
            cpx<T>* p = reinterpret_cast<cpx<T>*>(data + b + i);
            p[0] = cpx<T>{x[0], x[1]};
            p[1] = cpx<T>{x[2], x[3]};
        } else {
#pragma unroll
            for (int u = 0; u < 4; u++) wr(b, i + u, x[u]);
        }
    }
    // Makhoul's order v_j = x_2j, v_{n-1-j} = x_{2j+1} with z_m = v_2m + i
    // v_2m+1: elements 4h, .., 4h+3 are Re z_h, Im z_{N-1-h}, Im z_h and
    // Re z_{N-1-h} (h < N/2; for odd N, x_{n-2} and x_{n-1} are z_{(N-1)/2}).
    // The DHT keeps the natural order.
    __device__ __forceinline__ void put4(int h, const T* x, T* re, T* im) const {
        if constexpr (KIND == R2R_DHT) {
            re[lpos(2 * h)] = x[0];
            im[lpos(2 * h)] = x[1];
            re[lpos(2 * h + 1)] = x[2];
            im[lpos(2 * h + 1)] = x[3];
        } else {
            constexpr T sg = KIND == R2R_DST ? T(-1) : T(1);
            re[lpos(h)] = x[0];
            im[lpos(N - 1 - h)] = sg * x[1];
            im[lpos(h)] = x[2];
            re[lpos(N - 1 - h)] = sg * x[3];
        }
    }
    // the last pair of a line with odd N
    __device__ __forceinline__ void put_last(int64_t b, T* re, T* im) const {
        const int z = KIND == R2R_DHT ? N - 1 : (N - 1) / 2;
        const T y = rd(b, n - 1);
        re[lpos(z)] = rd(b, n - 2);
        im[lpos(z)] = KIND == R2R_DST ? -y : y;
    }
    // inverse: Z_k, Z_{N-k} from a'_k, a'_{n-k}, a'_{N-k}, a'_{N+k}
    __device__ __forceinline__ void inv_pair(int k, T ak, T ank, T akk, T ankk, T* re, T* im) const {
        const int kk = N - k;
        cpx<T> Zk, Zkk;
        half_inv(q[k], q[kk], rtw[k], ak, ank, akk, ankk, Zk, Zkk);
        re[lpos(k)] = Zk.x;
        im[lpos(k)] = Zk.y;
        if (kk != k) {
            re[lpos(kk)] = Zkk.x;
            im[lpos(kk)] = Zkk.y;
        }
    }

    template <int CN, int CTL>
    __device__ void pre(int64_t, int64_t b, T* re, T* im, int t, int nt) const {
        if constexpr (FWD || KIND == R2R_DHT) {
            // all loads of a batch before its LDS writes (compile-time
            // lengths: one batch)
            constexpr int IT = CN > 0 ? (CN / 2 + CTL - 1) / CTL : 2;
            const int half = (CN > 0 ? CN : N) / 2, step = CTL > 0 ? CTL : nt;
            for (int h0 = t; h0 < half; h0 += IT * step) {
                T x[IT][4];
#pragma unroll
                for (int u = 0; u < IT; u++)
                    if (h0 + u * step < half) rd4(b, 4 * (h0 + u * step), x[u]);
#pragma unroll
                for (int u = 0; u < IT; u++)
                    if (h0 + u * step < half) put4(h0 + u * step, x[u], re, im);
            }
            if constexpr (CN == 0) {
                if ((N & 1) && t == 0) put_last(b, re, im);
            }
        } else {
            // DCT-III / DST-III: V_k = conj(q_k)(a'_k - i a'_{n-k}), then the
            // real-inverse split into Z (N points)
            if (t == 0) {
                T v0 = ain(b, 0) * f0;
                T vN = T(1.41421356237309504880168872420970) * ain(b, N);
                re[lpos(0)] = v0 + vN;
                im[lpos(0)] = v0 - vN;
            }
            // all loads of a batch before its LDS writes (compile-time
            // lengths: one batch)
            constexpr int IT = CN > 0 ? (CN / 2 + CTL - 1) / CTL : 2;
            const int nn = CN > 0 ? CN : N, step = CTL > 0 ? CTL : nt;
            for (int k0 = 1 + t; k0 <= nn / 2; k0 += IT * step) {
                T a0[IT], a1[IT], a2[IT], a3[IT];
#pragma unroll
                for (int u = 0; u < IT; u++) {
                    const int k = k0 + u * step;
                    if (k <= nn / 2) {
                        a0[u] = ain(b, k);
                        a1[u] = ain(b, 2 * nn - k);
                        a2[u] = ain(b, nn - k);
                        a3[u] = ain(b, nn + k);
                    }
                }
#pragma unroll
                for (int u = 0; u < IT; u++) {
                    const int k = k0 + u * step;
                    if (k <= nn / 2) inv_pair(k, a0[u], a1[u], a2[u], a3[u], re, im);
                }
            }
        }
    }

    // output index map (DST reverses the DCT-II output)
    __device__ __forceinline__ void out_fwd(int64_t b, int k, T v) const {
        T s = g;
        if (KIND != R2R_DHT && k == 0) s *= f0;
        if (KIND == R2R_DST) wr(b, n - 1 - k, v * s);
        else wr(b, k, v * s);
    }

    template <int CN, int CTL>
    __device__ void post(int64_t, int64_t b, const T* re, const T* im, int t, int nt) const {
        if constexpr (FWD || KIND == R2R_DHT) {
            // real-FFT split V_k / V_{N-k} from Z, then the transform
            // outputs.  A wait for a load also waits for older stores, so a
            // batch loads all its factors first and stores last.
            if (t == 0) {
                const T zr = re[lpos(0)], zi = im[lpos(0)];
                out_fwd(b, 0, zr + zi);
                out_fwd(b, CN > 0 ? CN : N, KIND == R2R_DHT ? zr - zi : T(0.70710678118654752440084436210485) * (zr - zi));
            }
            constexpr int IT = CN > 0 ? ((CN / 2 + CTL - 1) / CTL < 4 ? (CN / 2 + CTL - 1) / CTL : 4) : 2;
            const int nn = CN > 0 ? CN : N, step = CTL > 0 ? CTL : nt;
            for (int k0 = 1 + t; k0 <= nn / 2; k0 += IT * step) {
                cpx<T> w[IT], qa[IT], qb[IT];
                T y[IT][4];
#pragma unroll
                for (int u = 0; u < IT; u++) {
                    const int k = k0 + u * step;
                    if (k > nn / 2) continue;
                    w[u] = rtw[k];
                    if constexpr (KIND != R2R_DHT) {
                        qa[u] = q[k];
                        qb[u] = q[nn - k];
                    }
                }
#pragma unroll
                for (int u = 0; u < IT; u++) {
                    const int k = k0 + u * step;
                    if (k > nn / 2) continue;
                    const int kk = nn - k;
                    cpx<T> A = {re[lpos(k)], im[lpos(k)]};
                    cpx<T> B = {re[lpos(kk)], -im[lpos(kk)]};
                    half_fwd<KIND>(A, B, w[u], qa[u], qb[u], y[u]);
                }
#pragma unroll
                for (int u = 0; u < IT; u++) {
                    const int k = k0 + u * step;
                    if (k > nn / 2) continue;
                    out_fwd(b, k, y[u][0]);
                    out_fwd(b, 2 * nn - k, y[u][1]);
                    if (nn - k != k) {
                        out_fwd(b, nn - k, y[u][2]);
                        out_fwd(b, nn + k, y[u][3]);
                    }
                }
            }
        } else {
            // inverse: LDS holds n * (v_2m + i v_2m+1); x_2j = v_j, x_2j+1 = v_{n-1-j}
            constexpr int IT = CN > 0 ? ((CN / 2 + CTL - 1) / CTL < 4 ? (CN / 2 + CTL - 1) / CTL : 4) : 2;
            constexpr T sg = KIND == R2R_DST ? T(-1) : T(1);
            const int nn = CN > 0 ? CN : N, half = nn / 2, step = CTL > 0 ? CTL : nt;
            for (int h0 = t; h0 < half; h0 += IT * step) {
                T x[IT][4];
#pragma unroll
                for (int u = 0; u < IT; u++) {
                    const int h = h0 + u * step, hh = nn - 1 - h;
                    if (h >= half) continue;
                    x[u][0] = re[lpos(h)] * g;
                    x[u][1] = im[lpos(hh)] * (sg * g);
                    x[u][2] = im[lpos(h)] * g;
                    x[u][3] = re[lpos(hh)] * (sg * g);
                }
#pragma unroll
                for (int u = 0; u < IT; u++)
                    if (h0 + u * step < half) wr4(b, 4 * (h0 + u * step), x[u]);
            }
            if constexpr (CN == 0) {
                if ((N & 1) && t == 0) {
                    wr(b, n - 2, re[lpos((N - 1) / 2)] * g);
                    wr(b, n - 1, im[lpos((N - 1) / 2)] * (sg * g));
                }
            }
        }
    }
};

// ---------------------------------------------------------------------------
// the same steps for even n whose n/2-point transform takes several launches:
// lines gathered to N complex points each in the workspace, and back
// ---------------------------------------------------------------------------
template <int KIND>
__device__ __forceinline__ int64_t half_vidx(int64_t j, int64_t n) {
    if (KIND == R2R_DHT) return j;
    return 2 * j < n ? 2 * j : 2 * (n - 1 - j) + 1;
}

template <typename T, int KIND, bool FWD>
__global__ void half_in(const T* __restrict__ x, cpx<T>* __restrict__ z, LineMap m, int64_t n,
                        const cpx<T>* __restrict__ q, const cpx<T>* __restrict__ rtw, T f0) {
    const int64_t N = n / 2, per = FWD ? N : N / 2 + 1;
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    for (; i < m.nlines * per; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t l = i / per, k = i - l * per, b = m.base(l);
        cpx<T>* zl = z + l * N;
        auto rd = [&](int64_t j) { return x[b + j * m.es]; };
        if constexpr (FWD) {
            const int64_t j0 = half_vidx<KIND>(2 * k, n), j1 = half_vidx<KIND>(2 * k + 1, n);
            const T v0 = rd(j0), v1 = rd(j1);
            zl[k] = cpx<T>{KIND == R2R_DST && (j0 & 1) ? -v0 : v0, KIND == R2R_DST && (j1 & 1) ? -v1 : v1};
        } else {
            // (halved: Z is then the result itself, not twice it)
            auto a = [&](int64_t j) { return rd(KIND == R2R_DST ? n - 1 - j : j) * T(0.5); };
            if (k == 0) {
                const T v0 = a(0) * f0, vN = T(1.41421356237309504880168872420970) * a(N);
                zl[0] = cpx<T>{v0 + vN, v0 - vN};
                continue;
            }
            cpx<T> Zk, Zkk;
            half_inv(q[k], q[N - k], rtw[k], a(k), a(n - k), a(N - k), a(N + k), Zk, Zkk);
            zl[k] = Zk;
            if (N - k != k) zl[N - k] = Zkk;
        }
    }
}

template <typename T, int KIND, bool FWD>
__global__ void half_out(const cpx<T>* __restrict__ z, T* __restrict__ x, LineMap m, int64_t n,
                         const cpx<T>* __restrict__ q, const cpx<T>* __restrict__ rtw, T f0, T g) {
    const int64_t N = n / 2, per = FWD ? N / 2 + 1 : N;
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    for (; i < m.nlines * per; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t l = i / per, k = i - l * per, b = m.base(l);
        const cpx<T>* zl = z + l * N;
        if constexpr (FWD) {
            auto wr = [&](int64_t j, T v) { x[b + (KIND == R2R_DST ? n - 1 - j : j) * m.es] = v * g; };
            if (k == 0) {
                const T s = zl[0].x + zl[0].y, d = zl[0].x - zl[0].y;
                wr(0, KIND == R2R_DHT ? s : s * f0);
                wr(N, KIND == R2R_DHT ? d : T(0.70710678118654752440084436210485) * d);
                continue;
            }
            T y[4];
            cpx<T> qa{}, qb{};
            if constexpr (KIND != R2R_DHT) {
                qa = q[k];
                qb = q[N - k];
            }
            half_fwd<KIND>(zl[k], cpx<T>{zl[N - k].x, -zl[N - k].y}, rtw[k], qa, qb, y);
            wr(k, y[0]);
            wr(n - k, y[1]);
            if (N - k != k) {
                wr(N - k, y[2]);
                wr(N + k, y[3]);
            }
        } else {
            const int64_t j0 = half_vidx<KIND>(2 * k, n), j1 = half_vidx<KIND>(2 * k + 1, n);
            const T v0 = zl[k].x * g, v1 = zl[k].y * g;
            x[b + j0 * m.es] = KIND == R2R_DST && (j0 & 1) ? -v0 : v0;
            x[b + j1 * m.es] = KIND == R2R_DST && (j1 & 1) ? -v1 : v1;
        }
    }
}

// The multi-D DHT: separable 1D transforms along each axis give
// T(k) = sum x cas(a1) cas(a2) (...); the reference then turns T into the
// transform with cas(a1 + a2 (+ a3)) (its yTransform, DoubleDHT_2D.java:
// 1288-1309, DoubleDHT_3D.java:2314-2356).  2D: cas(x+y) = (cas(x)cas(y) +
// cas(-x)cas(y) + cas(x)cas(-y) - cas(-x)cas(-y)) / 2, so over the group
// {r, -r} x {c, -c} with T values A, B, C, D at (r,c), (-r,c), (r,-c),
// (-r,-c) each member moves by E = (A + D - B - C) / 2 (A - E, B + E, ...).
template <typename T>
__global__ void ytransform2d(T* __restrict__ a, int64_t rows, int64_t cols) {
    int64_t nr = rows / 2 + 1, nc = cols / 2 + 1;
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    for (; i < nr * nc; i += (int64_t)gridDim.x * blockDim.x) {
        int64_t r = i / nc, c = i % nc;
        int64_t mr = (rows - r) % rows, mc = (cols - c) % cols;
        // each group {r,mr} x {c,mc} once: skip the duplicate visits that
        // the reference's loop makes for r == rows/2 or c == cols/2 (they are
        // self-mirrored, so the update is the identity there)
        T A = a[r * cols + c], B = a[mr * cols + c], C = a[r * cols + mc], D = a[mr * cols + mc];
        T E = ((A + D) - (B + C)) / 2;
        if (r == mr || c == mc) continue;  // E is zero for self-mirrored groups
        a[r * cols + c] = A - E;
        a[mr * cols + c] = B + E;
        a[r * cols + mc] = C + E;
        a[mr * cols + mc] = D - E;
    }
}

// 3D: from cas(x+y+z) = (cas(-x)cas(y)cas(z) + cas(x)cas(-y)cas(z) +
// cas(x)cas(y)cas(-z) - cas(-x)cas(-y)cas(-z)) / 2 the true transform at k is
//   H(k) = (T(-k1,k2,k3) + T(k1,-k2,k3) + T(k1,k2,-k3) - T(-k1,-k2,-k3)) / 2
// of the separable one T.  One thread per orbit of (s, r, c) under negation
// of each index: member b (bit 0 slice, bit 1 row, bit 2 column negated)
// gets (T[b^1] + T[b^2] + T[b^4] - T[b^7]) / 2; self-mirrored indices give
// coinciding members that receive equal values.
template <typename T>
__global__ void ytransform3d(T* __restrict__ a, int64_t sl, int64_t rows, int64_t cols) {
    const int64_t ns = sl / 2 + 1, nr = rows / 2 + 1, nc = cols / 2 + 1;
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    for (; i < ns * nr * nc; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t s = i / (nr * nc), r = (i / nc) % nr, c = i % nc;
        const int64_t sp[2] = {s * rows * cols, ((sl - s) % sl) * rows * cols};
        const int64_t rp[2] = {r * cols, ((rows - r) % rows) * cols};
        const int64_t cp[2] = {c, (cols - c) % cols};
        int64_t at[8];
        T t[8];
#pragma unroll
        for (int m = 0; m < 8; m++) {
            at[m] = sp[m & 1] + rp[(m >> 1) & 1] + cp[(m >> 2) & 1];
            t[m] = a[at[m]];
        }
#pragma unroll
        for (int m = 0; m < 8; m++) a[at[m]] = (t[m ^ 1] + t[m ^ 2] + t[m ^ 4] - t[m ^ 7]) / 2;
    }
}

// ---------------------------------------------------------------------------
// plan
// ---------------------------------------------------------------------------
template <typename T>
struct R2R1D {
    int kind = R2R_DCT;
    int64_t n = 0;
    std::unique_ptr<Fft1D<T>> half;  // n/2: fused if one launch, else through the workspace
    std::unique_ptr<Fft1D<T>> full;  // n: lines in pairs
    DevBuf q, rtw;
    bool fused() const { return half && half->single(); }
    bool one_launch() const { return n == 1 || fused() || (full && pair_one_launch(*full)); }
    int64_t ws_elems(int64_t lines) const {
        if (fused() || n == 1) return 0;
        // the bound that callers of the fixed-scratch entry point know: the
        // workspace of a 2n-point (DHT: n-point) complex transform of each line
        const int64_t L = kind == R2R_DHT ? n : 2 * n, pairs = (lines + 1) / 2;
        const int64_t need = half ? lines * (n / 2) + half->workspace(lines) : pairs * n + full->workspace(pairs);
        return std::max(need, lines * L + plan_workspace<T>(L, lines));
    }
};

template <typename T>
std::unique_ptr<R2R1D<T>> make_r2r1d(int family, int64_t n) {
    auto r = std::make_unique<R2R1D<T>>();
    r->kind = family == 1 ? R2R_DCT : (family == 2 ? R2R_DST : R2R_DHT);
    r->n = n;
    if (n == 1) return r;
    std::vector<cpx<T>> q(n + 1);
    for (int64_t k = 0; k <= n; k++) q[k] = expm<T>(k, 4 * n);
    upload(r->q, q);
    if (n % 2 == 0 && n >= 4) {
        auto h = make_fft1d<T>(n / 2);
        if (h->single() || next_smooth(2 * n - 1) > gen_max<T>()) {
            r->half = std::move(h);
            std::vector<cpx<T>> w(n / 4 + 2);
            for (int64_t k = 0; k < (int64_t)w.size(); k++) w[k] = expm<T>(k, n);
            upload(r->rtw, w);
            return r;
        }
    }
    r->full = make_fft1d<T>(n);
    return r;
}

template <typename T, int KIND, bool FWD>
void r2r_axis_k(const R2R1D<T>& r, T* data, LineMap lm, bool scale, cpx<T>* ws, hipStream_t st) {
    const int64_t n = r.n;
    // DHT: `scale` is only passed for the inverse (forward(a) has no scale)
    R2RScale sc = (KIND == R2R_DHT) ? R2RScale{1.0, scale ? 1.0 / (double)n : 1.0}
                                    : (FWD ? dct2_scale(n, scale) : dct3_scale(n, scale));
    if (r.fused()) {
        const int64_t N = n / 2;
        // inverse: LDS holds n * v; y(a') = (n/2) v  -> store factor g*(n/2)/n = g/2
        T g = FWD || KIND == R2R_DHT ? T(sc.g) : T(sc.g * 0.5);
        IOR2R<T, KIND, FWD> io{data, r.q.template as<cpx<T>>(), r.rtw.template as<cpx<T>>(), lm, lm.nlines,
                               (int)n, (int)N, T(sc.f0), g, lm.es != 1};
        if (lm.es == 1) run_single<T, (FWD || KIND == R2R_DHT) ? -1 : 1, false>(*r.half, io, st);
        else run_single<T, (FWD || KIND == R2R_DHT) ? -1 : 1, true>(*r.half, io, st);
        return;
    }
    // (the n-point and the half-length form halve an inverse's inputs instead)
    const T f0 = T(sc.f0), g = T(sc.g);
    const cpx<T>* q = r.q.template as<cpx<T>>();
    if (r.full) {
        pair_lines<T, KIND, FWD>(*r.full, data, q, lm, f0, g, ws, st);
        return;
    }
    need_ws(ws);
    const cpx<T>* rtw = r.rtw.template as<cpx<T>>();
    const int64_t N = n / 2;
    constexpr int D = FWD || KIND == R2R_DHT ? -1 : 1;
    { JT_PROF(st, "half_in");
    hipLaunchKernelGGL((half_in<T, KIND, FWD>), ew_grid(lm.nlines * N), dim3(256), 0, st, data, ws, lm, n, q, rtw, f0);
    }
    JT_HIP(hipGetLastError());
    c2c_contig<T, D>(*r.half, ws, ws, lm.nlines, T(1), ws + lm.nlines * N, st);
    { JT_PROF(st, "half_out");
    hipLaunchKernelGGL((half_out<T, KIND, FWD>), ew_grid(lm.nlines * N), dim3(256), 0, st, ws, data, lm, n, q, rtw, f0,
                       g);
    }
    JT_HIP(hipGetLastError());
}

template <typename T>
void r2r_axis(int family, const R2R1D<T>& r, T* data, LineMap lm, bool fwd, bool scale, cpx<T>* ws,
              hipStream_t st) {
    if (r.n == 1 || lm.nlines <= 0) return;
    if (!lm.div.exact(lm.nlines)) {
        exact_maps(lm, [&](int64_t off, const LineMap& m) { r2r_axis<T>(family, r, data + off, m, fwd, scale, ws, st); });
        return;
    }
    if (family == 1) {
        if (fwd) r2r_axis_k<T, R2R_DCT, true>(r, data, lm, scale, ws, st);
        else r2r_axis_k<T, R2R_DCT, false>(r, data, lm, scale, ws, st);
    } else if (family == 2) {
        if (fwd) r2r_axis_k<T, R2R_DST, true>(r, data, lm, scale, ws, st);
        else r2r_axis_k<T, R2R_DST, false>(r, data, lm, scale, ws, st);
    } else {
        r2r_axis_k<T, R2R_DHT, true>(r, data, lm, fwd ? false : scale, ws, st);
    }
}

template <typename T>
void run_r2r_nd(int family, int nd, const int64_t* d, const std::shared_ptr<R2R1D<T>>* r, T* a, bool fwd,
                bool scale, cpx<T>* ws, hipStream_t st) {
    if (nd == 1) {
        r2r_axis<T>(family, *r[0], a, LineMap{1, 1, d[0], 0, 1}, fwd, scale, ws, st);
        return;
    }
    if (nd == 2) {
        const int64_t R = d[0], C = d[1];
        r2r_axis<T>(family, *r[1], a, LineMap{R, R, C, 0, 1}, fwd, scale, ws, st);
        r2r_axis<T>(family, *r[0], a, LineMap{C, C, 1, 0, C}, fwd, scale, ws, st);
        if (family == 3) {
            { JT_PROF(st, "ytransform2d");
            hipLaunchKernelGGL((ytransform2d<T>), ew_grid((R / 2 + 1) * (C / 2 + 1)), dim3(256), 0, st, a, R, C);
            }
            JT_HIP(hipGetLastError());
        }
        return;
    }
    const int64_t S = d[0], R = d[1], C = d[2];
    r2r_axis<T>(family, *r[2], a, LineMap{S * R, S * R, C, 0, 1}, fwd, scale, ws, st);
    r2r_axis<T>(family, *r[1], a, LineMap{S * C, C, 1, R * C, C}, fwd, scale, ws, st);
    r2r_axis<T>(family, *r[0], a, LineMap{R * C, R * C, 1, 0, R * C}, fwd, scale, ws, st);
    if (family == 3) {
        { JT_PROF(st, "ytransform3d");
        hipLaunchKernelGGL((ytransform3d<T>), ew_grid((S / 2 + 1) * (R / 2 + 1) * (C / 2 + 1)), dim3(256), 0, st,
                           a, S, R, C);
        }
        JT_HIP(hipGetLastError());
    }
}

// Instantiated in jt_r2r_f64.hip and jt_r2r_f32.hip.
#define JT_R2R_INST(X, T)                                                                                        \
    X template void run_r2r_nd<T>(int, int, const int64_t*, const std::shared_ptr<R2R1D<T>>*, T*, bool, bool,      \
                                  cpx<T>*, hipStream_t);
JT_R2R_INST(extern, float)
JT_R2R_INST(extern, double)

}  // namespace jt
