// IO policies of the Stockham kernels: where a line's points come from, where
// the results go, and the O(N) pre/post passes fused around the FFT.
#pragma once
#include <string>

#include "jt_dft.hpp"
#include "jt_linemap.hpp"

namespace jt {

__device__ __forceinline__ int lpos(int k) { return k + (k >> 5); }

// Non-temporal (streaming) complex loads and stores: they skip the caches'
// allocation, which lets a pass that reads or writes each element once run
// closer to the HBM rate (a device copy: 6.4 TB/s with them, 5.7 without).
template <typename T>
__device__ __forceinline__ cpx<T> ld_nt(const cpx<T>* p) {
    typedef T v2 __attribute__((ext_vector_type(2)));
    v2 v = __builtin_nontemporal_load(reinterpret_cast<const v2*>(p));
    return cpx<T>{v.x, v.y};
}
template <typename T>
__device__ __forceinline__ void st_nt(cpx<T>* p, cpx<T> c) {
    typedef T v2 __attribute__((ext_vector_type(2)));
    v2 v = {c.x, c.y};
    __builtin_nontemporal_store(v, reinterpret_cast<v2*>(p));
}
enum { NT_LOAD = 1, NT_STORE = 2 };

// Plain complex lines, optionally scaled on store (complexInverse(scale)).
// NT: NT_LOAD / NT_STORE for a pass whose input is not read again / whose
// output is not read soon (contiguous lines of a large array).  A template
// argument, not a run-time flag: a branch per access costs the column
// kernels registers and load batching.
template <typename T, int NT = 0>
struct IOStrided {
    static constexpr bool pre_lds = false, post_lds = false, store_loads = false, conv = false;
    static constexpr int streaming = NT;
    static const char* tag() { return NT == 0 ? "c2c" : "c2c,nt"; }
    std::string desc() const { return ",es=" + std::to_string(m.es); }
    const cpx<T>* in;
    cpx<T>* out;
    LineMap m;
    int64_t nlines;
    T scale;
    bool xcd;
    __device__ __forceinline__ int64_t base(int64_t l) const { return m.base(l); }
    __device__ __forceinline__ cpx<T> load(int64_t b, int k, int rm) const {
        const cpx<T>* p = in + (b + k * m.es) + rm * m.es;
        if constexpr ((NT & NT_LOAD) != 0) return ld_nt(p);
        else return *p;
    }
    // one part (0 real, 1 imaginary) of element k
    __device__ __forceinline__ T loadf(int64_t b, int k, int part) const {
        return reinterpret_cast<const T*>(in + b + k * m.es)[part];
    }
    __device__ __forceinline__ void store(int64_t b, int k, int rm, cpx<T> v) const {
        const cpx<T> o{v.x * scale, v.y * scale};
        cpx<T>* p = out + (b + k * m.es) + rm * m.es;
        if constexpr ((NT & NT_STORE) != 0) st_nt(p, o);
        else *p = o;
    }
    template <int CN, int CTL>
    __device__ void pre(int64_t, int64_t, T*, T*, int, int) const {}
    template <int CN, int CTL>
    __device__ void post(int64_t, int64_t, const T*, const T*, int, int) const {}
};

// The column pass of a packed-real 2D transform with the rdft2d_sub fix of
// column 0 (reference: DoubleFFT_2D.java:2544-2574) done by the workgroup
// that transforms that column.  Column 0 holds the transform of
// Y[.][0] + i Y[.][cols/2]; for rows 0 < i < rows/2 and j = rows - i:
//   ISGN > 0 (realForward, after the FFT):  Z_j <- (Z_i - conj Z_j) / 2,
//                                           Z_i <- Z_i - Z_j(new);
//   ISGN < 0 (realInverse, before the FFT): Z_i <- Z_i + Z_j,
//                                           Z_j <- (Re(Z_i - Z_j), Im(Z_j - Z_i)).
template <typename T, int ISGN>
struct IOStridedFix2D : IOStrided<T> {
    static constexpr int line0_hook = ISGN;
    static const char* tag() { return ISGN > 0 ? "c2c,rdft2d" : "c2c,rdft2d_inv"; }
    int64_t rows;
    __device__ void line0(int tid, int nthreads) const {
        cpx<T>* col = this->out + this->m.base(0);
        const int64_t es = this->m.es;
        for (int64_t i = 1 + tid; i < rows / 2; i += nthreads) {
            const int64_t j = rows - i;
            const cpx<T> zi = col[i * es], zj = col[j * es];
            if constexpr (ISGN > 0) {
                const cpx<T> nj{T(0.5) * (zi.x - zj.x), T(0.5) * (zi.y + zj.y)};
                col[j * es] = nj;
                col[i * es] = cpx<T>{zi.x - nj.x, zi.y - nj.y};
            } else {
                col[i * es] = cpx<T>{zi.x + zj.x, zi.y + zj.y};
                col[j * es] = cpx<T>{zi.x - zj.x, zj.y - zi.y};
            }
        }
    }
};

// exp(DIR 2 pi i e / n) from two tables: hi[e >> 8] * lo[e & 255], both
// holding forward values exp(-2 pi i x/n).
template <int DIR, typename T>
__device__ __forceinline__ cpx<T> tw2(const cpx<T>* __restrict__ hi, const cpx<T>* __restrict__ lo,
                                     int64_t e) {
    cpx<T> w = cmul(hi[e >> 8], lo[e & 255]);
    return tw_dir<DIR>(w);
}

// Four-step pass A: transform length n = n1*n2 viewed as an n1 x n2 row-major
// matrix.  Line (b, j2) is column j2 of batch b (n1 points at stride n2); the
// result is multiplied by exp(DIR 2 pi i j2 k1 / n) and point k1 of column j2
// written to b*n + j2*oj + k1*ok: transposed (oj = n1, ok = 1) when the rows
// follow as columns of that n2 x n1 matrix, or in place (oj = 1, ok = n2).
template <typename T, int DIR>
struct IOFourA {
    static constexpr bool pre_lds = false, post_lds = false, store_loads = true, conv = false;
    static const char* tag() { return "fourA"; }
    std::string desc() const { return ",n1=" + std::to_string(n1) + ",n2=" + std::to_string(n2); }
    const cpx<T>* in;
    cpx<T>* out;
    const cpx<T>* hi;
    const cpx<T>* lo;
    int64_t nlines, n, n1, n2, oj, ok;
    bool xcd;
    LineDiv div;  // by n2
    struct At {
        int64_t i, o, j2;
    };
    __device__ __forceinline__ At base(int64_t l) const {
        const int64_t b = div(l), j2 = l - b * n2;
        return At{b * n + j2, b * n + j2 * oj, j2};
    }
    __device__ __forceinline__ cpx<T> load(At a, int k, int rm) const { return in[(a.i + k * n2) + rm * n2]; }
    __device__ __forceinline__ void store(At a, int k, int rm, cpx<T> v) const {
        const int64_t e = a.j2 * k + a.j2 * rm;  // j2 k1 < n2 n1: no reduction needed
        out[(a.o + k * ok) + rm * ok] = cmul(v, tw2<DIR>(hi, lo, e));
    }
    template <int CN, int CTL>
    __device__ void pre(int64_t, At, T*, T*, int, int) const {}
    template <int CN, int CTL>
    __device__ void post(int64_t, At, const T*, const T*, int, int) const {}
};

// Bluestein (DoubleFFT_1D.java:1864-2107): X_k = c'_k * sum_j (x_j c'_j)
// c_{k-j} with the chirp c_j = exp(i pi j^2/n) and c' its conjugate (forward)
// or itself (backward, with the conjugated kernel spectrum), as a cyclic
// convolution of length m >= 2n-1.
template <typename T>
struct Chirp {
    const cpx<T>* ch;  // n entries
    const cpx<T>* bs;  // kernel spectrum / m, m entries
    int64_t n;
    T sg;              // -1 forward, +1 backward
    __device__ __forceinline__ cpx<T> at(int64_t k) const { return cpx<T>{ch[k].x, sg * ch[k].y}; }
    // x[k] c'_k, 0 for k >= n; `at_k(k)` loads x[k] (without a branch, so that
    // all loads of a thread are in flight together)
    template <class F>
    __device__ __forceinline__ cpx<T> premul(int64_t k, F at_k) const {
        const bool in = k < n;
        const int64_t kk = in ? k : n - 1;
        const cpx<T> v = cmul(at_k(kk), at(kk));
        return in ? v : cpx<T>{T(0), T(0)};
    }
    __device__ __forceinline__ cpx<T> spec(int64_t k) const { return cpx<T>{bs[k].x, -sg * bs[k].y}; }
    __device__ __forceinline__ cpx<T> postmul(int64_t k, cpx<T> v, T scale) const {
        const cpx<T> o = cmul(v, at(k));
        return cpx<T>{o.x * scale, o.y * scale};
    }
};

// A whole Bluestein transform per line: the m-point convolution in one LDS
// residency, so a line is read and written once.  (As five to seven launches
// with the m points in memory between them, 2123 lines of 606 FP64 points took
// 133 us a direction, 42 this way; an axis of stride > 1 needs no gather.)
template <typename T>
struct IOBlue {
    static constexpr bool pre_lds = false, post_lds = false, store_loads = true, conv = true;
    static const char* tag() { return "blue"; }
    std::string desc() const { return ",n=" + std::to_string(c.n) + ",es=" + std::to_string(m.es); }
    const cpx<T>* in;
    cpx<T>* out;
    Chirp<T> c;
    LineMap m;
    int64_t nlines;
    T scale;
    bool xcd;
    __device__ __forceinline__ int64_t base(int64_t l) const { return m.base(l); }
    __device__ __forceinline__ cpx<T> load(int64_t b, int k, int rm) const {
        return c.premul(k + rm, [&](int64_t kk) { return in[b + kk * m.es]; });
    }
    __device__ __forceinline__ cpx<T> spec(int64_t, int k, int rm) const { return c.spec(k + rm); }
    __device__ __forceinline__ void store(int64_t b, int k, int rm, cpx<T> v) const {
        const int64_t kk = k + rm;
        if (kk < c.n) out[b + kk * m.es] = c.postmul(kk, cpx<T>{v.x, -v.y}, scale);
    }
};

// Contiguous lines of n reals in, n complex points out (realForwardFull and
// realInverseFull), per line or, with the chirp, as a Bluestein transform.
template <typename T>
struct IORealRows {
    static constexpr bool pre_lds = false, post_lds = false, store_loads = false, conv = false;
    static const char* tag() { return "real rows"; }
    std::string desc() const { return ",n=" + std::to_string(n); }
    const T* in;
    cpx<T>* out;
    int64_t n, nlines;
    T scale;
    bool xcd;
    __device__ __forceinline__ int64_t base(int64_t l) const { return l * n; }
    __device__ __forceinline__ cpx<T> load(int64_t b, int k, int rm) const { return cpx<T>{in[b + k + rm], T(0)}; }
    __device__ __forceinline__ void store(int64_t b, int k, int rm, cpx<T> v) const {
        out[b + k + rm] = cpx<T>{v.x * scale, v.y * scale};
    }
    template <int CN, int CTL>
    __device__ void pre(int64_t, int64_t, T*, T*, int, int) const {}
    template <int CN, int CTL>
    __device__ void post(int64_t, int64_t, const T*, const T*, int, int) const {}
};
template <typename T>
struct IORealRowsBlue : IORealRows<T> {
    static constexpr bool store_loads = true, conv = true;
    Chirp<T> c;
    __device__ __forceinline__ cpx<T> load(int64_t b, int k, int rm) const {
        return c.premul(k + rm, [&](int64_t kk) { return cpx<T>{this->in[b + kk], T(0)}; });
    }
    __device__ __forceinline__ cpx<T> spec(int64_t, int k, int rm) const { return c.spec(k + rm); }
    __device__ __forceinline__ void store(int64_t b, int k, int rm, cpx<T> v) const {
        const int64_t kk = k + rm;
        if (kk < c.n) this->out[b + kk] = c.postmul(kk, cpx<T>{v.x, -v.y}, this->scale);
    }
};

// Longer convolutions, m = n1*n2, in three passes over an n1 x n2 matrix in
// the workspace: the premultiplied, zero-padded columns (FFT over n1, times
// exp(-2 pi i j2 k1/m)); the rows (FFT over n2, spectrum product, inverse FFT,
// times exp(+2 pi i j2 k1/m), in place); the columns back, postmultiplied.
// Three launches instead of seven: one transform of 10158 FP64 points, which
// waits for launches and not for memory, 40.5 -> 26 us.
// The spectrum is stored in the order the rows meet it, [k1][k2].
template <typename T, int PASS>
struct IOBlueL {
    static constexpr bool pre_lds = false, post_lds = false, store_loads = true, conv = PASS == 2;
    static const char* tag() { return PASS == 1 ? "blueA" : PASS == 2 ? "blueB" : "blueC"; }
    std::string desc() const { return ",n1=" + std::to_string(n1) + ",n2=" + std::to_string(n2); }
    const cpx<T>* in;
    cpx<T>* out;
    cpx<T>* ws;
    Chirp<T> c;
    const cpx<T>* hi;
    const cpx<T>* lo;
    int64_t nlines, n1, n2;
    T scale;
    bool xcd;
    LineDiv div;  // by the lines of a transform
    struct At {
        int64_t x, w;  // offsets of the transform's data and matrix
        int64_t q;     // column j2 (passes 1, 3) or row k1 (pass 2)
    };
    __device__ __forceinline__ At base(int64_t l) const {
        const int64_t b = div(l);
        return At{b * c.n, b * n1 * n2, l - b * div.n0};
    }
    __device__ __forceinline__ cpx<T> load(At a, int k, int rm) const {
        if constexpr (PASS == 1)
            return c.premul((a.q + k * n2) + rm * n2, [&](int64_t kk) { return in[a.x + kk]; });
        else if constexpr (PASS == 2) return ws[(a.w + a.q * n2 + k) + rm];
        else return ws[(a.w + a.q + k * n2) + rm * n2];
    }
    __device__ __forceinline__ cpx<T> spec(At a, int k, int rm) const { return c.spec(a.q * n2 + k + rm); }
    __device__ __forceinline__ void store(At a, int k, int rm, cpx<T> v) const {
        if constexpr (PASS == 1) {
            ws[(a.w + a.q + k * n2) + rm * n2] = cmul(v, tw2<-1>(hi, lo, a.q * k + a.q * rm));
        } else if constexpr (PASS == 2) {
            ws[(a.w + a.q * n2 + k) + rm] = cmul(cpx<T>{v.x, -v.y}, tw2<1>(hi, lo, a.q * k + a.q * rm));
        } else {
            const int64_t kk = (a.q + k * n2) + rm * n2;
            if (kk < c.n) out[a.x + kk] = c.postmul(kk, v, scale);
        }
    }
    template <int CN, int CTL>
    __device__ void pre(int64_t, At, T*, T*, int, int) const {}
    template <int CN, int CTL>
    __device__ void post(int64_t, At, const T*, const T*, int, int) const {}
};

// realForward post pass (reference: CommonUtils.rftfsub :5750-5776 and the
// fold at DoubleFFT_1D.java:543-545).  The line holds the N-point complex FFT
// Z of the 2N reals taken pairwise; the packed result is
//   a[0] = X_0, a[1] = X_N, a[2k], a[2k+1] = Re, Im X_k  (0 < k < N),
// with X_k = (Z_k + conj Z_{N-k})/2 - i w^k (Z_k - conj Z_{N-k})/2,
// w = exp(-2 pi i/2N).  rtw[k] = w^k for k in [0, N/2].
template <typename T>
struct IOR2C {
    static constexpr bool pre_lds = false, post_lds = true, store_loads = false, conv = false;
    static const char* tag() { return "r2c"; }
    std::string desc() const { return ",es=" + std::to_string(m.es); }
    const cpx<T>* in;  // reals viewed as complex pairs
    T* out;            // packed reals
    const cpx<T>* rtw;
    LineMap m;  // in complex units; es must be 1
    int64_t nlines;
    int N;
    T scale;
    bool xcd;
    __device__ __forceinline__ int64_t base(int64_t l) const { return m.base(l); }
    __device__ __forceinline__ cpx<T> load(int64_t b, int k, int rm) const { return in[b + k + rm]; }
    __device__ void store(int64_t, int, int, cpx<T>) const {}
    template <int CN, int CTL>
    __device__ void pre(int64_t, int64_t, T*, T*, int, int) const {}
    template <int CN, int CTL>
    __device__ void post(int64_t, int64_t b, const T* re, const T* im, int t, int nt) const {
        // a[2k], a[2k+1] = Re, Im X_k are one complex store at o[k]
        cpx<T>* o = reinterpret_cast<cpx<T>*>(out + 2 * b);
        const T h = T(0.5) * scale;
        if (t == 0) {
            T zr = re[lpos(0)], zi = im[lpos(0)];
            o[0] = cpx<T>{(zr + zi) * scale, (zr - zi) * scale};
        }
        const int n = CN > 0 ? CN : N;
        const int step = CTL > 0 ? CTL : nt;
        // k = 1 .. n/2, with compile-time trip counts when CN, CTL are known
        constexpr int ITER = (CN > 0 && CTL > 0) ? (CN / 2 + CTL - 1) / CTL : 4;
        for (int k0 = 1 + t; k0 <= n / 2; k0 += ITER * step) {
#pragma unroll
            for (int i = 0; i < ITER; i++) {
                const int k = k0 + i * step;
                if (k > n / 2) break;
                const int kk = n - k;
                cpx<T> A = {re[lpos(k)], im[lpos(k)]};
                cpx<T> B = {re[lpos(kk)], -im[lpos(kk)]};  // conj Z_{N-k}
                cpx<T> fe = cadd(A, B);
                cpx<T> d = csub(A, B);
                cpx<T> fo = {d.y, -d.x};  // -i * d
                cpx<T> wf = cmul(rtw[k], fo);
                // X_k = (fe + w^k fo)/2 ; X_{N-k} = conj(fe - w^k fo)/2
                o[k] = cpx<T>{(fe.x + wf.x) * h, (fe.y + wf.y) * h};
                if (kk != k) o[kk] = cpx<T>{(fe.x - wf.x) * h, -(fe.y - wf.y) * h};
            }
        }
    }
};

// realInverse pre pass (reference: CommonUtils.rftbsub :5806-5831 and
// DoubleFFT_1D.java:946-989).  From the packed half spectrum X of 2N reals it
// builds Z_k = E_k + i O_k with E_k = X_k + conj X_{N-k} and
// O_k = (X_k - conj X_{N-k}) exp(+2 pi i k/2N); the N-point backward FFT of Z
// is sum-normalised (x_{2m} + i x_{2m+1}) * 2N, stored times `scale`.
template <typename T>
struct IOC2R {
    static constexpr bool pre_lds = true, post_lds = false, store_loads = false, conv = false;
    static const char* tag() { return "c2r"; }
    std::string desc() const { return ",es=" + std::to_string(m.es); }
    const T* in;     // packed reals
    cpx<T>* out;     // reals viewed as complex pairs
    const cpx<T>* rtw;
    LineMap m;
    int64_t nlines;
    int N;
    T scale;
    bool xcd;
    __device__ __forceinline__ int64_t base(int64_t l) const { return m.base(l); }
    __device__ cpx<T> load(int64_t, int, int) const { return cpx<T>{T(0), T(0)}; }
    __device__ __forceinline__ void store(int64_t b, int k, int rm, cpx<T> v) const {
        out[b + k + rm] = cpx<T>{v.x * scale, v.y * scale};
    }
    // Z_k and Z_{N-k} from X_k, X_{N-k} (k in (0, N/2]); Z_0 from X_0, X_N
    __device__ __forceinline__ void c2r_pair(int k, cpx<T> Xk, cpx<T> Xn, T* re, T* im) const {
        int kk = N - k;
        cpx<T> Xc = {Xn.x, -Xn.y};  // conj X_{N-k}
        cpx<T> E = cadd(Xk, Xc);
        cpx<T> D = csub(Xk, Xc);
        cpx<T> w = {rtw[k].x, -rtw[k].y};  // exp(+2 pi i k/2N)
        cpx<T> O = cmul(D, w);
        // Z_k = E + i O
        re[lpos(k)] = E.x - O.y;
        im[lpos(k)] = E.y + O.x;
        if (kk != k) {
            // E_{N-k} = conj E_k and O_{N-k} = conj O_k, so Z_{N-k} = conj E + i conj O
            re[lpos(kk)] = E.x + O.y;
            im[lpos(kk)] = O.x - E.y;
        }
    }
    template <int CN, int CTL>
    __device__ void pre(int64_t, int64_t b, T* re, T* im, int t, int nt) const {
        const T* a = in + 2 * b;
        if (t == 0) {
            T x0 = a[0], xn = a[1];
            // E_0 = X_0 + X_N, O_0 = X_0 - X_N
            re[lpos(0)] = x0 + xn;
            im[lpos(0)] = x0 - xn;
        }
        if constexpr (CN > 0) {
            // all loads first (compile-time trip count), then the LDS writes
            constexpr int IT = (CN / 2 + CTL - 1) / CTL;
            cpx<T> xk[IT], xn[IT];
#pragma unroll
            for (int q = 0; q < IT; q++) {
                int k = 1 + t + q * CTL;
                if (k <= CN / 2) {
                    xk[q] = cpx<T>{a[2 * k], a[2 * k + 1]};
                    xn[q] = cpx<T>{a[2 * (CN - k)], a[2 * (CN - k) + 1]};
                }
            }
#pragma unroll
            for (int q = 0; q < IT; q++) {
                int k = 1 + t + q * CTL;
                if (k <= CN / 2) c2r_pair(k, xk[q], xn[q], re, im);
            }
        } else {
            // a few points at a time, their loads issued together
            constexpr int IT = 4;
            for (int k0 = 1 + t; k0 <= N / 2; k0 += IT * nt) {
                cpx<T> xk[IT], xn[IT];
#pragma unroll
                for (int q = 0; q < IT; q++) {
                    const int k = k0 + q * nt;
                    if (k <= N / 2) {
                        xk[q] = cpx<T>{a[2 * k], a[2 * k + 1]};
                        xn[q] = cpx<T>{a[2 * (N - k)], a[2 * (N - k) + 1]};
                    }
                }
#pragma unroll
                for (int q = 0; q < IT; q++) {
                    const int k = k0 + q * nt;
                    if (k <= N / 2) c2r_pair(k, xk[q], xn[q], re, im);
                }
            }
        }
    }
    template <int CN, int CTL>
    __device__ void post(int64_t, int64_t, const T*, const T*, int, int) const {}
};

}  // namespace jt
