// 1D real-data transforms on top of the complex engine: realForward /
// realInverse in the reference's packed layout (DoubleFFT_1D.java:436-561,
// :946-989) and the full-spectrum variants (:678-755, :1112-1195).
#pragma once
#include "jt_fft1d.hpp"
#include "jt_pair.hpp"

namespace jt {

// ---- elementwise helpers ----------------------------------------------------

// packed post pass in place over lines of N complex (= 2N reals), pairs (k, N-k)
template <typename T>
__global__ void r2c_post_inplace(cpx<T>* __restrict__ z, const cpx<T>* __restrict__ rtw, int64_t loff, int64_t N,
                                 int64_t lines, T scale) {
    int64_t half = N / 2 + 1;
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    for (; i < lines * half; i += (int64_t)gridDim.x * blockDim.x) {
        int64_t b = i / half, k = i % half;
        cpx<T>* a = z + b * N;
        if (k == 0) {
            cpx<T> z0 = a[0];
            a[0] = cpx<T>{(z0.x + z0.y) * scale, (z0.x - z0.y) * scale};
            continue;
        }
        int64_t kk = N - k;
        cpx<T> A = a[k];
        cpx<T> Zc = a[kk];
        cpx<T> B = {Zc.x, -Zc.y};
        cpx<T> fe = cadd(A, B), d = csub(A, B);
        cpx<T> fo = {d.y, -d.x};
        cpx<T> wf = cmul(cmul(rtw[k >> 8], rtw[loff + (k & 255)]), fo);
        T h = T(0.5) * scale;
        a[k] = cpx<T>{(fe.x + wf.x) * h, (fe.y + wf.y) * h};
        if (kk != k) a[kk] = cpx<T>{(fe.x - wf.x) * h, -(fe.y - wf.y) * h};
    }
}

// packed pre pass in place (inverse of r2c_post up to the factor 2N)
template <typename T>
__global__ void c2r_pre_inplace(cpx<T>* __restrict__ z, const cpx<T>* __restrict__ rtw, int64_t loff, int64_t N,
                                int64_t lines) {
    int64_t half = N / 2 + 1;
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    for (; i < lines * half; i += (int64_t)gridDim.x * blockDim.x) {
        int64_t b = i / half, k = i % half;
        cpx<T>* a = z + b * N;
        if (k == 0) {
            cpx<T> x = a[0];
            a[0] = cpx<T>{x.x + x.y, x.x - x.y};
            continue;
        }
        int64_t kk = N - k;
        cpx<T> Xk = a[k];
        cpx<T> Xn = a[kk];
        cpx<T> Xc = {Xn.x, -Xn.y};
        cpx<T> E = cadd(Xk, Xc), D = csub(Xk, Xc);
        const cpx<T> wk = cmul(rtw[k >> 8], rtw[loff + (k & 255)]);
        cpx<T> w = {wk.x, -wk.y};
        cpx<T> O = cmul(D, w);
        a[k] = cpx<T>{E.x - O.y, E.y + O.x};
        if (kk != k) a[kk] = cpx<T>{E.x + O.y, O.x - E.y};
    }
}

// reals (line stride n) -> complex with zero imaginary parts (line stride n)
template <typename T>
__global__ void real_to_complex(const T* __restrict__ x, cpx<T>* __restrict__ y, int64_t n,
                                int64_t lines) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    for (; i < lines * n; i += (int64_t)gridDim.x * blockDim.x) y[i] = cpx<T>{x[i], T(0)};
}

template <typename T>
__global__ void copy_complex(const cpx<T>* __restrict__ s, cpx<T>* __restrict__ d, int64_t count) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    for (; i < count; i += (int64_t)gridDim.x * blockDim.x) d[i] = s[i];
}

// ---- real plan ----------------------------------------------------------------

template <typename T>
struct Real1D {
    int64_t n = 0;
    std::unique_ptr<Fft1D<T>> full;  // length n (odd n, *Full ops)
    std::unique_ptr<Fft1D<T>> half;  // length n/2 (even n)
    // w^k = exp(-2 pi i k/n): with a one-pass half plan, w^k for k in
    // [0, n/4 + 1] (the IO hooks of its kernel); otherwise (large n) as two levels,
    // w^k = rtw[k >> 8] * rtw[rlo + (k & 255)] for k in [0, n/4 + 1], so the
    // table stays O(n / 256) long
    DevBuf rtw;
    int64_t rlo = 0;
    int64_t ws_elems(int64_t lines) const {
        int64_t w = 0;
        if (half) w = std::max<int64_t>(w, half->workspace(lines));
        if (full) w = std::max<int64_t>(w, lines * n + full->workspace(lines));
        return w;
    }
};

template <typename T>
std::unique_ptr<Real1D<T>> make_real1d(int64_t n) {
    auto r = std::make_unique<Real1D<T>>();
    r->n = n;
    r->full = make_fft1d<T>(n);
    if (n % 2 == 0 && n >= 2) {
        r->half = make_fft1d<T>(n / 2);
        std::vector<cpx<T>> h;
        if (r->half->single()) {
            h.resize(n / 4 + 2);
            for (int64_t k = 0; k < (int64_t)h.size(); k++) h[k] = expm<T>(k, n);
        } else {
            const int64_t nhi = ((n / 4 + 1) >> 8) + 1;
            for (int64_t i = 0; i < nhi; i++) h.push_back(expm<T>(i << 8, n));
            r->rlo = nhi;
            for (int64_t i = 0; i < 256; i++) h.push_back(expm<T>(i, n));
        }
        upload(r->rtw, h);
    }
    return r;
}

// realForward on `lines` lines of n reals at stride n.
template <typename T>
void real_forward(const Real1D<T>& r, T* a, int64_t lines, cpx<T>* ws, hipStream_t st) {
    const int64_t n = r.n;
    if (n == 1 || lines <= 0) return;
    if (r.half) {
        const int64_t N = n / 2;
        cpx<T>* z = reinterpret_cast<cpx<T>*>(a);
        if (r.half->single()) {
            IOR2C<T> io{z, a, r.rtw.template as<cpx<T>>(), LineMap{lines, lines, N, 0, 1}, lines, (int)N,
                        T(1), false};
            run_single<T, -1, false>(*r.half, io, st);
        } else {
            c2c_contig<T, -1>(*r.half, z, z, lines, T(1), ws, st);
            { JT_PROF(st, "r2c_post_inplace");
            hipLaunchKernelGGL((r2c_post_inplace<T>), ew_grid(lines * (N / 2 + 1)), dim3(256), 0, st, z,
                               r.rtw.template as<cpx<T>>(), r.rlo, N, lines, T(1));
            }
            JT_HIP(hipGetLastError());
        }
        return;
    }
    // odd n (a line per transform)
    pair_lines<T, R2R_PACKED, true>(*r.full, a, nullptr, LineMap{lines, lines, n, 0, 1}, T(1), T(1), ws, st);
}

// Unscaled realInverse returns (n/2) x for powers of two and n x otherwise
// (DoubleFFT_1D.java:965 vs :977/:983).
template <typename T>
inline T real_inverse_factor(int64_t n, bool scale) {
    if (scale) return T(1.0 / (double)n);
    return (is_pow2(n) && n > 1) ? T(0.5) : T(1);
}

template <typename T>
void real_inverse(const Real1D<T>& r, T* a, int64_t lines, bool scale, cpx<T>* ws, hipStream_t st) {
    const int64_t n = r.n;
    if (n == 1 || lines <= 0) return;
    const T f = real_inverse_factor<T>(n, scale);
    if (r.half) {
        const int64_t N = n / 2;
        cpx<T>* z = reinterpret_cast<cpx<T>*>(a);
        if (r.half->single()) {
            IOC2R<T> io{a, z, r.rtw.template as<cpx<T>>(), LineMap{lines, lines, N, 0, 1}, lines, (int)N, f,
                        false};
            run_single<T, 1, false>(*r.half, io, st);
        } else {
            { JT_PROF(st, "c2r_pre_inplace");
            hipLaunchKernelGGL((c2r_pre_inplace<T>), ew_grid(lines * (N / 2 + 1)), dim3(256), 0, st, z,
                               r.rtw.template as<cpx<T>>(), r.rlo, N, lines);
            }
            JT_HIP(hipGetLastError());
            c2c_contig<T, 1>(*r.half, z, z, lines, f, ws, st);
        }
        return;
    }
    // the backward sum is n x; unscaled non-power-of-two result is n x
    pair_lines<T, R2R_PACKED, false>(*r.full, a, nullptr, LineMap{lines, lines, n, 0, 1}, T(1),
                                     scale ? T(1.0 / (double)n) : T(1), ws, st);
}

// One launch from lines of n reals to their complex transforms, for a plan of
// one launch.  A single line may be transformed onto itself (a workgroup has
// read its lines before it writes).
template <typename T, int DIR>
void real_rows(const Fft1D<T>& p, const T* in, cpx<T>* out, int64_t lines, T scale, hipStream_t st) {
    const IORealRows<T> io{in, out, p.n, lines, scale, false};
    if (p.blue_single()) {
        const Chirp<T> c{p.chirp.template as<cpx<T>>(), p.bspec.template as<cpx<T>>(), p.n, T(DIR)};
        go_gen<T, -1>(*p.pm, IORealRowsBlue<T>{io, c}, false, st);
    } else {
        run_single<T, DIR, false>(p, io, st);
    }
}

// realForwardFull / realInverseFull: complex transform of the real input
// a[0..n) written as 2n values (dir -1 forward, +1 inverse with scale).
template <typename T, int DIR>
void real_full(const Real1D<T>& r, T* a, bool scale, cpx<T>* ws, hipStream_t st) {
    const int64_t n = r.n;
    const T s = (DIR > 0 && scale) ? T(1.0 / (double)n) : T(1);
    cpx<T>* z = reinterpret_cast<cpx<T>*>(a);
    if (r.full->one_launch()) {
        real_rows<T, DIR>(*r.full, a, z, 1, s, st);
        return;
    }
    need_ws(ws);
    { JT_PROF(st, "real_to_complex");
    hipLaunchKernelGGL((real_to_complex<T>), ew_grid(n), dim3(256), 0, st, a, ws, n, (int64_t)1);
    }
    JT_HIP(hipGetLastError());
    c2c_contig<T, DIR>(*r.full, ws, z, 1, s, ws + n, st);
}

// Instantiated in jt_full_f64.hip and jt_full_f32.hip.
#define JT_FULL_INST1(X, T, D)                                                                            \
    X template void real_rows<T, D>(const Fft1D<T>&, const T*, cpx<T>*, int64_t, T, hipStream_t);          \
    X template void real_full<T, D>(const Real1D<T>&, T*, bool, cpx<T>*, hipStream_t);
#define JT_FULL_INST(X, T) JT_FULL_INST1(X, T, -1) JT_FULL_INST1(X, T, 1)
JT_FULL_INST(extern, float)
JT_FULL_INST(extern, double)

}  // namespace jt
