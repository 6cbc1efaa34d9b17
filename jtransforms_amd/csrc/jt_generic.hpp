// Runtime-radix Stockham kernel: one workgroup transforms W lines, the radices
// come from the kernel arguments.
//
// Bound: HBM (or the last-level cache) for axes that fill the chip, latency of
// the stage chain below that.  Layout, against one line per workgroup in two
// LDS buffers with a copy in and a copy out (as this kernel first was):
//   - W adjacent lines per workgroup with lanes across them, so that a strided
//     axis is read and written in 64- to 128-byte segments, not 16-byte ones;
//   - the first stage reads and the last one writes memory directly, the inner
//     ones run in place in LDS: one buffer, one LDS trip per stage boundary;
//   - composite radices 6, 9, 10, 12, 14, 15: 180 = 15 * 12 takes two stages
//     instead of three, 1080 = 9 * 10 * 12 three instead of five;
//   - twiddles laid out along jm, so that lanes read consecutive entries.
// Measured per axis pass (FP64 180^3: 187 MB; FP32 1080 x 1920: 33 MB):
//   180^3 strided axes 200-207 -> 33 us (5.7 TB/s), contiguous 100 -> 38 us;
//   1080-point columns 64 -> 15 us, 1920-point rows 24 -> 13 us.  Serves all lengths that have no
// compile-time kernel: the mixed-radix sizes of the reference's FFTPACK path
// (DoubleFFT_1D.java:6630-8008) and the sub-lengths of the four-step and
// Bluestein plans.
#pragma once
#include "jt_dft.hpp"

namespace jt {

constexpr int GEN_MAX_STAGES = 20;

// Stages of the runtime-radix kernel: radices up to 16, composite ones among
// them, so a length up to 8192 takes at most GEN_STAGES of them (5 for 5^5).
constexpr int GEN_STAGES = 6;

struct GenStage {
    int radix;
    int m;      // n / radix: butterflies per line
    int ns;     // product of the earlier radices
    int twoff;  // twiddles of the stage: (r-1)*ns + jm from here
    float rm, rns;
};

struct GenPlan {
    GenStage st[GEN_STAGES];
    int n;
    int nst;
    // the launch's shape
    int W;      // lines per workgroup (a power of two in column mode)
    int lgW;    // log2 W (column mode)
    int pitch;  // LDS elements from line to line
    int col;    // lanes across adjacent lines (1) or along a line (0)
};

__device__ __forceinline__ int gpos(int k) { return k + (k >> 5); }

// q = a / d for 0 <= a < 2^22, d >= 1, from a float reciprocal with one
// correction step (exact: the float quotient a*(1/d) is within 3*2^-24 a/d
// of the true one, i.e. within 1 for these ranges)
__device__ __forceinline__ int fdiv(int a, int d, float rcp) {
    int q = (int)((float)a * rcp);
    int r = a - q * d;
    if (r < 0) q--;
    else if (r >= d) q++;
    return q;
}

// cos / sin (2 pi m / P), m = 0..P-1, for the prime radices 11 and 13
template <int P>
struct PrimeTw;
template <>
struct PrimeTw<11> {
    static constexpr double C[11] = {1.0, 0.841253532831181168862, 0.415415013001886425529,
                                     -0.142314838273285140444, -0.654860733945285064057, -0.95949297361449738989,
                                     -0.95949297361449738989, -0.654860733945285064057, -0.142314838273285140444,
                                     0.415415013001886425529, 0.841253532831181168862};
    static constexpr double S[11] = {0.0, 0.540640817455597582108, 0.909631995354518371412,
                                     0.989821441880932732376, 0.755749574354258283774, 0.281732556841429697711,
                                     -0.281732556841429697711, -0.755749574354258283774, -0.989821441880932732376,
                                     -0.909631995354518371412, -0.540640817455597582108};
};
template <>
struct PrimeTw<13> {
    static constexpr double C[13] = {1.0, 0.8854560256532098959, 0.568064746731155802512,
                                     0.120536680255323053349, -0.35460488704253562597, -0.748510748171101098635,
                                     -0.970941817426052027157, -0.970941817426052027157, -0.748510748171101098635,
                                     -0.35460488704253562597, 0.120536680255323053349, 0.568064746731155802512,
                                     0.8854560256532098959};
    static constexpr double S[13] = {0.0, 0.464723172043768545656, 0.82298386589365639458,
                                     0.992708874098053992801, 0.93501624268541482344, 0.663122658240795202377,
                                     0.239315664287557767149, -0.239315664287557767149, -0.663122658240795202377,
                                     -0.93501624268541482344, -0.992708874098053992801, -0.82298386589365639458,
                                     -0.464723172043768545656};
};

// Prime radix P (11, 13), X_k = sum_j v_j exp(DIR 2 pi i jk/P), by pairing
// j with P-j: with a_j = v_j + v_{P-j}, b_j = v_j - v_{P-j} (j = 1..H,
// H = (P-1)/2) and m = jk mod P,
//   X_0     = v_0 + sum a_j
//   X_k     = v_0 + sum a_j C_m + i DIR sum b_j S_m
//   X_{P-k} = v_0 + sum a_j C_m - i DIR sum b_j S_m       (k = 1..H)
// All indices are compile-time constants after unrolling.
template <int P, int DIR, typename T>
__device__ __forceinline__ void dft_prime(cpx<T>* v) {
    constexpr int H = (P - 1) / 2;
    cpx<T> a[H + 1], b[H + 1];
    cpx<T> x0 = v[0];
#pragma unroll
    for (int j = 1; j <= H; j++) {
        a[j] = cadd(v[j], v[P - j]);
        b[j] = csub(v[j], v[P - j]);
        x0 = cadd(x0, a[j]);
    }
#pragma unroll
    for (int k = 1; k <= H; k++) {
        T re = v[0].x, im = v[0].y, sr = T(0), si = T(0);
#pragma unroll
        for (int j = 1; j <= H; j++) {
            const T c = (T)PrimeTw<P>::C[(j * k) % P];
            const T sn = (T)PrimeTw<P>::S[(j * k) % P];
            re += a[j].x * c;
            im += a[j].y * c;
            sr += b[j].y * sn;
            si += b[j].x * sn;
        }
        // i DIR (b S) = DIR (-(b.y S), b.x S)
        v[k] = cpx<T>{re - T(DIR) * sr, im + T(DIR) * si};
        v[P - k] = cpx<T>{re + T(DIR) * sr, im - T(DIR) * si};
    }
    v[0] = x0;
}

template <int R, int DIR, typename T>
__device__ __forceinline__ void dft_any(cpx<T>* v) {
    if constexpr (R == 11 || R == 13) dft_prime<R, DIR>(v);
    else dft<R, DIR>(v);
}

// Points a thread holds across the barrier of an in-place stage.
constexpr int GEN_PTS = 16;
constexpr int gen_butterflies(int R) { return GEN_PTS / R > 0 ? GEN_PTS / R : 1; }

// One Stockham stage of radix R over the workgroup's W lines.  Butterfly
// (line w, j) belongs to thread (idx = its place in the flattened order) mod
// NT: column mode orders j-major (lanes across the W adjacent lines), row
// mode line-major (lanes along the line), so every global access of a first or
// last stage is coalesced.  FROMG: the inputs come through io.load; else from
// LDS.  TOG: the outputs go through io.store; else to LDS, in place (all
// inputs are in registers before the barrier that precedes the first write;
// the host sizes NT so that gen_butterflies(R) per thread cover the stage).
// SPEC: each output k is multiplied by io.spec(at, k) and conjugated (the
// middle of a convolution).
template <int R, int DIR, bool FROMG, bool TOG, bool SPEC, typename T, class IO>
__device__ __forceinline__ void gen_stage(const IO& io, GenStage S, int W, int lgW, int pitch, bool col,
                                          const cpx<T>* __restrict__ tw, T* re, T* im, int64_t line0, int nl,
                                          int tid) {
    constexpr int NB = gen_butterflies(R);
    const int NT = blockDim.x;
    const int m = S.m, ns = S.ns;
    cpx<T> v[NB][R];
    int jj[NB], ww[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int idx = tid + b * NT;
        int w, j;
        if (col) {
            w = idx & (W - 1);
            j = idx >> lgW;
        } else {
            w = fdiv(idx, m, S.rm);
            j = idx - w * m;
        }
        jj[b] = (w < nl && j < m) ? j : -1;
        ww[b] = w;
        if (jj[b] >= 0) {
            if constexpr (FROMG) {
                const auto at = io.base(line0 + w);
#pragma unroll
                for (int r = 0; r < R; r++) v[b][r] = io.load(at, j, r * m);
            } else {
                const T* lr = re + w * pitch;
                const T* li = im + w * pitch;
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const int k = gpos(j + r * m);
                    v[b][r] = cpx<T>{lr[k], li[k]};
                }
            }
        }
    }
    if constexpr (!FROMG && !TOG) __syncthreads();
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int j = jj[b];
        if (j >= 0) {
            int jh = j, jm = 0;
            if (!FROMG && ns > 1) {
                jh = fdiv(j, ns, S.rns);
                jm = j - jh * ns;
                const cpx<T>* t = tw + S.twoff + jm;
#pragma unroll
                for (int r = 1; r < R; r++) v[b][r] = cmul(v[b][r], tw_dir<DIR>(t[(r - 1) * ns]));
            }
            dft_any<R, DIR>(v[b]);
            if constexpr (TOG) {
                const auto at = io.base(line0 + ww[b]);
#pragma unroll
                for (int r = 0; r < R; r++) {
                    io.store(at, j, r * m, v[b][r]);
                    // a store that loads factors of its own: a few at a time,
                    // or their registers spill
                    if constexpr (IO::store_loads)
                        if (r % (sizeof(T) == 8 ? 2 : 4) == 1) __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                T* lr = re + ww[b] * pitch;
                T* li = im + ww[b] * pitch;
                const int d = jh * ns * R + jm;
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const int k = gpos(d + r * ns);
                    if constexpr (SPEC) {
                        const cpx<T> p = cmul(v[b][r], io.spec(io.base(line0 + ww[b]), d, r * ns));
                        v[b][r] = cpx<T>{p.x, -p.y};
                        if (sizeof(T) == 8 || r % 2 == 1) __builtin_amdgcn_sched_barrier(0);
                    }
                    lr[k] = v[b][r].x;
                    li[k] = v[b][r].y;
                }
            }
        }
    }
}

template <int DIR, bool FROMG, bool TOG, bool SPEC = false, typename T, class IO>
__device__ __forceinline__ void gen_stage_rt(const IO& io, GenStage S, int W, int lgW, int pitch, bool col,
                                             const cpx<T>* __restrict__ tw, T* re, T* im, int64_t line0, int nl,
                                             int tid) {
    // an empty asm that "changes" the thread index: a stage's addresses are
    // then computed inside the stage instead of being hoisted over the switch
    asm volatile("" : "+v"(tid));
    switch (S.radix) {
#define JT_GEN_CASE(R) \
    case R: gen_stage<R, DIR, FROMG, TOG, SPEC>(io, S, W, lgW, pitch, col, tw, re, im, line0, nl, tid); break;
        JT_GEN_CASE(2)
        JT_GEN_CASE(3)
        JT_GEN_CASE(4)
        JT_GEN_CASE(5)
        JT_GEN_CASE(6)
        JT_GEN_CASE(7)
        JT_GEN_CASE(8)
        JT_GEN_CASE(9)
        JT_GEN_CASE(10)
        JT_GEN_CASE(11)
        JT_GEN_CASE(12)
        JT_GEN_CASE(13)
        JT_GEN_CASE(14)
        JT_GEN_CASE(15)
        JT_GEN_CASE(16)
#undef JT_GEN_CASE
        default: break;
    }
}

// Map workgroup id to line group so that consecutive groups (adjacent in
// memory) land on the same XCD (workgroups are dispatched round-robin over
// the 8 XCDs); keeps partial cache lines of neighbouring groups in one L2.
__device__ __forceinline__ int64_t xcd_group(int64_t bid, int64_t ngroups) {
    const int64_t nx = 8;
    int64_t per = ngroups / nx;
    int64_t full = per * nx;
    if (bid >= full) return bid;
    return (bid % nx) * per + bid / nx;
}

// Read-only tables of a plan are read through the constant address space: the
// compiler then knows that the kernel's stores never change them, so their
// loads are hoisted and batched across stores, and loads at a wave-uniform
// address become scalar loads.
template <class X>
using ro_ptr = const __attribute__((address_space(4))) X*;
template <class X>
__device__ __forceinline__ ro_ptr<X> ro(const X* p) { return (ro_ptr<X>)p; }
__device__ __forceinline__ GenStage stage_of(const GenPlan& P, int s) { return P.st[s]; }
__device__ __forceinline__ GenStage stage_of(ro_ptr<GenPlan> P, int s) {
    return GenStage{P->st[s].radix, P->st[s].m, P->st[s].ns, P->st[s].twoff, P->st[s].rm, P->st[s].rns};
}

// The lines line0 .. line0+nl-1 (nl <= W) through all stages.  IO contract as
// for stockham_kernel, except that loads and stores name the element as j + rm
// with rm uniform over the workgroup; pre/post hooks work on one line with the
// threads (t, nt) of that line and address LDS through gpos(k).  A policy with
// conv = true runs the transform twice with the spectrum product between:
// out = DFT(conj(spec * DFT(in))), i.e. a cyclic convolution up to a
// conjugation that its store undoes, in one LDS residency (nst >= 2).
// `stages` is the plan's stage list, as a kernel argument or in memory.
template <typename T, int DIR, class IO, class Stages>
__device__ __forceinline__ void gen_lines(const IO& io, const cpx<T>* __restrict__ tw, const Stages& stages, int nst,
                                          int n, int W, int lgW, int pitch, bool col, int64_t line0, int nl) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* re = reinterpret_cast<T*>(smem_raw);
    T* im = re + W * pitch;
    const int tid = threadIdx.x;
    // the hooks' view: line hw, thread ht of hn
    int hw = 0, ht = tid, hn = blockDim.x;
    if constexpr (IO::pre_lds || IO::post_lds) {
        hn = blockDim.x / W;
        if (col) {
            hw = tid & (W - 1);
            ht = tid >> lgW;
        } else if (W > 1) {
            hw = tid / hn;
            ht = tid - hw * hn;
        }
    }
    int s = 0;
    if constexpr (IO::pre_lds) {
        if (hw < nl)
            io.template pre<0, 0>(line0 + hw, io.base(line0 + hw), re + hw * pitch, im + hw * pitch, ht, hn);
    } else if (nst > 0) {
        gen_stage_rt<DIR, true, false>(io, stage_of(stages, 0), W, lgW, pitch, col, tw, re, im, line0, nl, tid);
        s = 1;
    } else if (tid < nl) {  // n == 1
        const cpx<T> x = io.load(io.base(line0 + tid), 0, 0);
        re[tid * pitch] = x.x;
        im[tid * pitch] = x.y;
    }
    // (one loop over both transforms of a convolution: with two, the compiler
    // keeps a copy of the stage list in scratch)
    const int all = IO::conv ? 2 * nst : nst;
    const int inner = IO::post_lds ? all : all - 1;
    for (; s < inner; s++) {
        const GenStage S = stage_of(stages, IO::conv && s >= nst ? s - nst : s);
        __syncthreads();
        if constexpr (IO::conv) {
            if (s == nst - 1) {
                gen_stage_rt<DIR, false, false, true>(io, S, W, lgW, pitch, col, tw, re, im, line0, nl, tid);
                continue;
            }
        }
        gen_stage_rt<DIR, false, false>(io, S, W, lgW, pitch, col, tw, re, im, line0, nl, tid);
    }
    __syncthreads();
    if constexpr (IO::post_lds) {
        if (hw < nl)
            io.template post<0, 0>(line0 + hw, io.base(line0 + hw), re + hw * pitch, im + hw * pitch, ht, hn);
    } else if (s < all) {
        gen_stage_rt<DIR, false, true>(io, stage_of(stages, nst - 1), W, lgW, pitch, col, tw, re, im, line0, nl, tid);
    } else {
        // one stage at most: the results are in LDS
        for (int idx = tid; idx < nl * n; idx += blockDim.x) {
            const int w = col ? idx % nl : idx / n, k = col ? idx / nl : idx % n;
            io.store(io.base(line0 + w), k, 0, cpx<T>{re[w * pitch + gpos(k)], im[w * pitch + gpos(k)]});
        }
    }
}

template <typename T, int DIR, class IO>
__global__ void __launch_bounds__(1024) generic_kernel(IO io, const cpx<T>* __restrict__ tw, GenPlan P) {
    const int W = P.W;
    const int64_t ngroups = (io.nlines + W - 1) / W;
    const int64_t bid = blockIdx.x + (int64_t)blockIdx.y * gridDim.x;
    if (bid >= ngroups) return;  // whole workgroup exits together
    const int64_t line0 = (io.xcd ? xcd_group(bid, ngroups) : bid) * W;
    const int nl = (int)(io.nlines - line0 < W ? io.nlines - line0 : W);
    gen_lines<T, DIR>(io, tw, P, P.nst, P.n, W, P.lgW, P.pitch, P.col, line0, nl);
}

}  // namespace jt
