// Ragged batches, the form of one launch per pass: every kind of work item
// (whole lines, four-step columns and rows, Bluestein's phases) is a kernel of
// its own over the items of all lengths, and the launches follow each other on
// the stream, so a later phase needs no waits.
//
// Bound: HBM.  Against the persistent kernel (jt_ragged.hpp) an item here runs
// the runtime-radix engine's direct first and last stages and composite
// radices, with the code of one item kind only in the instruction cache and
// registers; it pays for that with the idle tail of up to seven launches.
#pragma once
#include <algorithm>
#include <functional>
#include <map>

#include "jt_fft1d.hpp"

namespace jt {

enum PKind { PK_SINGLE = 0, PK_FOUR_A, PK_FOUR_B, PK_BLUE_S, PK_BLUE_1, PK_BLUE_2, PK_BLUE_3, PK_COUNT };

// A distinct length.
struct PLen {
    int64_t n, n1, n2;      // the length; four-step split (of n, or of m for Bluestein)
    int64_t hi, lo;         // four-step twiddles, offsets into the table
    int64_t choff, bsoff;   // Bluestein chirp and spectrum
};
// A workgroup's work: cnt lines from c0 (transforms listed from tlist[c0], or
// columns / rows of transform tr).
struct PItem {
    int plan, len, c0, cnt;
    int64_t tr;
};

template <typename T>
struct PArgs {
    cpx<T>* data;
    cpx<T>* ws;
    const PLen* lens;
    const GenPlan* plans;
    const cpx<T>* tab;
    const int64_t* off;    // complex offset of each transform
    const int64_t* wsoff;  // workspace offset of each transform
    const int64_t* tlist;
    int inv, scaled;
};

// Whole lines, listed.
template <typename T>
struct IOListed {
    static constexpr bool pre_lds = false, post_lds = false, store_loads = false, conv = false;
    cpx<T>* data;
    const int64_t* off;
    const int64_t* tl;
    T scale;
    __device__ __forceinline__ int64_t base(int64_t l) const { return off[tl[l]]; }
    __device__ __forceinline__ cpx<T> load(int64_t b, int k, int rm) const { return data[b + k + rm]; }
    __device__ __forceinline__ void store(int64_t b, int k, int rm, cpx<T> v) const {
        data[b + k + rm] = cpx<T>{v.x * scale, v.y * scale};
    }
    template <int CN, int CTL>
    __device__ void pre(int64_t, int64_t, T*, T*, int, int) const {}
    template <int CN, int CTL>
    __device__ void post(int64_t, int64_t, const T*, const T*, int, int) const {}
};

// Whole Bluestein lines, listed.
template <typename T>
struct IOListedBlue : IOListed<T> {
    static constexpr bool store_loads = true, conv = true;
    Chirp<T> c;
    __device__ __forceinline__ cpx<T> load(int64_t b, int k, int rm) const {
        return c.premul(k + rm, [&](int64_t kk) { return this->data[b + kk]; });
    }
    __device__ __forceinline__ cpx<T> spec(int64_t, int k, int rm) const { return c.spec(k + rm); }
    __device__ __forceinline__ void store(int64_t b, int k, int rm, cpx<T> v) const {
        const int64_t kk = k + rm;
        if (kk < c.n) this->data[b + kk] = c.postmul(kk, cpx<T>{v.x, -v.y}, this->scale);
    }
};

// DIR: the transform's direction (Bluestein's passes run their own, and take
// it as the chirp's sign).
template <typename T, int KIND, int DIR>
__global__ void __launch_bounds__(1024) ragged_pass(PArgs<T> a, const PItem* __restrict__ items) {
    ro_ptr<PItem> it = ro(items) + (KIND == PK_SINGLE || KIND == PK_BLUE_S ? (int64_t)blockIdx.x
                                                                           : xcd_group(blockIdx.x, gridDim.x));
    ro_ptr<PLen> L = ro(a.lens) + it->len;
    ro_ptr<GenPlan> P = ro(a.plans) + it->plan;
    const int64_t n = L->n, n1 = L->n1, n2 = L->n2;
    const T scale = a.scaled ? T(1) / T(n) : T(1);
    const Chirp<T> c{a.tab + L->choff, a.tab + L->bsoff, n, T(a.inv ? 1 : -1)};
    const cpx<T>* hi = a.tab + L->hi;
    const cpx<T>* lo = a.tab + L->lo;
    int64_t line0 = it->c0;
    cpx<T>* x = nullptr;
    cpx<T>* w = nullptr;
    if constexpr (KIND != PK_SINGLE && KIND != PK_BLUE_S) {
        x = a.data + ro(a.off)[it->tr];
        w = a.ws + ro(a.wsoff)[it->tr];
    }
    auto run = [&](auto io, auto dir) {
        gen_lines<T, decltype(dir)::value>(io, a.tab, P, P->nst, P->n, P->W, P->lgW, P->pitch, P->col != 0, line0,
                                           it->cnt);
    };
    using D = std::integral_constant<int, DIR>;
    using Fwd = std::integral_constant<int, -1>;
    using Inv = std::integral_constant<int, 1>;
    if constexpr (KIND == PK_SINGLE) run(IOListed<T>{a.data, a.off, a.tlist, scale}, D{});
    else if constexpr (KIND == PK_BLUE_S)
        run(IOListedBlue<T>{{a.data, a.off, a.tlist, scale}, c}, Fwd{});
    else if constexpr (KIND == PK_FOUR_A)
        run(IOFourA<T, DIR>{x, w, hi, lo, n2, n, n1, n2, n1, 1, true, LineDiv(n2, n2)}, D{});
    else if constexpr (KIND == PK_FOUR_B)
        run(IOStrided<T>{w, x, LineMap{n1, n1, 1, 0, n1}, n1, scale, true}, D{});
    else if constexpr (KIND == PK_BLUE_1)
        run(IOBlueL<T, 1>{x, x, w, c, hi, lo, n2, n1, n2, scale, true, LineDiv(n2, n2)}, Fwd{});
    else if constexpr (KIND == PK_BLUE_2)
        run(IOBlueL<T, 2>{x, x, w, c, hi, lo, n1, n1, n2, scale, true, LineDiv(n1, n1)}, Fwd{});
    else
        run(IOBlueL<T, 3>{x, x, w, c, hi, lo, n2, n1, n2, scale, true, LineDiv(n2, n2)}, Inv{});
}

template <typename T>
struct RaggedPasses {
    struct Launch {
        int kind, nt;
        size_t shm;
        int64_t first, count;  // items
    };
    std::vector<Launch> launches;
    DevBuf lens, plans, tab, items, off, wsoff, tlist, ws;
};

inline const char* pass_name(int kind) {
    static const char* names[PK_COUNT] = {"lines", "fourA", "fourB", "blue", "blueA", "blueB", "blueC"};
    return names[kind];
}

// Workgroups: up to PASS_POINTS points in PASS_NT threads, two to a CU; lines
// that need more threads (FP32, above 4096 points) take launches of their own.
// 4000 and 300 FP64 transforms of 16 to 65536 points, both directions, us:
// 4096 points in 512 threads 1560 and 278, in 256 threads 1839 and 398, 2048
// in 256 1671 and 336, 2048 in 512 2071 and 358, 1024 in 128 1753 and 339.
// (Rounds of transforms through one workspace of 16 to 128 MiB, for the
// last-level cache, lose more to each launch's tail than they save: 4114 to
// 1837 against 1681 in one round, all with 2048 points.)
constexpr int PASS_NT = 512, PASS_POINTS = 4096;

// The kernel of a pass: Bluestein's are the same in both directions.
template <typename T, int KIND>
auto pass_kernel(bool inv) {
    return inv ? ragged_pass<T, KIND, KIND >= PK_BLUE_S ? -1 : 1> : ragged_pass<T, KIND, -1>;
}

template <typename T, int KIND>
void pass_go(const PArgs<T>& a, const typename RaggedPasses<T>::Launch& l, const PItem* items, hipStream_t st) {
    hipLaunchKernelGGL((pass_kernel<T, KIND>(a.inv != 0)), dim3((unsigned)l.count), dim3(l.nt), l.shm,
                       st, a, items + l.first);
    JT_HIP(hipGetLastError());
}

// Raises the LDS limits of a kind's kernels (at plan creation: a plan's first
// launch may be under stream capture).
template <typename T, int KIND>
void pass_limits() {
    for (int inv = 0; inv < 2; inv++)
        JT_HIP(hipFuncSetAttribute((const void*)pass_kernel<T, KIND>(inv != 0),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
}
template <typename T>
void passes_limits() {
    pass_limits<T, PK_SINGLE>();
    pass_limits<T, PK_FOUR_A>();
    pass_limits<T, PK_FOUR_B>();
    pass_limits<T, PK_BLUE_S>();
    pass_limits<T, PK_BLUE_1>();
    pass_limits<T, PK_BLUE_2>();
    pass_limits<T, PK_BLUE_3>();
}

template <typename T>
void passes_launch(const RaggedPasses<T>& R, cpx<T>* data, int dir, bool scaled, const std::string& label,
                   hipStream_t st) {
    const PArgs<T> a{data, R.ws.template as<cpx<T>>(), R.lens.template as<PLen>(), R.plans.template as<GenPlan>(),
                     R.tab.template as<cpx<T>>(), R.off.template as<int64_t>(), R.wsoff.template as<int64_t>(),
                     R.tlist.template as<int64_t>(), dir > 0 ? 1 : 0, scaled ? 1 : 0};
    const PItem* items = R.items.template as<PItem>();
    for (const auto& l : R.launches) {
        JT_PROF(st, label + ",pass=" + pass_name(l.kind) + (l.nt > PASS_NT ? ",wide>" : ">"));
        switch (l.kind) {
            case PK_SINGLE: pass_go<T, PK_SINGLE>(a, l, items, st); break;
            case PK_FOUR_A: pass_go<T, PK_FOUR_A>(a, l, items, st); break;
            case PK_FOUR_B: pass_go<T, PK_FOUR_B>(a, l, items, st); break;
            case PK_BLUE_S: pass_go<T, PK_BLUE_S>(a, l, items, st); break;
            case PK_BLUE_1: pass_go<T, PK_BLUE_1>(a, l, items, st); break;
            case PK_BLUE_2: pass_go<T, PK_BLUE_2>(a, l, items, st); break;
            default: pass_go<T, PK_BLUE_3>(a, l, items, st); break;
        }
    }
}

// Instantiated in jt_ragpass_f64.hip and jt_ragpass_f32.hip.
#define JT_RAGPASS_INST(X, T)           \
    X template void passes_limits<T>(); \
    X template void passes_launch<T>(const RaggedPasses<T>&, cpx<T>*, int, bool, const std::string&, hipStream_t);
JT_RAGPASS_INST(extern, float)
JT_RAGPASS_INST(extern, double)

// Chirp and spectrum of a Bluestein length (natural order): supplied by the
// caller, which may hold them from another plan.
using BlueTables = std::function<void(int64_t n, int64_t m, std::vector<cpx<double>>& chirp, std::vector<cpx<double>>& spec)>;

// Returns null for batches with a length that this form does not cover (a
// four-step factor beyond one workgroup).
template <typename T>
std::unique_ptr<RaggedPasses<T>> make_passes(const int64_t* lengths, int64_t count, const BlueTables& blue) {
    auto R = std::make_unique<RaggedPasses<T>>();
    const int64_t lim = gen_max<T>();
    std::vector<cpx<T>> tab;
    std::vector<GenPlan> plans;
    std::vector<int> plan_nt;
    std::vector<PLen> lens;
    std::vector<int> len_kind;   // PK_SINGLE, PK_FOUR_A, PK_BLUE_S or PK_BLUE_1
    std::vector<int64_t> len_m;  // points of a phase

    std::map<int64_t, GenPlan> stages;  // by line length, twiddles in the table
    auto stages_of = [&](int64_t n) -> GenPlan {
        auto it = stages.find(n);
        if (it != stages.end()) return it->second;
        const std::vector<int> r = gen_radices(n);
        std::vector<int> offs;
        const std::vector<cpx<T>> tw = stage_twiddles_gen<T>(r, &offs);
        GenPlan g{};
        g.n = (int)n;
        g.nst = (int)r.size();
        int ns = 1;
        for (int i = 0; i < g.nst; i++) {
            const int m = (int)(n / r[i]);
            g.st[i] = GenStage{r[i], m, ns, (int)tab.size() + offs[i], 1.0f / (float)m, 1.0f / (float)ns};
            ns *= r[i];
        }
        tab.insert(tab.end(), tw.begin(), tw.end());
        return stages[n] = g;
    };
    std::map<std::pair<int64_t, int>, int> plan_idx;  // (line length, column mode)
    auto plan_of = [&](int64_t n, bool col) -> int {
        auto key = std::make_pair(n, col ? 1 : 0);
        auto it = plan_idx.find(key);
        if (it != plan_idx.end()) return it->second;
        GenPlan g = stages_of(n);
        int W = 1;
        while (2 * W * n <= PASS_POINTS && W < 64 && gen_threads(g, 2 * W) <= PASS_NT &&
               4 * (size_t)W * gen_pitch((int)n, 2 * W) * sizeof(T) <= 80 * 1024)
            W *= 2;
        const int nt = std::max(gen_threads(g, W), PASS_NT);
        gen_set_shape(g, W, col);
        plans.push_back(g);
        plan_nt.push_back(nt);
        return plan_idx[key] = (int)plans.size() - 1;
    };
    auto four_tables = [&](int64_t n, PLen& L) -> bool {
        const int64_t n1 = four_split<T>(n);
        if (!n1 || n / n1 > lim) return false;
        L.n1 = n1;
        L.n2 = n / n1;
        L.hi = (int64_t)tab.size();
        for (int64_t i = 0; i <= (n >> 8); i++) tab.push_back(expm<T>(i << 8, n));
        L.lo = (int64_t)tab.size();
        for (int64_t i = 0; i < 256; i++) tab.push_back(expm<T>(i, n));
        return true;
    };
    std::map<int64_t, int> len_idx;
    for (int64_t i = 0; i < count; i++) {
        const int64_t n = lengths[i];
        if (len_idx.count(n)) continue;
        PLen L{};
        L.n = n;
        std::vector<int> r;
        if (factor_radices(n, r)) {
            if (n > lim && !four_tables(n, L)) return nullptr;
            len_kind.push_back(n <= lim ? PK_SINGLE : PK_FOUR_A);
            len_m.push_back(n);
        } else {
            const int64_t m = next_smooth(2 * n - 1);
            if (m > lim && !four_tables(m, L)) return nullptr;
            std::vector<cpx<double>> ch, bs;
            blue(n, m, ch, bs);
            L.choff = (int64_t)tab.size();
            for (auto& c : ch) tab.push_back(cpx<T>{(T)c.x, (T)c.y});
            L.bsoff = (int64_t)tab.size();
            const int64_t n1 = m > lim ? L.n1 : 1, n2 = m / n1;
            tab.resize(tab.size() + m);
            for (int64_t k = 0; k < m; k++)  // [k1][k2] of k = k1 + n1*k2
                tab[L.bsoff + (k % n1) * n2 + k / n1] = cpx<T>{(T)bs[k].x, (T)bs[k].y};
            len_kind.push_back(m <= lim ? PK_BLUE_S : PK_BLUE_1);
            len_m.push_back(m);
        }
        len_idx[n] = (int)lens.size();
        lens.push_back(L);
        if ((int64_t)tab.size() > INT32_MAX / 2) return nullptr;
    }

    std::vector<int64_t> off(count), wsoff(count, 0), order(count);
    for (int64_t i = 0, tot = 0; i < count; i++) {
        off[i] = tot;
        tot += lengths[i];
        order[i] = i;
    }
    // transforms largest first, so that a launch ends on small items
    std::stable_sort(order.begin(), order.end(), [&](int64_t a, int64_t b) { return lengths[a] > lengths[b]; });

    std::vector<PItem> items, by_kind[PK_COUNT][2];  // [wide]
    std::vector<int64_t> tlist;
    auto add = [&](int kind, PItem it) { by_kind[kind][plan_nt[it.plan] > PASS_NT].push_back(it); };
    auto lines = [&](int kind, int64_t n, bool col, int len, int64_t tr, int64_t total) {
        const int p = plan_of(n, col);
        const int W = plans[p].W;
        for (int64_t c0 = 0; c0 < total; c0 += W)
            add(kind, PItem{p, len, (int)c0, (int)std::min<int64_t>(W, total - c0), tr});
    };
    // the launches of the collected items, a phase after the one that it reads
    auto flush = [&]() {
        for (int kind : {PK_FOUR_A, PK_BLUE_1, PK_SINGLE, PK_BLUE_S, PK_FOUR_B, PK_BLUE_2, PK_BLUE_3})
            for (int wide : {1, 0}) {
                auto& v = by_kind[kind][wide];
                if (v.empty()) continue;
                size_t shm = 0;
                int nt = 0;
                for (const PItem& it : v) {
                    const GenPlan& g = plans[it.plan];
                    shm = std::max(shm, 2 * (size_t)g.W * g.pitch * sizeof(T));
                    nt = std::max(nt, plan_nt[it.plan]);
                }
                R->launches.push_back({kind, nt, shm, (int64_t)items.size(), (int64_t)v.size()});
                items.insert(items.end(), v.begin(), v.end());
                v.clear();
            }
    };
    int64_t wtot = 0;
    std::vector<int64_t> multi, same;
    for (int64_t q = 0; q < count;) {
        const int64_t n = lengths[order[q]];
        const int l = len_idx[n];
        same.clear();
        for (; q < count && lengths[order[q]] == n; q++) same.push_back(order[q]);
        if (len_kind[l] != PK_SINGLE && len_kind[l] != PK_BLUE_S) {
            multi.insert(multi.end(), same.begin(), same.end());
            continue;
        }
        const int p = plan_of(len_m[l], false);
        const int W = plans[p].W;
        for (size_t c = 0; c < same.size(); c += W) {
            const int cnt = (int)std::min<size_t>(W, same.size() - c);
            add(len_kind[l], PItem{p, l, (int)tlist.size(), cnt, same[c]});
            tlist.insert(tlist.end(), same.begin() + c, same.begin() + c + cnt);
        }
    }
    for (int64_t tr : multi) {
        const int l = len_idx[lengths[tr]];
        const PLen& L = lens[l];
        wsoff[tr] = wtot;
        wtot += len_m[l];
        if (len_kind[l] == PK_FOUR_A) {
            lines(PK_FOUR_A, L.n1, true, l, tr, L.n2);
            lines(PK_FOUR_B, L.n2, true, l, tr, L.n1);
        } else {
            lines(PK_BLUE_1, L.n1, true, l, tr, L.n2);
            lines(PK_BLUE_2, L.n2, false, l, tr, L.n1);
            lines(PK_BLUE_3, L.n1, true, l, tr, L.n2);
        }
    }
    flush();
    passes_limits<T>();
    auto up = [](DevBuf& d, const auto& v) {
        d.alloc(std::max<size_t>(1, v.size()) * sizeof(v[0]));
        if (!v.empty()) JT_HIP(hipMemcpy(d.p, v.data(), v.size() * sizeof(v[0]), hipMemcpyHostToDevice));
    };
    up(R->lens, lens);
    up(R->plans, plans);
    up(R->tab, tab);
    up(R->items, items);
    up(R->off, off);
    up(R->wsoff, wsoff);
    up(R->tlist, tlist);
    R->ws.alloc(std::max<int64_t>(wtot, 1) * sizeof(cpx<T>));
    return R;
}

}  // namespace jt
