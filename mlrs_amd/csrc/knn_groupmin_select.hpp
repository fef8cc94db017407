// The selection pass of the group-minimum search (knn_groupmin.hpp).  Included
// by the sources that instantiate it, so that the arms compile side by side.
#pragma once

#include "knn_common.hpp"
#include "knn_groupmin.hpp"

namespace mlrs {

namespace {

// ---------------------------------------------------------------------------
// Selection: one workgroup per query.
// ---------------------------------------------------------------------------
constexpr int kSelCap = 1024;    // candidate groups listed before the query falls back to a pass over all of them
constexpr int kSelRefine = 512;  // lists up to this long have their k-th minimum found exactly

// Orders this wave's LDS writes before its later LDS reads by other lanes: the
// LDS serves a wave's accesses in order, so the compiler's order is all.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// 16 bytes of a row that is aligned to its elements only.
template <typename TS> struct RowVec;
template <> struct RowVec<float> {
    static constexpr int V = 4;
    typedef float type __attribute__((ext_vector_type(4), aligned(4)));
};
template <> struct RowVec<double> {
    static constexpr int V = 2;
    typedef double type __attribute__((ext_vector_type(2), aligned(8)));
};

template <typename T, int ARM>
__device__ __forceinline__ void gm_step(T& acc, T& ya, T x, T y, const MetricParams<T>& mp) {
    using F = FloatTraits<T>;
    if (ARM == ARM_EUCLID_FMA) {
        const T diff = x - y;
        acc = F::fma_(diff, diff, acc);
    } else if (ARM == ARM_EUCLID_MULADD) {
        const T diff = x - y;
        acc = acc + diff * diff;
    } else if (ARM == ARM_COS_FOLD) {
        acc = F::fma_(x, y, acc);
        ya = ya + y * y;
    } else if (ARM == ARM_COS_HOST) {
        acc = acc + x * y;
        ya = ya + y * y;
    } else {
        acc = metric_step<T, ARM>(acc, x, y, mp);
    }
}

// The exact value of (query sq, row X[r]), accumulated over ascending columns
// in the arm's order; for cosine ya is the row's row_sumsq.  A lane reads its
// own row, 128 bytes of it in flight: the 64 rows of a wave lie in four runs
// of neighbours, and a line's eight pieces are requested together, so the
// cache serves seven of them.  (Staging the rows through LDS with coalesced
// loads, two barriers per 128 bytes, took three to ten times as long.)
template <typename T, typename TS, int ARM>
__device__ __forceinline__ T gm_exact(const T* __restrict__ sq, const TS* __restrict__ row, int d, T& ya,
                                      const MetricParams<T>& mp) {
    constexpr int V = RowVec<TS>::V;
    constexpr int U = 8;
    typedef typename RowVec<TS>::type vec;
    typedef const __attribute__((address_space(1))) vec* vptr;
    typedef const __attribute__((address_space(1))) TS* sptr;
    T acc = T(0);
    ya = T(0);
    int c = 0;
    for (; c + U * V <= d; c += U * V) {
        vec p[U];
#pragma unroll
        for (int u = 0; u < U; ++u) p[u] = *(vptr)(row + c + u * V);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < V; ++e) gm_step<T, ARM>(acc, ya, sq[c + u * V + e], (T)p[u][e], mp);
    }
    if (c < d) {
        vec p[U];
        TS tail[V];
        const int nv = (d - c) / V, rest = (d - c) % V;  // uniform
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (u < nv) p[u] = *(vptr)(row + c + u * V);
#pragma unroll
        for (int e = 0; e + 1 < V; ++e)
            if (e < rest) tail[e] = *(sptr)(row + c + nv * V + e);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (u < nv) {
#pragma unroll
                for (int e = 0; e < V; ++e) gm_step<T, ARM>(acc, ya, sq[c + u * V + e], (T)p[u][e], mp);
            }
#pragma unroll
        for (int e = 0; e + 1 < V; ++e)
            if (e < rest) gm_step<T, ARM>(acc, ya, sq[c + nv * V + e], (T)tail[e], mp);
    }
    return acc;
}

// The largest minimum a group with a row of the answer can have, from the k-th
// smallest minimum t.  A pair's screen value and exact value (less ||q||^2)
// differ by at most e (||q||^2 + ||x||^2) + e_abs, e = eps_rel.  The bias is
// lowered by e ||x||^2, so a minimum m is at most its row's exact value plus
// eq = e ||q||^2 + e_abs, and the exact value is at most m + eq + 2 e ||x||^2.
// That norm is at most the index's largest, xmax, and, since the row is near,
// at most (||q|| + its distance)^2: one outlier in the index does not widen the
// bound of the others (200k x 5k, d = 128, k = 16, f64, one row a thousand times
// the others' norm: 109 ms with xmax alone, 0.97 with both, as without the row).
// Two estimates of the distance's square D (the exact value's rounding is below
// 2^-12 of it): from ||x||^2 <= 2 (||q||^2 + D) follows D <= (||q||^2 + t + eq +
// 4.01 e ||q||^2) / (1 - 4.01 e), which then gives the norm.
__device__ __forceinline__ float gm_bound(float t, float qn, float xmax, double e, float eq) {
    if (!(t < __builtin_huge_valf())) return __builtin_huge_valf();
    double b = (double)t + 2.0 * (double)eq;
    if (e != 0.0) {
        const double D = fmax(((double)t + (double)qn + (double)eq + 4.01 * e * (double)qn) * (1.0 + 4.1 * e), 0.0);
        const float r = __builtin_sqrtf(qn) + __builtin_sqrtf((float)D);
        b += 2.0 * e * (double)fminf(xmax, 1.002f * r * r);
    }
    return round_up_f(b);
}

// The same for the precise scan's minima, which are distances: |value - exact| <=
// e (||q||^2 + ||x||^2) + e_abs + e_t value, and ||x|| <= ||q|| + the distance.
__device__ __forceinline__ float gm_bound_precise(double v, float qn, float xmax, double e, double e_abs, int sides) {
    double b = v + sides * e_abs;
    if (e != 0.0) {
        const float r = __builtin_sqrtf(qn) + __builtin_sqrtf((float)fmax((v + 5.0 * e * (double)qn) * (1.0 + 5.0 * e), 0.0));
        b += sides * e * ((double)qn + (double)fminf(xmax, 1.002f * r * r));
    }
    return round_up_f(b);
}

// What both selection kernels read of a query.  What an arm's minima cannot be
// is known when it is compiled: METRIC ones are exact, precise ones come with f64
// values only.
template <typename T, typename TS, int ARM>
struct GmQuery {
    static constexpr bool COS = ARM == ARM_COS_FOLD || ARM == ARM_COS_HOST;
    static constexpr bool exact = !COS && ARM != ARM_EUCLID_FMA && ARM != ARM_EUCLID_MULADD;
    static constexpr bool twice = !exact && sizeof(T) == 8;
    __device__ __forceinline__ bool precise() const { return twice && a.kind == GM_PRECISE; }
    const float* G;   // its group minima, [2][ntp]
    int n, ntp;
    uint32_t nt;
    float qn;
    uint32_t nforced;
    bool all_rows;  // a query the screen is not trusted with
    float eps;      // the part of the error that does not depend on the row
    float xmax;
    float base;     // a value and its minimum's unit differ by this
    const GmSelectArgs<TS>& a;
    const float* bias;
    double width;   // bound's distance above its argument, which only shrinks with it
    __device__ __forceinline__ GmQuery(const GmSelectArgs<TS>& args, int64_t q, int64_t i) : a(args), width(0.0) {
        G = a.gmin + i * 2 * a.ntp;
        ntp = (int)a.ntp;
        n = 2 * ntp;  // a multiple of 8
        nt = (uint32_t)a.nt;
        if constexpr (exact) {
            base = 0.0f;
            qn = 0.0f;
            nforced = 0u;
            all_rows = false;
            eps = xmax = 0.0f;
        } else {
            qn = a.qnorm[q];
            base = precise() ? 0.0f : COS ? 1.0f : qn;
            nforced = a.stats->nforced;
            all_rows = !(qn == qn);
            xmax = __uint_as_float(a.stats->xmax_bits);
            eps = round_up_f(a.eps_rel * (double)qn + a.eps_abs);
        }
        bias = a.bias;
    }
    // row j of group f; rows left out by the scan are evaluated from their list
    __device__ __forceinline__ uint32_t row(int f, int j) const {
        const int half = f >= ntp ? 1 : 0;
        const uint32_t r = (uint32_t)(f - (half ? ntp : 0)) * kGmRows + (uint32_t)gm_group_row(half, j);
        bool on = r < nt;
        if (nforced) {
            on = on && bias[r] < __builtin_huge_valf();
        }
        return on ? r : kSentinelIdx;
    }
    // the group's first row
    __device__ __forceinline__ uint32_t first_row(int f) const {
        const int half = f >= ntp ? 1 : 0;
        return (uint32_t)(f - (half ? ntp : 0)) * kGmRows + (uint32_t)gm_group_row(half, 0);
    }
    // no row of a group with this minimum has a smaller exact value (minima near
    // f32's subnormals are not rounded down)
    __device__ __forceinline__ float least(float gm, bool ranked) const {
        return exact && !ranked && gm > 0x1p-100f ? gm : 0.0f;
    }
    // every row of the answer lies in a group whose minimum is at or below this
    __device__ __forceinline__ float bound(float t) {
        if (!(t < __builtin_huge_valf())) return __builtin_huge_valf();
        const double v = (double)t + a.eps_t * (double)t;
        if constexpr (exact) return round_up_f(v + a.eps_abs);
        const float b = precise() ? gm_bound_precise(v, qn, xmax, a.eps_rel, a.eps_abs, 2)
                                  : gm_bound(t, qn, xmax, a.eps_rel, eps);
        width = (double)b - (double)t;
        return b;
    }
    // bound of a smaller argument than before
    __device__ __forceinline__ float bound_again(float t) {
        if (exact || !(width > 0.0)) return bound(t);
        return round_up_f((double)t + width);
    }
};

// A wave's answer so far: the 64 KL smallest (value, row) pairs it has seen.
template <typename T, typename TS, int ARM, int KL>
struct GmList {
    using F = FloatTraits<T>;
    static constexpr bool COS = ARM == ARM_COS_FOLD || ARM == ARM_COS_HOST;
    static constexpr bool MINK = ARM == ARM_MINKOWSKI_INT || ARM == ARM_MINKOWSKI_POW;
    T lv[KL];
    uint32_t li[KL];      // rows of the whole index
    uint32_t row0;
    T qa = T(0);  // cosine: the query's row_sumsq (fold) or its reciprocal norm (host)
    bool qzero = false;
    MetricParams<T> mp;

    __device__ __forceinline__ GmList(const GmSelectArgs<TS>& a)
        : row0((uint32_t)a.row0), mp{(T)a.pexp, a.pint, (T)a.root_exp} {
#pragma unroll
        for (int b = 0; b < KL; ++b) {
            lv[b] = F::inf();
            li[b] = kSentinelIdx;
        }
    }
    __device__ __forceinline__ void set_query(const T* __restrict__ sq, int d) {
        if (!COS) return;
        for (int c = 0; c < d; ++c) qa = qa + sq[c] * sq[c];
        qzero = qa == T(0);
        if (ARM == ARM_COS_HOST) qa = (qa > T(0)) ? T(1) / F::sqrt_(qa) : T(0);
    }
    __device__ __forceinline__ T kth(int k) const { return list_value_at<T, KL>(lv, k - 1); }
    __device__ __forceinline__ uint32_t kth_row(int k) const {
        uint32_t r = li[0];
#pragma unroll
        for (int b = 1; b < KL; ++b)
            if (((k - 1) >> 6) == b) r = li[b];
        return bcast_u(r, (k - 1) & 63);
    }
    __device__ __forceinline__ void merge(T v, uint32_t ix, int lane) {
        if constexpr (KL == 1) wave_merge64<T>(lv[0], li[0], v, ix, lane);
        else wave_merge_blocks<T, KL>(lv, li, v, ix, lane);
    }
    // The list the parts before this one left in the outputs.
    __device__ __forceinline__ void resume(const T* __restrict__ ov, const uint32_t* __restrict__ oi, int k, int lane) {
#pragma unroll
        for (int b = 0; b < KL; ++b) {
            const int s = 64 * b + lane;
            if (s < k) {
                lv[b] = ov[s];
                li[b] = oi[s];
            }
        }
    }
    // 64 rows of the part (kSentinelIdx: none) evaluated exactly and merged in
    __device__ __forceinline__ void evaluate(uint32_t mine, const T* __restrict__ sq, const TS* __restrict__ X, int d,
                                             int k, int mode, int lane) {
        if (__builtin_amdgcn_ballot_w64(mine != kSentinelIdx) == 0ull) return;
        T ya;
        T v = gm_exact<T, TS, ARM>(sq, X + (mine != kSentinelIdx ? (int64_t)mine : 0) * d, d, ya, mp);
        if (ARM == ARM_COS_FOLD) {
            const T denom = F::sqrt_(qa * ya);
            const T sim = (denom > T(0)) ? v / denom : T(0);
            v = clamp02<T>(T(1) - sim);
        } else if (ARM == ARM_COS_HOST) {
            const T iy = (ya > T(0)) ? T(1) / F::sqrt_(ya) : T(0);
            v = clamp02<T>(T(1) - v * qa * iy);
        }
        if (mode == EMIT_ROOT_RANKED) v = MINK ? F::pow_(v, mp.root) : F::sqrt_(v);
        const bool on = mine != kSentinelIdx && v == v;  // NaN is never admitted
        v = on ? v : F::inf();
        uint32_t ix = on ? row0 + mine : kSentinelIdx;
        // a batch with nothing at or below the list's k-th value leaves it as it
        // is (the k-th value is taken with all lanes: behind `on &&` its lane
        // need not be running, and a list of two blocks is selected from first)
        const T last = kth(k);
        if (__builtin_amdgcn_ballot_w64(on && !(last < v)) == 0ull) return;
        wave_sort64<T>(v, ix, lane);
        merge(v, ix, lane);
    }
    // A minimum no row of the answer exceeds, from the k-th exact value: exact
    // <= R means a value of at most R in its units + eps.
    __device__ __forceinline__ float screen_bound(const GmQuery<T, TS, ARM>& Q) const {
        const int mode = Q.a.mode;
        if (MINK && mode == EMIT_ROOT_RANKED) return __builtin_huge_valf();
        double R = (double)kth(Q.a.k);
        if (mode == EMIT_ROOT_RANKED) R = R * R * (1.0 + 0x1p-40);
        if (!(R < (double)__builtin_huge_valf())) return __builtin_huge_valf();
        if (!COS && Q.precise())
            return gm_bound_precise(R + Q.a.eps_t * R, Q.qn, Q.xmax, Q.a.eps_rel, Q.a.eps_abs, 1);
        return round_up_f(R - (double)Q.base + (double)Q.eps + Q.a.eps_t * R);
    }
    // A query every row of which is evaluated: a zero query's values are all
    // exactly 1 (or NaN, never admitted), so the first k rows are its answer.
    __device__ __forceinline__ bool settled(int k) const {
        if (!COS) return false;
        const T last = kth(k);
        return qzero && last < F::inf();
    }
    __device__ __forceinline__ void emit(T* __restrict__ ov, uint32_t* __restrict__ oi, int k, int mode, int last,
                                         int lane) const {
#pragma unroll
        for (int b = 0; b < KL; ++b) {
            const int s = 64 * b + lane;
            if (s < k) {
                ov[s] = last && mode == EMIT_SQRT ? F::sqrt_(lv[b]) : lv[b];
                oi[s] = last && li[b] == kSentinelIdx ? 0u : li[b];
            }
        }
    }
};

typedef _Float16 gm_f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 gm_row16 __attribute__((ext_vector_type(8)));

// Sixteen columns of a pair decide most of the rows of a group that only has
// one near row: their share of the squared distance (cosine: of the unit
// vectors, 2 (1 - cos)) is a lower bound of the whole.  The columns are those
// where the query lies farthest from the centre; both sides come from the
// scan's operands, 64 bytes of a row.
template <typename TS, bool COS>
struct GmProbe {
    float* v;        // -q, in LDS (16 floats of the wave's own)
    const char* x;   // the columns of row 0
    int64_t stride;
    __device__ __forceinline__ GmProbe(const GmSelectArgs<TS>& a, int64_t q, float* lds, int lane) : v(lds) {
        const int c0 = 4 * lane;
        float e[4] = {0.f, 0.f, 0.f, 0.f}, s = 0.0f;
        if (c0 < (int)a.dp) {
            const char* o = reinterpret_cast<const char*>(a.qop + q * a.dp) + 4 * (c0 & ~15) + 2 * (c0 & 15);
            const gm_f16x4 hi = *reinterpret_cast<const gm_f16x4*>(o), lo = *reinterpret_cast<const gm_f16x4*>(o + 32);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                e[i] = (float)hi[i] + (float)lo[i];
                s = __builtin_fmaf(e[i], e[i], s);
            }
        }
        s = s + shfl_xor_f(s, 1);
        s = s + shfl_xor_f(s, 2);
        float m = s;
#pragma unroll
        for (int i = 4; i < 64; i <<= 1) m = fmaxf(m, shfl_xor_f(m, i));
        const int at = __builtin_ctzll(__builtin_amdgcn_ballot_w64(s == m)) & ~3;
        const float inv = a.qinv[q] * (COS ? 1.0f : 0.5f);
        if ((lane & ~3) == at) {
#pragma unroll
            for (int i = 0; i < 4; ++i) v[4 * (lane & 3) + i] = e[i] * inv;
        }
        wave_lds_fence();
        // a query of no extent has its largest share anywhere: within the row
        x = reinterpret_cast<const char*>(a.xcopy) + 16 * at;
        stride = 4 * a.ldx;
    }
    __device__ __forceinline__ float share(uint32_t row, float xinv) const {
        typedef const __attribute__((address_space(1))) gm_row16* vptr;
        const char* o = x + (int64_t)row * stride;
        const gm_row16 h0 = *(vptr)o, h1 = *(vptr)(o + 16), l0 = *(vptr)(o + 32), l1 = *(vptr)(o + 48);
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float f = __builtin_fmaf((float)h0[i] + (float)l0[i], xinv, v[i]);
            const float g = __builtin_fmaf((float)h1[i] + (float)l1[i], xinv, v[8 + i]);
            s = __builtin_fmaf(f, f, s);
            s = __builtin_fmaf(g, g, s);
        }
        return s;
    }
    // What no row of the answer exceeds, given that none has a minimum above
    // thr: its exact value is then at most thr + base, eps and the factor take
    // the roundings of that sum and of the exact value; the operands hold 2^-22 of
    // their elements, a distance of at most 2^-20 of (||q|| + ||x||), ||x|| <= ||q||
    // + the distance.
    static __device__ __forceinline__ float limit(float thr, float base, float qn, float eps) {
        if (!(thr < __builtin_huge_valf())) return __builtin_huge_valf();
        const float D = (COS ? 2.0f : 1.0f) * (thr + base + eps);
        const float r = __builtin_sqrtf(fmaxf(1.001f * D, 0.0f));
        const float m = r + 0x1p-18f * ((COS ? 1.0f : __builtin_sqrtf(qn)) + r);
        return m * m * (1.0f + 0x1p-15f) + 0x1p-100f;
    }
};

// Too many groups to list (ties, or distances the screen does not resolve): every
// group at or below thr, four at a time, the bound following the k-th
// exact value of the waves that share the query (shared: their bounds).  A
// group that can at best tie with the k-th value, behind its row, is passed
// over: of equal values the list has the first rows already (100,000 rows of
// three values in 30 columns, Chebyshev, 2,000 queries, f32: 5.8 -> 0.64 ms).
// Rows the probe rules out are not evaluated (200k x 5k, d = 128, k = 16, in 100
// clusters a thousandth of their spacing wide, ms, every row of a group and
// with the probe: f32 9.4 / 3.6, cosine 9.5 / 3.5, f64 18.6 / 4.3); the
// others gather in buf, 128 entries of the wave's own; cols: 16 floats of it.
// Where a precise scan may follow (a.flag), a query is left to it, and false
// returned, once it has evaluated a 32nd of the index: that is what its share
// of that scan costs (f64, 200k x 5k in clusters as above, ms: 100 of them, d =
// 128: 4.3 this way, 6.0 by the scan; 5 of them, d = 250: 79.5 and 12.0).
template <typename T, typename TS, int ARM, int KL>
__device__ __forceinline__ bool gm_pass(GmList<T, TS, ARM, KL>& L, const GmQuery<T, TS, ARM>& Q, const GmSelectArgs<TS>& a,
                                        int64_t q, const T* __restrict__ sq, float thr, int wv, int nw,
                                        volatile float* __restrict__ shared, volatile int* __restrict__ stop,
                                        float* __restrict__ cols, uint32_t* __restrict__ buf, int lane) {
    using List = GmList<T, TS, ARM, KL>;
    constexpr bool METRIC = GmQuery<T, TS, ARM>::exact;
    const int d = (int)a.d, k = a.k, mode = a.mode;
    const float inf = __builtin_huge_valf();
    const bool ranked = List::MINK && mode == EMIT_ROOT_RANKED;
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t held = 0;
    // batches of 64 rows left to this wave
    const bool bounded = GmQuery<T, TS, ARM>::twice && a.flag;
    int batches = bounded ? ((int)(Q.nt / 2048u) + 16) / nw : 0;
    auto pass = [&](auto rules_out) -> bool {
        for (int f0 = 64 * wv; f0 < Q.n; f0 += 64 * nw) {
            if (bounded && *stop) return false;
            const float gm = f0 + lane < Q.n ? Q.G[f0 + lane] : inf;
            const uint32_t row = L.row0 + Q.first_row(f0 + lane);
            const T least = (T)Q.least(gm, ranked);
            for (int w = 0; w < nw; ++w) thr = fminf(thr, shared[w]);
            auto open = [&]() -> uint64_t {
                const T last = L.kth(k);
                const uint32_t at = L.kth_row(k);
                return __builtin_amdgcn_ballot_w64(gm <= thr && gm < inf && !(least >= last && row > at));
            };
            uint64_t todo = open();
            while (todo) {
                int f = -1;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int bit = todo ? __builtin_ctzll(todo) : -1;
                    if ((lane >> 4) == i) f = bit;
                    todo &= todo - 1;  // 0 stays 0
                }
                uint32_t mine = f >= 0 ? Q.row(f0 + f, lane & 15) : kSentinelIdx;
                const bool in = mine != kSentinelIdx && !rules_out(mine);
                const uint64_t bal = __builtin_amdgcn_ballot_w64(in);
                if (in) buf[held + (uint32_t)__builtin_popcountll(bal & below)] = mine;
                held += (uint32_t)__builtin_popcountll(bal);
                wave_lds_fence();
                if (held >= 64) {
                    held -= 64;
                    mine = buf[held + lane];
                    wave_lds_fence();
                    L.evaluate(mine, sq, a.x, d, k, mode, lane);
                    thr = fminf(thr, L.screen_bound(Q));
                    todo &= open();
                    if (bounded && --batches < 0) {
                        *stop = 1;
                        return false;
                    }
                }
            }
            if (lane == 0) shared[wv] = thr;
        }
        return true;
    };
    if constexpr (METRIC) {
        pass([](uint32_t) { return false; });
    } else {
        const GmProbe<TS, List::COS> probe(a, q, cols, lane);
        if (!pass([&](uint32_t r) { return probe.share(r, a.xinv[r]) > probe.limit(thr, Q.base, Q.qn, Q.eps); }))
            return false;
    }
    if (held) L.evaluate((uint32_t)lane < held ? buf[lane] : kSentinelIdx, sq, a.x, d, k, mode, lane);
    return true;
}

// The forced rows, where there are more than are listed: a wave's share of the
// marks (256 rows from `first` on, every `stride`), the marked rows gathered
// and evaluated 64 at a time.  buf: 320 entries of the wave's own.
// (200,000 rows, 300 of them with a NaN, cosine at d = 100, 2,000 queries, f32:
// 0.69 ms; evaluating every row took 16.8.)
template <typename T, typename TS, int ARM, int KL>
__device__ __forceinline__ void gm_marked(GmList<T, TS, ARM, KL>& L, const GmSelectArgs<TS>& a, uint32_t first,
                                          uint32_t stride, const T* __restrict__ sq, uint32_t* __restrict__ buf,
                                          int lane) {
    const int d = (int)a.d, k = a.k;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint32_t n = (uint32_t)a.ntp * kGmRows;
    uint32_t held = 0;
    for (uint32_t r0 = first; r0 < n; r0 += stride) {
        const uint32_t r = r0 + 4 * lane;
        const float4 s = r < n ? gload4(a.xinv + r) : make_float4(1.f, 1.f, 1.f, 1.f);
        const float e[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const bool in = e[c] < 0.0f;
            const uint64_t bal = __builtin_amdgcn_ballot_w64(in);
            if (in) buf[held + (uint32_t)__builtin_popcountll(bal & below)] = r + c;
            held += (uint32_t)__builtin_popcountll(bal);
        }
        wave_lds_fence();
        while (held >= 64) {
            held -= 64;
            L.evaluate(buf[held + lane], sq, a.x, d, k, a.mode, lane);
        }
        wave_lds_fence();
    }
    if (held) L.evaluate((uint32_t)lane < held ? buf[lane] : kSentinelIdx, sq, a.x, d, k, a.mode, lane);
}

// A workgroup per query: few queries, long indexes.
template <typename T, typename TS, int ARM, int KL>
__global__ __launch_bounds__(256, 4) void gm_select_kernel(GmSelectArgs<TS> a) {
    __shared__ __attribute__((aligned(16))) T sq[kGmMaxD];
    __shared__ __attribute__((aligned(16))) float cm[kSelCap];
    __shared__ uint32_t cg[kSelCap + 4 * 64];
    __shared__ T mv[3 * 64 * KL];
    __shared__ uint32_t s_cnt;
    __shared__ float s_kth;
    __shared__ float s_wthr[4];
    __shared__ int s_stop;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t at_ = blockIdx.x;  // the query's place among those of the launch
    const bool listed = GmQuery<T, TS, ARM>::twice && a.list;
    if (listed && at_ >= (int64_t)a.stats->nflag) return;
    const int64_t q = listed ? (int64_t)a.list[at_] : at_;
    const int d = (int)a.d, k = a.k, mode = a.mode;
    const TS* __restrict__ X = a.x;
    const float inf = __builtin_huge_valf();
    GmQuery<T, TS, ARM> Q(a, q, at_);
    const int n = Q.n;
    GmList<T, TS, ARM, KL> L(a);
    T* const ov = static_cast<T*>(a.out_val) + q * k;
    uint32_t* const oi = a.out_idx + q * k;
    // earlier parts' list: wave 0 goes on with it, and its k-th value bounds all
    float carried = inf;
    if (!a.first) {
        L.resume(ov, oi, k, lane);
        carried = L.screen_bound(Q);
        if (wv > 0) L = GmList<T, TS, ARM, KL>(a);
    }
    if (tid < d) sq[tid] = (T)a.q[q * d + tid];
    if (tid == 0) {
        s_cnt = 0u;
        s_kth = inf;
    }

    // ---- the group minima: up to 4096 of them stay in registers ----
    const bool held = n <= 4096;
    float4 g[4];
    float m = inf;
    auto load_minima = [&](int i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int at = i + 1024 * j;
            g[j] = at < n ? gload4(Q.G + at) : make_float4(inf, inf, inf, inf);
        }
    };
    if (!Q.all_rows) {
        for (int i = 4 * tid; i < n; i += 4096) {
            load_minima(i);
#pragma unroll
            for (int j = 0; j < 4; ++j) m = fminf(m, fminf(fminf(g[j].x, g[j].y), fminf(g[j].z, g[j].w)));
        }
    }
    cm[tid] = m;
    __syncthreads();
    L.set_query(sq, d);

    if (Q.all_rows) {
        for (uint32_t r0 = 0; r0 < Q.nt; r0 += 256) {
            L.evaluate(r0 + tid < Q.nt ? r0 + tid : kSentinelIdx, sq, X, d, k, mode, lane);
            if (L.settled(k)) break;  // this wave's rows; the others' end alike
        }
    } else {
        if (Q.nforced > (uint32_t)kGmForced)
            gm_marked<T, TS, ARM, KL>(L, a, 256u * wv, 1024u, sq, cg + 320 * wv, lane);
        else if (Q.nforced)
            L.evaluate(tid < (int)Q.nforced ? a.forced[tid] : kSentinelIdx, sq, X, d, k, mode, lane);
        // ---- a first bound: the k-th smallest of the 256 threads' minima ----
        auto rank_of = [&](float v, int at, int count) -> int {
            int less = 0;
            int j = 0;
            for (; j + 4 <= count; j += 4) {
                const float4 o = *reinterpret_cast<const float4*>(cm + j);
                less += (o.x < v || (o.x == v && j < at)) ? 1 : 0;
                less += (o.y < v || (o.y == v && j + 1 < at)) ? 1 : 0;
                less += (o.z < v || (o.z == v && j + 2 < at)) ? 1 : 0;
                less += (o.w < v || (o.w == v && j + 3 < at)) ? 1 : 0;
            }
            for (; j < count; ++j) {
                const float o = cm[j];
                less += (o < v || (o == v && j < at)) ? 1 : 0;
            }
            return less;
        };
        if (rank_of(m, tid, 256) == k - 1) s_kth = m;
        __syncthreads();
        float thr = fminf(Q.bound(s_kth), carried);
        // ---- the groups at or below it ----
        for (int i = 4 * tid; i < n; i += 4096) {
            if (!held) load_minima(i);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float e[4] = {g[j].x, g[j].y, g[j].z, g[j].w};
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (e[c] <= thr && e[c] < inf) {
                        const uint32_t at = atomicAdd(&s_cnt, 1u);
                        if (at < (uint32_t)kSelCap) {
                            cm[at] = e[c];
                            cg[at] = (uint32_t)(i + 1024 * j + c);
                        }
                    }
            }
        }
        __syncthreads();
        int count = (int)s_cnt;
        if (count <= kSelCap) {
            // ---- the exact k-th smallest minimum, and the list cut to it.
            //      (All groups at or below the first bound are listed, the k
            //      smallest among them.) ----
            if (count > k && count <= kSelRefine) {
                float v[2];
                uint32_t gi[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int at = tid + 256 * j;
                    v[j] = at < count ? cm[at] : inf;
                    gi[j] = at < count ? cg[at] : 0u;
                    if (at < count && rank_of(v[j], at, count) == k - 1) s_kth = v[j];
                }
                __syncthreads();
                thr = fminf(Q.bound_again(s_kth), carried);
                if (tid == 0) s_cnt = 0u;
                __syncthreads();
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    if (tid + 256 * j < count && v[j] <= thr) cg[atomicAdd(&s_cnt, 1u)] = gi[j];
                __syncthreads();
                count = (int)s_cnt;
            }
            for (int g0 = 4 * wv; g0 < count; g0 += 16) {
                const int at = g0 + (lane >> 4);
                L.evaluate(at < count ? Q.row((int)cg[at], lane & 15) : kSentinelIdx, sq, X, d, k, mode, lane);
            }
        } else {
            if (GmQuery<T, TS, ARM>::twice && a.flag && (uint32_t)count > a.flag_above) {
                if (tid == 0) a.flag[atomicAdd(&a.stats->nflag, 1u)] = (uint32_t)q;
                return;
            }
            if (tid < 4) s_wthr[tid] = thr;
            if (tid == 0) s_stop = 0;
            __syncthreads();
            gm_pass<T, TS, ARM, KL>(L, Q, a, q, sq, thr, wv, 4, s_wthr, &s_stop, cm + 16 * wv, cg + 320 * wv, lane);
            if (GmQuery<T, TS, ARM>::twice && a.flag) {
                __syncthreads();
                if (s_stop) {
                    if (tid == 0) a.flag[atomicAdd(&a.stats->nflag, 1u)] = (uint32_t)q;
                    return;
                }
            }
        }
    }

    // ---- the four waves' lists into wave 0's, and out ----
    uint32_t* mi = cg;
    __syncthreads();
    if (wv > 0) {
#pragma unroll
        for (int b = 0; b < KL; ++b) {
            mv[(wv - 1) * 64 * KL + 64 * b + lane] = L.lv[b];
            mi[(wv - 1) * 64 * KL + 64 * b + lane] = L.li[b];
        }
    }
    __syncthreads();
    if (wv > 0) return;
#pragma unroll
    for (int b = 0; b < 3 * KL; ++b) L.merge(mv[64 * b + lane], mi[64 * b + lane], lane);
    L.emit(ov, oi, k, mode, a.last, lane);
}

// A wave per query: many queries.  No barrier, no atomic: the bound is the
// k-th smallest of the lanes' two smallest minima, the groups below it are
// compacted with ballots, and the wave's own list is the answer.
constexpr int kSelWaveCap = 256;
// Five waves per SIMD where the arm's state fits 96 registers (200k x 5k, d = 256,
// k = 16, f64 cosine: 1.90 ms with 102 registers, 1.84 with 96).
constexpr int gm_select_waves(int arm, int kl) {
    return kl == 1 && arm != ARM_COS_FOLD && arm != ARM_MINKOWSKI_INT && arm != ARM_MINKOWSKI_POW ? 5 : 4;
}
template <typename T, typename TS, int ARM, int KL>
__global__ __launch_bounds__(256, gm_select_waves(ARM, KL)) void gm_select_wave_kernel(GmSelectArgs<TS> a) {
    __shared__ __attribute__((aligned(16))) T sq_[4][kGmMaxD];
    __shared__ float cm_[4][kSelWaveCap];
    __shared__ uint32_t cg_[4][kSelWaveCap + 64];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t at_ = (int64_t)blockIdx.x * 4 + wv;  // the query's place among those of the launch
    const bool listed = GmQuery<T, TS, ARM>::twice && a.list;
    if (at_ >= (listed ? (int64_t)a.stats->nflag : a.nq)) return;
    const int64_t q = listed ? (int64_t)a.list[at_] : at_;
    T* __restrict__ sq = sq_[wv];
    float* __restrict__ cm = cm_[wv];
    uint32_t* __restrict__ cg = cg_[wv];
    const int d = (int)a.d, k = a.k, mode = a.mode;
    const TS* __restrict__ X = a.x;
    const float inf = __builtin_huge_valf();
    const uint64_t below = (1ull << lane) - 1ull;
    GmQuery<T, TS, ARM> Q(a, q, at_);
    const int n = Q.n;
    GmList<T, TS, ARM, KL> L(a);
    T* const ov = static_cast<T*>(a.out_val) + q * k;
    uint32_t* const oi = a.out_idx + q * k;
    float carried = inf;  // what the earlier parts' list bounds
    if (!a.first) {
        L.resume(ov, oi, k, lane);
        carried = L.screen_bound(Q);
    }
    for (int c = lane; c < d; c += 64) sq[c] = (T)a.q[q * d + c];
    wave_lds_fence();
    L.set_query(sq, d);

    if (Q.all_rows) {
        for (uint32_t r0 = 0; r0 < Q.nt; r0 += 64) {
            L.evaluate(r0 + lane < Q.nt ? r0 + lane : kSentinelIdx, sq, X, d, k, mode, lane);
            if (L.settled(k)) break;
        }
        L.emit(ov, oi, k, mode, a.last, lane);
        return;
    }
    if (Q.nforced > (uint32_t)kGmForced)
        gm_marked<T, TS, ARM, KL>(L, a, 0u, 256u, sq, cg, lane);
    else
        for (uint32_t f0 = 0; f0 < Q.nforced; f0 += 64)
            L.evaluate(f0 + lane < Q.nforced ? a.forced[f0 + lane] : kSentinelIdx, sq, X, d, k, mode, lane);

    // ---- the minima (up to 1024 stay in registers) and the first bound ----
    const bool held = n <= 1024;
    float4 g[4];
    auto load_minima = [&](int i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int at = i + 256 * j;
            g[j] = at < n ? gload4(Q.G + at) : make_float4(inf, inf, inf, inf);
        }
    };
    float m1 = inf, m2 = inf;
    for (int i0 = 0; i0 < n; i0 += 1024) {
        load_minima(i0 + 4 * lane);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float e[4] = {g[j].x, g[j].y, g[j].z, g[j].w};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                m2 = fminf(m2, fmaxf(m1, e[c]));
                m1 = fminf(m1, e[c]);
            }
        }
    }
    float bv[KL];
    uint32_t bi[KL];
#pragma unroll
    for (int b = 0; b < KL; ++b) {
        bv[b] = inf;
        bi[b] = kSentinelIdx;
    }
    {
        uint32_t i1 = (uint32_t)lane, i2 = 64u + (uint32_t)lane;
        wave_sort64<float>(m1, i1, lane);
        bv[0] = m1;
        bi[0] = i1;
        if (KL > 1 || k > 16) {
            wave_sort64<float>(m2, i2, lane);
            if constexpr (KL == 1) wave_merge64<float>(bv[0], bi[0], m2, i2, lane);
            else wave_merge_blocks<float, KL>(bv, bi, m2, i2, lane);
        }
    }
    float thr = fminf(Q.bound(list_value_at<float, KL>(bv, k - 1)), carried);

    // ---- the groups at or below it ----
    uint32_t cnt = 0;
    for (int i0 = 0; i0 < n; i0 += 1024) {
        if (!held) load_minima(i0 + 4 * lane);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float e[4] = {g[j].x, g[j].y, g[j].z, g[j].w};
            const float lo = fminf(fminf(e[0], e[1]), fminf(e[2], e[3]));
            if (__builtin_amdgcn_ballot_w64(lo <= thr && lo < inf) == 0ull) continue;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const bool in = e[c] <= thr && e[c] < inf;
                const uint64_t bal = __builtin_amdgcn_ballot_w64(in);
                const uint32_t at = cnt + (uint32_t)__builtin_popcountll(bal & below);
                if (in && at < (uint32_t)kSelWaveCap) {
                    cm[at] = e[c];
                    cg[at] = (uint32_t)(i0 + 256 * j + 4 * lane + c);
                }
                cnt += (uint32_t)__builtin_popcountll(bal);
            }
        }
    }
    wave_lds_fence();
    if (cnt <= (uint32_t)kSelWaveCap) {
        // ---- the exact k-th smallest minimum, and the list cut to it ----
        if (cnt > (uint32_t)k) {
#pragma unroll
            for (int b = 0; b < KL; ++b) {
                bv[b] = inf;
                bi[b] = kSentinelIdx;
            }
            for (uint32_t b0 = 0; b0 < cnt; b0 += 64) {
                float v = b0 + lane < cnt ? cm[b0 + lane] : inf;
                uint32_t ix = b0 + lane;
                wave_sort64<float>(v, ix, lane);
                if constexpr (KL == 1) wave_merge64<float>(bv[0], bi[0], v, ix, lane);
                else wave_merge_blocks<float, KL>(bv, bi, v, ix, lane);
            }
            thr = fminf(Q.bound_again(list_value_at<float, KL>(bv, k - 1)), carried);
            uint32_t kept = 0;
            for (uint32_t b0 = 0; b0 < cnt; b0 += 64) {
                const bool in = b0 + lane < cnt && cm[b0 + lane] <= thr;
                const uint32_t gi = b0 + lane < cnt ? cg[b0 + lane] : 0u;
                const uint64_t bal = __builtin_amdgcn_ballot_w64(in);
                wave_lds_fence();
                if (in) cg[kept + (uint32_t)__builtin_popcountll(bal & below)] = gi;
                wave_lds_fence();
                kept += (uint32_t)__builtin_popcountll(bal);
            }
            cnt = kept;
        }
        for (uint32_t g0 = 0; g0 < cnt; g0 += 4) {
            const uint32_t at = g0 + (lane >> 4);
            L.evaluate(at < cnt ? Q.row((int)cg[at], lane & 15) : kSentinelIdx, sq, X, d, k, mode, lane);
        }
    } else {
        if (GmQuery<T, TS, ARM>::twice && a.flag && cnt > a.flag_above) {
            if (lane == 0) a.flag[atomicAdd(&a.stats->nflag, 1u)] = (uint32_t)q;
            return;
        }
        // the list of one wave bounds itself
        if (lane == 0) {
            cm[16] = thr;
            cm[17] = 0.0f;
        }
        wave_lds_fence();
        if (!gm_pass<T, TS, ARM, KL>(L, Q, a, q, sq, thr, 0, 1, cm + 16, reinterpret_cast<volatile int*>(cm + 17), cm, cg,
                                     lane)) {
            if (lane == 0) a.flag[atomicAdd(&a.stats->nflag, 1u)] = (uint32_t)q;
            return;
        }
    }
    L.emit(ov, oi, k, mode, a.last, lane);
}

// A wave per query where there are queries enough to fill the chip with four
// times fewer workgroups, and few groups to read; longer lists take more of the
// wave's serial work.  A search, us, wave / workgroup per query, f32, d = 64:
//   k = 10: 10k x 500: 49.2 / 48.7, 10k x 1k: 51.2 / 53.7, 10k x 2k: 60.5 / 77.3,
//   100k x 500: 100.9 / 96.5, 100k x 1k: 121 / 120, 100k x 4k: 241 / 271,
//   260k x 2k (16,250 groups): 293 / 298, 520k x 2k: 556 / 563, 1M x 2k: 1084 / 1044;
//   k = 50: 10k x 1k: 86 / 75, 10k x 2k: 97 / 112, 100k x 1k: 160 / 140,
//   100k x 2k: 200 / 207, 260k x 2k: 346 / 362, 1M x 2k: 1132 / 1094
//   (f64: 10k x 1k: 113 / 97, 10k x 2k: 141 / 154).
template <typename T, typename TS, int ARM, int KL>
void gm_select_launch(const GmSelectArgs<TS>& a, hipStream_t s) {
    if (KL == 1 && a.nq >= (a.k <= 16 ? 1000 : 2000) && 2 * a.ntp <= 16384)
        hipLaunchKernelGGL((gm_select_wave_kernel<T, TS, ARM, KL>), dim3((unsigned)((a.nq + 3) / 4)), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((gm_select_kernel<T, TS, ARM, KL>), dim3((unsigned)a.nq), dim3(256), 0, s, a);
}

template <typename T, typename TS, int ARM>
void gm_select_k(const GmSelectArgs<TS>& a, hipStream_t s) {
    if (a.k <= 64) gm_select_launch<T, TS, ARM, 1>(a, s);
    else gm_select_launch<T, TS, ARM, 2>(a, s);
}

}  // namespace

}  // namespace mlrs
