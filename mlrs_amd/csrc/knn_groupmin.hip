// Group-minimum search: operand preparation and the selection pass
// (knn_groupmin.hpp says how the search works).
#include "knn_groupmin_select.hpp"

namespace mlrs {

namespace {

// ---------------------------------------------------------------------------
// Preparation: norms, the rows the screen cannot be trusted with, and the
// scaled copy of two halves per element.  LPR lanes share a row, four consecutive columns each.
// Bound by the read of the rows.
// ---------------------------------------------------------------------------
template <typename T> struct GmRange;
// Squared norms the screen's error bound holds for: no sum of products
// overflows f32 and none of the arms' own norm products leaves the range.
template <> struct GmRange<float> {
    static __device__ __forceinline__ bool euclid(float s) { return s <= 0x1p120f; }
    static __device__ __forceinline__ bool cosine(float s) { return s >= 0x1p-60f && s <= 0x1p60f; }
};
template <> struct GmRange<double> {
    static __device__ __forceinline__ bool euclid(double s) { return s <= 0x1p120; }
    static __device__ __forceinline__ bool cosine(double s) { return s >= 0x1p-500 && s <= 0x1p500; }
};

template <typename T, int LPR>
__global__ __launch_bounds__(256) void gm_prep_kernel(GmPrepArgs a) {
    constexpr int RPW = 64 / LPR;      // rows a wave takes at once
    constexpr int U = 4;               // row groups in flight
    const int lane = threadIdx.x & 63;
    const int sub = lane % LPR, rsub = lane / LPR;
    const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const T* __restrict__ X = static_cast<const T*>(a.rows);
    const int d = (int)a.d;
    const int c0 = 4 * sub;
    if (a.queries && blockIdx.x == 0 && threadIdx.x == 0) {
        a.stats->nflag = 0u;
        if (a.reset) {
            // the index launch behind this one fills them
            a.stats->xmax_bits = 0u;
            a.stats->nforced = 0u;
        }
    }
    T ctr[4] = {T(0), T(0), T(0), T(0)};
    if (a.centre) {
        const T* C = static_cast<const T*>(a.centre);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (c0 + e < d) ctr[e] = gm_centre(C, a.centre_n, d, c0 + e);
    }
    const int64_t n = a.n, n_out = a.n_out;
    const int64_t n_all = n_out > a.n_norm ? n_out : a.n_norm;
    const bool vec = (d % 4 == 0) && ((reinterpret_cast<uintptr_t>(X) & 15) == 0);
    float xmax = 0.0f;
    for (int64_t r0 = wave * (RPW * U); r0 < n_all; r0 += (int64_t)gridDim.x * 4 * (RPW * U)) {
        T v[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t r = r0 + u * RPW + rsub;
            const T* p = X + (r < n ? r : 0) * d + c0;
            if (vec) {
                if (c0 < d) {
                    if (sizeof(T) == 4) {
                        const float4 f = *reinterpret_cast<const float4*>(p);
                        v[u][0] = (T)f.x;
                        v[u][1] = (T)f.y;
                        v[u][2] = (T)f.z;
                        v[u][3] = (T)f.w;
                    } else {
                        const double2 f = reinterpret_cast<const double2*>(p)[0], g = reinterpret_cast<const double2*>(p)[1];
                        v[u][0] = (T)f.x;
                        v[u][1] = (T)f.y;
                        v[u][2] = (T)g.x;
                        v[u][3] = (T)g.y;
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[u][e] = T(0);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[u][e] = (c0 + e < d) ? p[e] : T(0);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t r = r0 + u * RPW + rsub;
            const bool on = r < n;
            // Euclidean: the f32 values the scan works on, and their norm;
            // cosine: the row's own norm, in T
            float f[4];
            T s = T(0);
            if (!a.cosine) {
                float sf = 0.0f;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    f[e] = (c0 + e < d) ? (float)(v[u][e] - ctr[e]) : 0.0f;
                    sf = __builtin_fmaf(f[e], f[e], sf);
                }
                s = (T)sf;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) s = s + v[u][e] * v[u][e];
            }
#pragma unroll
            for (int m = 1; m < LPR; m <<= 1) s = s + shfl_xor_f(s, m);
            bool trusted, zero = false;
            T inv = T(0);
            if (!a.cosine) {
                trusted = GmRange<T>::euclid(s);
            } else {
                zero = s == T(0);
                trusted = GmRange<T>::cosine(s);
                if (trusted) inv = T(1) / FloatTraits<T>::sqrt_(s);
                if (!a.queries) trusted = trusted || zero;  // a zero row scores exactly 1, as its screen value does
#pragma unroll
                for (int e = 0; e < 4; ++e) f[e] = (float)(v[u][e] * inv);
            }
            // The row's scale: the power of two that takes its norm to at most
            // 2^15, so that no element leaves f16's range and what f16 cannot
            // resolve (2^-14 and less) is below 2^-27 of the norm.  Norms below
            // 2^-50 share one scale; what they lose is in eps_abs.
            int ex = 14;
            if (!a.cosine) ex = 15 - ((__builtin_amdgcn_frexp_expf(fmaxf((float)s, 0x1p-100f)) + 1) >> 1);
            if (!on || !trusted) ex = 0;
            if (r < n_out && c0 < a.ldo) {
                gm_f16x4 hi, lo;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float v_ = __builtin_ldexpf((on && trusted) ? (a.queries ? -f[e] : f[e]) : 0.0f, ex);
                    hi[e] = (_Float16)v_;
                    lo[e] = (_Float16)(v_ - (float)hi[e]);
                }
                // 16 columns are four 16-byte chunks: high halves of the first
                // and the last eight, then the low halves
                char* o = reinterpret_cast<char*>(a.out + r * a.ldo) + 4 * (c0 & ~15) + 2 * (c0 & 15);
                *reinterpret_cast<gm_f16x4*>(o) = hi;
                *reinterpret_cast<gm_f16x4*>(o + 32) = lo;
            }
            if (sub != 0 || r >= a.n_norm) continue;
            const float nan = __builtin_nanf(""), inf = __builtin_huge_valf();
            // Euclidean: a row with a NaN scores NaN against every query and
            // is never admitted; cosine's fold arm scores it 1
            const bool force = on && !trusted && !a.queries && (a.cosine || s == s);
            a.inv[r] = force ? -1.0f : __builtin_ldexpf(1.0f, (a.queries && !a.cosine ? 1 : 0) - ex);
            if (a.queries) {
                a.norm[r] = trusted ? (a.cosine ? 0.0f : (float)s) : nan;
                continue;
            }
            const bool keep = on && trusted;
            a.norm[r] = keep ? (a.cosine ? 0.0f : (float)s - a.eps_rel * (float)s) : inf;
            if (keep && !a.cosine) xmax = fmaxf(xmax, (float)s);
            if (force) {
                const unsigned int at = atomicAdd(&a.stats->nforced, 1u);
                if (at < (unsigned int)kGmForced) a.forced[at] = (uint32_t)r;
            }
        }
    }
    if (!a.queries && !a.cosine) {
        for (int m = 32; m > 0; m >>= 1) xmax = fmaxf(xmax, shfl_xor_f(xmax, m));
        __shared__ float wmax[4];
        if (lane == 0) wmax[threadIdx.x >> 6] = xmax;
        __syncthreads();
        if (threadIdx.x == 0) {
            const unsigned int b =
                __float_as_uint(fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3])));
            if (b > __hip_atomic_load(&a.stats->xmax_bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                atomicMax(&a.stats->xmax_bits, b);
        }
    }
}

template <typename T, int LPR>
void gm_prep_lpr(const GmPrepArgs& a, int64_t n_all, hipStream_t s) {
    const int64_t per = (64 / LPR) * 4 * 4;  // rows a workgroup takes at once
    const int64_t blocks = (n_all + per - 1) / per;
    hipLaunchKernelGGL((gm_prep_kernel<T, LPR>), dim3((unsigned)(blocks < 2048 ? blocks : 2048)), dim3(256), 0, s, a);
}

}  // namespace

template <typename T>
hipError_t launch_gm_prep(const GmPrepArgs& a, hipStream_t s) {
    const int64_t n_all = a.n_out > a.n_norm ? a.n_out : a.n_norm;
    const int64_t cols = a.ldo > a.d ? a.ldo : a.d;
    if (cols <= 16) gm_prep_lpr<T, 4>(a, n_all, s);
    else if (cols <= 32) gm_prep_lpr<T, 8>(a, n_all, s);
    else if (cols <= 64) gm_prep_lpr<T, 16>(a, n_all, s);
    else if (cols <= 128) gm_prep_lpr<T, 32>(a, n_all, s);
    else if (cols <= 256) gm_prep_lpr<T, 64>(a, n_all, s);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}
template hipError_t launch_gm_prep<float>(const GmPrepArgs&, hipStream_t);
template hipError_t launch_gm_prep<double>(const GmPrepArgs&, hipStream_t);

template <typename T, typename TS>
hipError_t launch_gm_select(const GmSelectArgs<TS>& a, int arm, hipStream_t s) {
    if (a.nq == 0) return hipSuccess;
    if constexpr (sizeof(T) == sizeof(TS)) {
        switch (arm) {
        case ARM_EUCLID_FMA: gm_select_k<T, TS, ARM_EUCLID_FMA>(a, s); break;
        case ARM_EUCLID_MULADD: gm_select_k<T, TS, ARM_EUCLID_MULADD>(a, s); break;
        case ARM_COS_FOLD: gm_select_k<T, TS, ARM_COS_FOLD>(a, s); break;
        case ARM_COS_HOST: gm_select_k<T, TS, ARM_COS_HOST>(a, s); break;
        default: return hipErrorInvalidValue;
        }
    } else {
        if (arm != ARM_EUCLID_MULADD) return hipErrorInvalidValue;
        gm_select_k<T, TS, ARM_EUCLID_MULADD>(a, s);
    }
    return hipGetLastError();
}
template hipError_t launch_gm_select<float, float>(const GmSelectArgs<float>&, int, hipStream_t);
template hipError_t launch_gm_select<double, double>(const GmSelectArgs<double>&, int, hipStream_t);
template hipError_t launch_gm_select<double, float>(const GmSelectArgs<float>&, int, hipStream_t);

}  // namespace mlrs
