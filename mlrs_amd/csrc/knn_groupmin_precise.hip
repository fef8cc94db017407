// The precise scan of the group-minimum search (knn_groupmin.hpp): for queries
// whose neighbours the f16 screen cannot tell apart, the minima over 16 index
// rows on the f64 matrix cores, from the rows as given (float rows are
// widened), around the copies' centre.
//
// A workgroup is 4 waves of 16 queries; a wave holds its queries as the B
// operand of v_mfma_f64_16x16x4f64 (lane l: query l % 16, quarter l / 16 of the
// columns), and the index is walked a group of 16 rows at a time through two
// LDS buffers, the next group staged in registers meanwhile: 16 threads a row,
// centred and its norm summed on the way.  The result's lane l holds rows l / 16
// + 4 r of its query.  Bound by the f64 matrix rate (200k x 5k, d = 128, all queries
// left to it: about 5 ms, 51 TFLOP/s, 65% of that peak).  How many queries there are
// is read on the device: with none a workgroup ends at once (5 us).
#include "knn_common.hpp"
#include "knn_groupmin.hpp"

namespace mlrs {

namespace {

constexpr int kPrQpb = 64;  // queries per workgroup
typedef double pr_f64x4 __attribute__((ext_vector_type(4)));

// Workgroups per CU: what the query operand's 2 NS registers leave.
constexpr int pr_waves(int ns) { return ns <= 16 ? 4 : ns <= 32 ? 3 : 2; }

template <typename TS, int NS, bool COS>
__global__ __launch_bounds__(256, pr_waves(NS)) void gm_precise_kernel(GmPreciseArgs<TS> a) {
    constexpr int DP = 4 * NS;
    constexpr int STRIDE = DP + 2;  // rows 16 bytes apart in the banks
    constexpr int PR = DP / 16;     // columns a thread stages: c0 + 16 p
    __shared__ __attribute__((aligned(16))) double tile[2][16][STRIDE];
    __shared__ double tn[2][16];    // ||x||^2 (cosine: -1 / ||x||), +inf for rows left out
    __shared__ double ctr[DP];
    const int64_t count = a.stats->nflag;
    if (count == 0) return;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, jl = lane & 15;
    const int srow = tid >> 4, c0 = tid & 15;
    const int d = (int)a.d;
    const double inf = __builtin_huge_val();
    for (int c = tid; c < DP; c += 256) ctr[c] = (!COS && c < d) ? (double)gm_centre(a.centre, a.centre_n, d, c) : 0.0;
    __syncthreads();

    TS v[PR];
    bool kept = false;
    auto fetch = [&](int64_t group) {
        const int64_t r = (group >> 1) * kGmRows + gm_group_row((int)(group & 1), srow);
        kept = r < a.nt && a.bias[r < a.nt ? r : 0] < __builtin_huge_valf();
        const TS* __restrict__ p = a.x + (r < a.nt ? r : 0) * d;
#pragma unroll
        for (int i = 0; i < PR; ++i) v[i] = c0 + 16 * i < d ? p[c0 + 16 * i] : TS(0);
    };
    auto put = [&](int b) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < PR; ++i) {
            const double x = (double)v[i] - ctr[c0 + 16 * i];
            tile[b][srow][c0 + 16 * i] = x;
            s = __builtin_fma(x, x, s);
        }
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) s = s + shfl_xor_f(s, m);
        if (c0 == 0) tn[b][srow] = !kept ? inf : COS ? (s > 0.0 ? -1.0 / __builtin_sqrt(s) : 0.0) : s;
    };

    const StreamSplit sp(count, a.tiles * kGmRows, kPrQpb, kGmRows * kGmQuad, gridDim.x);
    const int64_t wg = xcd_grouped_wg(blockIdx.x, gridDim.x);
    const int64_t u_hi = ((wg + 1) * sp.P < sp.T) ? (wg + 1) * sp.P : sp.T;
    for (int64_t u = wg * sp.P; u < u_hi;) {
        int64_t panel, qblock, quad0, left;
        sp.decode(u, panel, qblock, quad0, left);
        const int64_t quads = left < u_hi - u ? left : u_hi - u;
        u += quads;
        const int64_t qi = qblock * kPrQpb + w * 16 + jl;
        const bool on = qi < count;
        const TS* __restrict__ qp = a.q + (int64_t)a.list[on ? qi : 0] * d;
        double qreg[NS], qn = 0.0;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int c = g * NS + s;
            qreg[s] = c < d ? (double)qp[c] - ctr[c] : 0.0;
            qn = __builtin_fma(qreg[s], qreg[s], qn);
        }
        qn = qn + shfl_xor_f(qn, 16);
        qn = qn + shfl_xor_f(qn, 32);
        const double scale = COS ? 1.0 / __builtin_sqrt(qn) : -2.0;  // (a zero query evaluates every row: never listed)
#pragma unroll
        for (int s = 0; s < NS; ++s) qreg[s] *= scale;
        const int64_t g_lo = 8 * quad0, g_hi = 8 * (quad0 + quads);  // groups of 16 rows
        __syncthreads();  // the buffers of the range before are no longer read
        fetch(g_lo);
        put(0);
        __syncthreads();
        float keep[2] = {0.f, 0.f};
        for (int64_t gi = g_lo; gi < g_hi; ++gi) {
            const int b = (int)(gi & 1);
            if (gi + 1 < g_hi) fetch(gi + 1);
            // two chains: one dependent chain leaves the matrix unit idle
            // between its instructions
            pr_f64x4 acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = acc0;
            const double* arow = &tile[b][jl][g * NS];
            double2 av = *reinterpret_cast<const double2*>(arow);
#pragma unroll
            for (int p = 0; p < NS / 2; ++p) {
                double2 an = av;
                if (p + 1 < NS / 2) an = *reinterpret_cast<const double2*>(arow + 2 * (p + 1));
                __builtin_amdgcn_sched_barrier(0);
                acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(av.x, qreg[2 * p], acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(av.y, qreg[2 * p + 1], acc1, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                av = an;
            }
            double m = inf;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double n = tn[b][g + 4 * r], s = acc0[r] + acc1[r];
                // a row left out may hold anything: NaN is ignored
                m = fmin(m, COS ? (n < inf ? 1.0 + s * n : inf) : n + qn + s);
            }
            float f = round_down_f(fmax(m, 0.0));
            f = fminf(f, shfl_xor_f(f, 16));
            f = fminf(f, shfl_xor_f(f, 32));
            // lane group t keeps the t-th tile's two minima, four tiles' go out together
            const int t = (int)(gi >> 1) & 3;
            if (g == t) keep[gi & 1] = f;
            if ((gi & 7) == 7 && on) {
                float* o = a.gmin + qi * 2 * a.ntp + (gi >> 1) - 3 + g;
                o[0] = keep[0];
                o[a.ntp] = keep[1];
            }
            if (gi + 1 < g_hi) put(b ^ 1);
            __syncthreads();
        }
    }
}

template <typename TS, int NS, bool COS>
void precise_ns(const GmPreciseArgs<TS>& a, hipStream_t s) {
    const dim3 grid((unsigned)(pr_waves(NS) * (a.grid_wgs > 0 ? a.grid_wgs : 1)));
    hipLaunchKernelGGL((gm_precise_kernel<TS, NS, COS>), grid, dim3(256), 0, s, a);
}

template <typename TS, bool COS>
hipError_t precise_launch(const GmPreciseArgs<TS>& a, hipStream_t s) {
    const int64_t ns = (a.d + 3) / 4;
    if (ns <= 8) precise_ns<TS, 8, COS>(a, s);
    else if (ns <= 16) precise_ns<TS, 16, COS>(a, s);
    else if (ns <= 32) precise_ns<TS, 32, COS>(a, s);
    else if (ns <= 48) precise_ns<TS, 48, COS>(a, s);
    else if (ns <= 64) precise_ns<TS, 64, COS>(a, s);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace

template <typename TS>
hipError_t launch_gm_precise(const GmPreciseArgs<TS>& a, bool cosine, hipStream_t s) {
    if constexpr (sizeof(TS) == 8) {
        if (cosine) return precise_launch<TS, true>(a, s);
    } else if (cosine) {
        return hipErrorInvalidValue;  // the graph's cosine works on normalised f64 rows
    }
    return precise_launch<TS, false>(a, s);
}
template hipError_t launch_gm_precise<float>(const GmPreciseArgs<float>&, bool, hipStream_t);
template hipError_t launch_gm_precise<double>(const GmPreciseArgs<double>&, bool, hipStream_t);

}  // namespace mlrs
