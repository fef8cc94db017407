// Fused f32 Gram-MFMA nearest row with exact rescoring (gfx950): the k-means
// assignment (argmin_dist_rows, crates/mlrs-kernels/src/kmeans.rs:284-310)
// where the centres do not fit knn_k1_resident.hip, and k = 1 Euclidean
// searches of short indexes.  d <= 256.
//
// Two register shapes (GramShape below): d <= 128, 4 waves x 32 queries =
// 128 queries per workgroup on v_mfma_f32_32x32x2f32; 128 < d <= 256, 4 waves
// x 16 queries = 64 per workgroup on v_mfma_f32_16x16x4f32.  Either walks one
// strip of index rows 32 at a time.
//  * Each wave keeps its query rows in VGPRs as the B operand (pre-scaled by
//    -2), loaded once per segment.
//  * The 32-row index tile is staged in LDS (row stride d_pad + 4 floats, so
//    16 consecutive rows fall on distinct bank groups; rows of 128 floats in
//    pairs that share one 1 KB slot), double-buffered in two distinct LDS
//    objects, the next tile prefetched into registers.
//  * The accumulator starts at ||x_t||^2, so after the contraction acc =
//    ||x_t||^2 - 2 x_t.q_j, the expansion minus the per-query constant.
//  * Screen: acc is compared against a per-query threshold derived from the
//    best value known for the query (its own, any segment's through a
//    per-query word in global memory) plus a rigorous bound eps on the
//    expansion's rounding error and the reference's own, tightened every tile
//    with the tile's smallest expansion value.  A pair that can still win
//    always passes; the comparison is !(acc > thr), so NaN passes too.
//  * Passing rows are queued per query in LDS (queue lengths live in
//    registers; the lanes screening a query append with a popcount prefix, no
//    atomics) and evaluated EXACTLY in lane-parallel batches, in the arm's
//    operation order; one (value, index) pair per query and segment is kept.
//  * The merge kernel takes the best pair of a query's segments.
//  * Work split: StreamSplit (knn_kernels.hpp), panel-major, with XCD-grouped
//    workgroup numbering, so the workgroups on one XCD stream the same index
//    panel in lockstep.
// The kept pair is therefore the reference's own: the full distance matrix
// never reaches HBM and no tolerance is involved.
#include "knn_common.hpp"
#include "knn_kernels.hpp"

namespace mlrs {

namespace {

constexpr int kWaves = 4;                // waves per workgroup, narrow shape (the wide shape: 6)
constexpr int kBn = 32;                  // index rows per tile
constexpr int kQcap = 48;                // queued rows per query: the screen tightens every tile, queues stay short
constexpr int kFlushAt = kQcap - kBn;    // flush when a queue may overflow on the next tile
constexpr int kShareEvery = 64;          // tiles between reads of the shared thresholds
// The two register shapes of a wave's block of (row, query) values.
//  d <= 128 (W16 = false): 32 queries per wave, v_mfma_f32_32x32x2f32 over
//    the 32-row tile; lane (h = lane / 32, jl = lane % 32) holds 16 of query
//    jl's rows, and the query operand is d/2 VGPRs.
//  128 < d <= 256 (W16 = true): 16 queries per wave, v_mfma_f32_16x16x4f32
//    on the tile's two 16-row halves; lane (g = lane / 16, jl = lane % 16)
//    holds 8 of query jl's rows, and lane group g contracts the g-th quarter
//    of the feature axis, so the query operand is d/4 VGPRs (64 at d = 256).
//  Both shapes run 4 waves per workgroup.  (For the wide shape, whose two
//  33 KB tiles leave room for only two workgroups per CU, a third wave per
//  SIMD from larger workgroups did not pay: two 6-wave workgroups are seldom
//  placed so that both fit a CU (d256 7.0 ms), and one 12-wave workgroup runs
//  its waves in lockstep behind one barrier (5.6 ms against 5.3-5.4).)
template <bool W16>
struct GramShape {
    static constexpr int qpw = W16 ? 16 : 32;      // queries per wave
    static constexpr int waves = kWaves;           // waves per workgroup
    static constexpr int threads = 64 * waves;
    static constexpr int qpb = waves * qpw;        // queries per workgroup
    static constexpr int vals = W16 ? 8 : 16;      // tile values per lane
};
constexpr int kQpbNarrow = GramShape<false>::qpb;
constexpr int kQpbWide = GramShape<true>::qpb;
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Per-wave LDS state.
template <int QPW>
struct WaveLds {
    uint32_t qidx[QPW][kQcap];
    float thr[QPW];
    float qs[QPW];   // ||q||^2
    float eps[QPW];  // screen error bound
    uint32_t off[QPW];                 // queue offsets of the batched flush
    uint32_t mode[QPW];                // 0: screen values lie within eps of exact values; 1: a sum may overflow
    unsigned long long best[QPW];      // (value bits << 32 | index) of the kept pair
};

// (value, index) packed so that unsigned order is the (value, index) order
// for the non-negative values every served arm produces.
constexpr unsigned long long kBestEmpty = (0x7F800000ull << 32) | 0xFFFFFFFFull;

__device__ __forceinline__ float screen_threshold(float R, float qs, float eps) {
    const float inf = __builtin_huge_valf();
    if (!(R < inf)) return inf;  // no finite value known yet
    // exact <= R  =>  ||x||^2 - 2 x.q <= R - ||q||^2 + eps
    return round_up_f((double)R - (double)qs + (double)eps);
}

// Exact value of one (query, row) pair in the arm's operation order, loads
// issued U 16-byte chunks at a time.
template <int ARM, bool VEC4, int U = 4>
__device__ __forceinline__ float exact_f32(const float* __restrict__ q, const float* __restrict__ y,
                                           int64_t d) {
    if (!VEC4) return exact_pair<float, ARM>(q, y, d, 0.0f, 0.0f);
    const float4* q4 = reinterpret_cast<const float4*>(q);
    const float4* y4 = reinterpret_cast<const float4*>(y);
    const int n4 = (int)(d >> 2);
    float acc = 0.0f;
    int c = 0;
    for (; c + U <= n4; c += U) {
        float4 a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            a[u] = q4[c + u];
            b[u] = y4[c + u];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (ARM == ARM_EUCLID_FMA) {
                float d0 = a[u].x - b[u].x, d1 = a[u].y - b[u].y, d2 = a[u].z - b[u].z, d3 = a[u].w - b[u].w;
                acc = __builtin_fmaf(d0, d0, acc);
                acc = __builtin_fmaf(d1, d1, acc);
                acc = __builtin_fmaf(d2, d2, acc);
                acc = __builtin_fmaf(d3, d3, acc);
            } else {
                float d0 = a[u].x - b[u].x, d1 = a[u].y - b[u].y, d2 = a[u].z - b[u].z, d3 = a[u].w - b[u].w;
                acc = acc + d0 * d0;
                acc = acc + d1 * d1;
                acc = acc + d2 * d2;
                acc = acc + d3 * d3;
            }
        }
    }
    for (; c < n4; ++c) {
        float4 a = q4[c], b = y4[c];
        if (ARM == ARM_EUCLID_FMA) {
            float d0 = a.x - b.x, d1 = a.y - b.y, d2 = a.z - b.z, d3 = a.w - b.w;
            acc = __builtin_fmaf(d0, d0, acc);
            acc = __builtin_fmaf(d1, d1, acc);
            acc = __builtin_fmaf(d2, d2, acc);
            acc = __builtin_fmaf(d3, d3, acc);
        } else {
            float d0 = a.x - b.x, d1 = a.y - b.y, d2 = a.z - b.z, d3 = a.w - b.w;
            acc = acc + d0 * d0;
            acc = acc + d1 * d1;
            acc = acc + d2 * d2;
            acc = acc + d3 * d3;
        }
    }
    return acc;
}

// Workgroups per CU: three (at most 168 VGPRs, 53 KB LDS) with d <= 64; the
// LDS queues allow no more above.  A third wave per SIMD keeps the matrix core
// fed while the other two wait at a tile barrier.
__host__ __device__ constexpr int gram_f32_wgs_per_cu(int ng) { return ng <= 8 ? 3 : 2; }

// (__launch_bounds__' second argument is waves per SIMD: workgroups per CU x
// waves per workgroup / 4.)
template <int NG, int ARM, bool VEC4>
__global__ __launch_bounds__(GramShape<(NG > 16)>::threads, (gram_f32_wgs_per_cu(NG) * GramShape<(NG > 16)>::waves / 4))
void knn_gram_f32_kernel(GramArgs32 a) {
    constexpr bool W16 = NG > 16;     // the wide shape (GramShape)
    typedef GramShape<W16> SH;
    constexpr int QPW = SH::qpw;
    constexpr int QPB = SH::qpb;
    constexpr int WV = SH::waves;     // waves per workgroup
    constexpr int NT = SH::threads;   // threads per workgroup
    constexpr int DP = NG * 8;        // padded feature count
    constexpr int CPR = DP / 4;       // 16-byte chunks per tile row
    // LDS row stride (floats): DP + 4, an odd number of 16-byte chunks, so
    // the A-operand ds_read_b128 of 16 consecutive rows (one chunk column)
    // hit 16 distinct groups of four banks.  Narrow rows of 128 floats are
    // kept in pairs instead: slot s (0..15) holds rows s and s + 16 back to
    // back (1 KB, one wave-wide direct load) and slots are 2 DP + 4 floats
    // apart, so rows 0..15 (and 16..31) still fall on distinct bank groups.
    constexpr int STRIDE = DP + 4;
    constexpr bool PAIRS = !W16 && NG == 16;
    constexpr int SLOT = 2 * DP + 4;
    constexpr int TILE_FL = PAIRS ? 16 * SLOT : kBn * STRIDE;
    constexpr int TILE_F4 = kBn * DP / 4;
    constexpr int PF = (TILE_F4 + NT - 1) / NT;
    constexpr int QQ = DP / 4;        // wide: features per lane-group quarter
    constexpr int NQR = W16 ? QQ / 4 : NG;  // 16-byte query-operand chunks per lane

    __shared__ __attribute__((aligned(16))) float tileA[TILE_FL];
    __shared__ __attribute__((aligned(16))) float tileB[TILE_FL];
    __shared__ __attribute__((aligned(16))) float tnA[kBn];
    __shared__ __attribute__((aligned(16))) float tnB[kBn];
    __shared__ WaveLds<QPW> wl[WV];

    // Kernel arguments as locals: they stay in SGPRs.
    const float* __restrict__ Q = a.q;
    const float* __restrict__ X = a.x;
    const float* __restrict__ QSQ = a.qsq;
    const float* __restrict__ XSQ = a.xsq;
    unsigned int* __restrict__ SHARED_R = a.shared_r;
    const int64_t nq = a.nq, nt = a.nt, d = a.d;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
    // narrow: h = lane / 32 picks the 4-row group of each 8-row slab;
    // wide: g = lane / 16 picks the 4-row group of each 16-row half and the
    // feature quarter.  jl: the lane's query within the wave.
    const int h = W16 ? (lane >> 4) : (lane >> 5);
    const int jl = lane & (QPW - 1);
    WaveLds<QPW>& L = wl[w];
    const float inf = __builtin_huge_valf();
    // Tile row of value r of this lane.
    auto row_of = [&](int r) -> int {
        return W16 ? 16 * (r >> 2) + 4 * h + (r & 3) : 8 * (r >> 2) + 4 * h + (r & 3);
    };
    // LDS float offset of 16-byte chunk c of tile row r.
    auto row_at = [&](int r) -> int { return PAIRS ? (r & 15) * SLOT + (r >> 4) * DP : r * STRIDE; };
    auto chunk_at = [&](int r, int c) -> int { return row_at(r) + 4 * c; };

    // ---- work split (StreamSplit): this workgroup's range of (query block,
    //      tile) units, panel-major; each piece of a job in the range is a
    //      segment with its own best pair [slot][nq], merged at the end. ----
    const StreamSplit sp(nq, nt, QPB, kBn, a.grid_wgs);
    const int64_t wg = xcd_grouped_wg(blockIdx.x, gridDim.x);
    const int64_t u_hi = ((wg + 1) * sp.P < sp.T) ? (wg + 1) * sp.P : sp.T;
    for (int64_t u = wg * sp.P; u < u_hi;) {
    int64_t panel, qblock, tile0, left;
    sp.decode(u, panel, qblock, tile0, left);
    const int64_t tile1 = tile0 + ((left < u_hi - u) ? left : (u_hi - u));
    const int64_t slot = sp.slot(wg, panel, qblock);
    float* __restrict__ LV = a.part_val + slot * nq;
    uint32_t* __restrict__ LI = a.part_idx + slot * nq;
    const int64_t qwave = qblock * QPB + w * QPW;  // first query of this wave
    const int64_t qmine = qwave + jl;
    const bool qvalid = qmine < nq;
    const int64_t t_begin = tile0 * kBn;
    int64_t t_end = tile1 * kBn;
    if (t_end > nt) t_end = nt;

    // Feature of chunk element e of the lane's query-operand chunk i.
    auto qfeat = [&](int i, int e) -> int64_t {
        return W16 ? (int64_t)h * QQ + 4 * i + e : (int64_t)8 * i + 4 * h + e;
    };

    // ---- segment start: the loads first, from clamped rows so that they are
    //      unconditional and all in flight together (a segment of k-means
    //      assignment lasts only 32 tiles), then the per-query state.  Wide
    //      rows (NG > 8) load the operand later: early it would spill. ----
    constexpr bool kEarlyQ = NG <= 8;
    const int64_t qrow = qvalid ? qmine : nq - 1;
    const float qsq_l = QSQ[qrow];
    const float r0_l = SHARED_R ? __uint_as_float(SHARED_R[qrow]) : inf;
    float4 qreg[NQR];
    if (VEC4 && kEarlyQ) {
        const float* qp = Q + qrow * d;
#pragma unroll
        for (int g = 0; g < NQR; ++g) {
            const int64_t c = qfeat(g, 0);
            const float4 v = *reinterpret_cast<const float4*>(qp + (c < d ? c : d - 4));
            qreg[g] = (qvalid && c < d) ? v : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }

    // ---- per-query constants, queues ----
    uint32_t cntr = 0u;  // queued candidates of query jl
    if (lane < QPW) {
        const float qsq = qvalid ? qsq_l : 0.0f;
        L.thr[lane] = qvalid ? inf : -inf;
        L.qs[lane] = qsq;
        L.eps[lane] = (float)(a.eps_rel * ((double)qsq + (double)a.stats->xsq_max) + a.eps_abs);
        // |screen distance - exact| <= eps holds while no sum can overflow:
        // norms well inside the float range.
        const bool sv = qvalid && ((double)qsq + (double)a.stats->xsq_max <= 0x1p124) && (L.eps[lane] < inf);
        L.mode[lane] = sv ? 0u : 1u;
    }
    if (lane < QPW) L.best[lane] = kBestEmpty;
    // Strips that start late begin from the bound earlier strips have reached.
    if (SHARED_R && lane < QPW && qvalid)
        L.thr[lane] = fminf(L.thr[lane], screen_threshold(r0_l, L.qs[lane], L.eps[lane]));

    // ---- query operand: qreg[i] = scale * q[qfeat(i, 0..3)] (aligned rows:
    //      one 16-byte load per chunk) ----
    {
        const float scale = -2.0f;
        const float* qp = Q + qmine * d;
        if (VEC4) {
            if (!kEarlyQ) {
#pragma unroll
                for (int g = 0; g < NQR; ++g) {
                    const int64_t c = qfeat(g, 0);
                    qreg[g] = (qvalid && c < d) ? *reinterpret_cast<const float4*>(qp + c)
                                                : make_float4(0.f, 0.f, 0.f, 0.f);
                }
            }
#pragma unroll
            for (int g = 0; g < NQR; ++g) {
                qreg[g].x *= scale;
                qreg[g].y *= scale;
                qreg[g].z *= scale;
                qreg[g].w *= scale;
            }
        } else {
#pragma unroll
            for (int g = 0; g < NQR; ++g) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int64_t c = qfeat(g, e);
                    v[e] = (qvalid && c < d) ? qp[c] * scale : 0.0f;
                }
                qreg[g] = make_float4(v[0], v[1], v[2], v[3]);
            }
        }
    }

    // ---- tile prefetch into registers (rows past the strip: zeros, norm +inf) ----
    // Each thread owns PF fixed 16-byte chunks of the tile: row pf_r[p], column
    // chunk pf_c[p]; its source pointer walks down one tile (kBn rows) per step.
    const uint32_t t_end32 = (uint32_t)t_end;
    int pf_r[PF];
    bool pf_on[PF];
    const float* pf_src[PF];
#pragma unroll
    for (int p = 0; p < PF; ++p) {
        const int f = tid + NT * p;
        pf_r[p] = f / (DP / 4);
        const int c4 = f % (DP / 4);
        pf_on[p] = (f < TILE_F4) && (4 * c4 < d);
        pf_src[p] = X + (t_begin + pf_r[p]) * d + 4 * c4;
    }
    // Whole tiles of rows without padded columns load unconditionally.
    const bool pf_fast = VEC4 && (PF * NT == TILE_F4) && (d == DP);
    // Wide rows: a thread's chunks lie in one column, PF_RPP rows apart, so one
    // pointer and uniform offsets address them (eight live 64-bit pointers
    // would not fit next to the 64-register query operand).
    constexpr int PF_RPP = (NT % (DP / 4) == 0) ? NT / (DP / 4) : 0;
    constexpr bool PF_ONE_PTR = W16 && PF_RPP > 0;
    // The address, row and on-flag of prefetch chunk p (wide rows: derived
    // from chunk 0's).
#define MLRS_PF_SRC(p) (PF_ONE_PTR ? pf_src[0] + (int64_t)(p) * PF_RPP * d : pf_src[p])
#define MLRS_PF_ROW(p) (PF_ONE_PTR ? pf_r[0] + (p) * PF_RPP : pf_r[p])
#define MLRS_PF_ON(p) (PF_ONE_PTR ? pf_on[0] : pf_on[p])
#define MLRS_PREFETCH(T0)                                                                    \
    do {                                                                                     \
        const uint32_t t0_ = (uint32_t)(T0);                                                 \
        if (pf_fast && t_end32 - t0_ >= (uint32_t)kBn) { /* not t0 + kBn: no wrap */        \
            _Pragma("unroll") for (int p = 0; p < PF; ++p) pf[p] = gload4(MLRS_PF_SRC(p));   \
        } else {                                                                             \
        _Pragma("unroll") for (int p = 0; p < PF; ++p) {                                     \
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);                                      \
            const uint32_t t = t0_ + (uint32_t)MLRS_PF_ROW(p);                               \
            if (MLRS_PF_ON(p) && t < t_end32) {                                              \
                const float* src = MLRS_PF_SRC(p);                                           \
                if (VEC4) {                                                                  \
                    v = gload4(src);                                                         \
                } else {                                                                     \
                    const int c0_ = (int)((tid + NT * p) % (DP / 4)) * 4;                    \
                    float e4[4];                                                             \
                    _Pragma("unroll") for (int e = 0; e < 4; ++e) e4[e] =                    \
                        (c0_ + e < d) ? src[e] : 0.0f;                                       \
                    v = make_float4(e4[0], e4[1], e4[2], e4[3]);                             \
                }                                                                            \
            }                                                                                \
            pf[p] = v;                                                                       \
        }                                                                                    \
        }                                                                                    \
        _Pragma("unroll") for (int p = 0; p < (PF_ONE_PTR ? 1 : PF); ++p) pf_src[p] += kBn * d; \
        if (tid < kBn) {                                                                     \
            const uint32_t t = t0_ + (uint32_t)tid;                                          \
            pfn = (t < t_end32) ? XSQ[t] : inf;                                              \
        }                                                                                    \
    } while (0)

    // ---- flush: every queued pair of the wave evaluated in lane-parallel
    //      batches, kept with a 64-bit LDS atomicMin on (value, index) ----
#define MLRS_FLUSH()                                                                      \
    do {                                                                                     \
        const uint32_t c_ = (lane < QPW) ? cntr : 0u;                                        \
        uint32_t incl_ = c_;                                                                 \
        _Pragma("unroll") for (int m_ = 1; m_ < QPW; m_ <<= 1) {                             \
            const uint32_t o_ = (uint32_t)__shfl_up((int)incl_, m_, 64);                     \
            if ((lane & (QPW - 1)) >= m_) incl_ += o_;                                       \
        }                                                                                    \
        const uint32_t total_ = (uint32_t)__shfl((int)incl_, QPW - 1, 64);                   \
        if (lane < QPW) L.off[lane] = incl_ - c_;                                            \
        for (uint32_t base_ = 0; base_ < total_; base_ += 64) {                              \
            const uint32_t e_ = base_ + (uint32_t)lane;                                      \
            if (e_ < total_) {                                                               \
                int j_ = 0;                                                                  \
                _Pragma("unroll") for (int m_ = QPW / 2; m_ >= 1; m_ >>= 1) if (L.off[j_ + m_] <= e_) \
                    j_ += m_;                                                                \
                const uint32_t t_ = L.qidx[j_][e_ - L.off[j_]];                              \
                const float v_ = exact_f32<ARM, VEC4>(Q + (qwave + j_) * d, X + (int64_t)t_ * d, d); \
                if (v_ == v_)                                                                \
                    atomicMin(&L.best[j_], ((unsigned long long)__float_as_uint(v_) << 32) | t_); \
            }                                                                                \
        }                                                                                    \
        cntr = 0u;                                                                           \
        qlo = qlo0;                                                                          \
        if (lane < QPW) {                                                                    \
            float R_ = __uint_as_float((uint32_t)(L.best[lane] >> 32));                      \
            if (SHARED_R && qvalid && R_ < inf) {                                            \
                const unsigned int old_ = atomicMin(&SHARED_R[qmine], __float_as_uint(R_));  \
                R_ = fminf(R_, __uint_as_float(old_));                                       \
            }                                                                                \
            L.thr[lane] = fminf(L.thr[lane], screen_threshold(R_, L.qs[lane], L.eps[lane])); \
        }                                                                                    \
    } while (0)

    float4 pf[PF];
    float pfn = 0.0f;
    if (t_begin < t_end) MLRS_PREFETCH(t_begin);
    __syncthreads();  // per-wave LDS init visible to the wave
    // Sign-bit screen (below): waves whose valid queries all have mode 0 (no
    // screen sum can overflow), where a NaN screen value comes only from a row
    // holding a NaN, whose exact value is NaN and never kept, so the screen may
    // drop it.  The wide shape measured no faster with it.
    constexpr bool kSignScreen = !W16;
    const bool nan_free =
        kSignScreen && __builtin_amdgcn_ballot_w64(lane < QPW && qvalid && L.mode[lane] != 0u) == 0;

    float thr = L.thr[jl];
    const float eps2 = 2.0f * L.eps[jl];  // exact doubling
    // A lower bound on the screen values of the rows in query jl's queue.  A NaN
    // screen value can hide a finite exact value only where a sum may overflow,
    // so queries of mode 1 keep -inf and never drop queued rows; otherwise NaN
    // screen values come from rows holding a NaN, whose exact values are NaN and
    // never kept.
    const float qlo0 = (L.mode[jl] == 0u) ? inf : -inf;
    float qlo = qlo0;
    int tiles = 0;
    // One tile: CUR receives the rows at T0 from the staging registers, which
    // then take the next tile.
    auto tile_step = [&](float (&cur)[TILE_FL], float* __restrict__ tncur, int64_t t0) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            const int f = tid + NT * p;
            if (f < TILE_F4) {
                const int r = f / (DP / 4);
                const int c4 = f % (DP / 4);
                *reinterpret_cast<float4*>(&cur[0] + chunk_at(r, c4)) = pf[p];
            }
        }
        if (tid < kBn) tncur[tid] = pfn;
        __syncthreads();
        if (t_end32 - (uint32_t)t0 > (uint32_t)kBn) MLRS_PREFETCH(t0 + kBn);

        // The lane's tile values: narrow, acc[r] = row row_of(r); wide, r < 4
        // in acc0 (the first 16-row half) and r >= 4 in acc1.
        f32x16 acc;
        f32x4 acc0, acc1;
        if constexpr (!W16) {
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                float4 n4 = *reinterpret_cast<const float4*>(&tncur[8 * g4 + 4 * h]);
                acc[4 * g4 + 0] = n4.x;
                acc[4 * g4 + 1] = n4.y;
                acc[4 * g4 + 2] = n4.z;
                acc[4 * g4 + 3] = n4.w;
            }
            // A operands double-buffered: the next group's LDS read is issued
            // before the current group's four MFMAs (the scheduling barriers keep
            // that order), so its latency hides under ~256 MFMA cycles.
            const float* arow = &cur[row_at(jl) + 4 * h];
            float4 av = *reinterpret_cast<const float4*>(arow);
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                float4 an = av;
                if (g + 1 < NG) an = *reinterpret_cast<const float4*>(arow + 8 * (g + 1));
                __builtin_amdgcn_sched_barrier(0);
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.x, qreg[g].x, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.y, qreg[g].y, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.z, qreg[g].z, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.w, qreg[g].w, acc, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                av = an;
            }
        } else {
            const float4 n0 = *reinterpret_cast<const float4*>(&tncur[4 * h]);
            const float4 n1 = *reinterpret_cast<const float4*>(&tncur[16 + 4 * h]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                acc0[r] = (&n0.x)[r];
                acc1[r] = (&n1.x)[r];
            }
            // A operands: this lane's rows jl and 16 + jl, its quarter's chunk
            // i, one group ahead; each chunk feeds eight MFMAs (four k-steps
            // on each half).
            const float* t0p = &cur[0];
            const int c0 = h * (QQ / 4);
            float4 av0 = *reinterpret_cast<const float4*>(t0p + chunk_at(jl, c0));
            float4 av1 = *reinterpret_cast<const float4*>(t0p + chunk_at(16 + jl, c0));
#pragma unroll
            for (int i = 0; i < NQR; ++i) {
                float4 an0 = av0, an1 = av1;
                if (i + 1 < NQR) {
                    an0 = *reinterpret_cast<const float4*>(t0p + chunk_at(jl, c0 + i + 1));
                    an1 = *reinterpret_cast<const float4*>(t0p + chunk_at(16 + jl, c0 + i + 1));
                }
                __builtin_amdgcn_sched_barrier(0);
                acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av0.x, qreg[i].x, acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(av1.x, qreg[i].x, acc1, 0, 0, 0);
                acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av0.y, qreg[i].y, acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(av1.y, qreg[i].y, acc1, 0, 0, 0);
                acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av0.z, qreg[i].z, acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(av1.z, qreg[i].z, acc1, 0, 0, 0);
                acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av0.w, qreg[i].w, acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(av1.w, qreg[i].w, acc1, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                av0 = an0;
                av1 = an1;
            }
        }
        auto val = [&](int r) -> float {
            if constexpr (W16) return r < 4 ? acc0[r] : acc1[r - 4];
            else return acc[r];
        };

        // ---- tighten with this tile's smallest expansion value ----
        {
            float m = inf;
#pragma unroll
            for (int r = 0; r < SH::vals; ++r) m = fminf(m, val(r));  // NaN ignored; past-end rows are +inf
            if (W16) m = fminf(m, shfl_xor_f(m, 16));
            m = fminf(m, shfl_xor_f(m, 32));
            if (m < inf) {
                // m + 2 eps rounded to nearest, then stepped up by at least one
                // ulp (2^-126 near zero): an upper bound of the exact sum
                const float s_ = m + eps2;
                thr = fminf(thr, s_ + (__builtin_fabsf(s_) * 0x1p-23f + 0x1p-126f));
            }
            // Rows queued on earlier tiles whose screen values all exceed
            // the tightened threshold cannot be the nearest row (nor tie
            // with it): the queue restarts before this tile's rows join it.
            // Each new running minimum used to leave its predecessors queued
            // (about ln(tiles) rows per query at each flush).
            if (qlo > thr) {
                cntr = 0u;
                qlo = inf;
            }
            qlo = fminf(qlo, m);
        }

        // ---- screen: value r of the lane is tile row row_of(r) for query jl.
        //      Passing rows are appended to the query's queue at cntr (kept in
        //      registers, equal in every lane of the query); the lanes of a
        //      query write in lane order, each after the earlier lanes' entries. ----
        uint32_t m = 0;
        if (kSignScreen && nan_free) {
            // pass <=> thr - value >= +0: the rounded difference has the sign
            // of the exact one (x - x = +0), thr + 0 turns a -0 threshold into
            // +0, and v_alignbit shifts each sign bit into the fail mask:
            // two instructions per value and no compare-mask hazards
            const float t_ = thr + 0.0f;
            uint32_t f = 0;
#pragma unroll
            for (int r = SH::vals - 1; r >= 0; --r)
                f = __builtin_amdgcn_alignbit(f, __float_as_uint(t_ - val(r)), 31);
            m = f ^ ((1u << SH::vals) - 1u);
        } else {
#pragma unroll
            for (int r = 0; r < SH::vals; ++r) m |= (uint32_t)!(val(r) > thr) << r;
        }
        if (!qvalid) m = 0;
        // Partial tile (the segment's last): rows past the segment are not
        // candidates.  Rows left are compared in 32 bits, a scalar branch; a
        // 64-bit ordered compare is a vector instruction, and the compiler
        // then computed this mask on every tile.
        if (t_end32 - (uint32_t)t0 < (uint32_t)kBn) {
#pragma unroll
            for (int r = 0; r < SH::vals; ++r)
                if ((uint32_t)t0 + (uint32_t)row_of(r) >= t_end32) m &= ~(1u << r);
        }
        if (__builtin_amdgcn_ballot_w64(m != 0)) {
            const uint32_t c = (uint32_t)__builtin_popcount(m);
            uint32_t before, total;
            if constexpr (W16) {
                // exclusive prefix and total over the query's four lanes (h = 0..3)
                const uint32_t u1 = (uint32_t)__shfl_up((int)c, 16, 64);
                const uint32_t s1 = c + (h >= 1 ? u1 : 0u);
                const uint32_t u2 = (uint32_t)__shfl_up((int)s1, 32, 64);
                const uint32_t incl = s1 + (h >= 2 ? u2 : 0u);
                before = incl - c;
                total = (uint32_t)__shfl((int)incl, 48 + jl, 64);
            } else {
                const uint32_t co = shfl_xor_u(c, 32);
                before = h ? co : 0u;
                total = c + co;
            }
            uint32_t pos = cntr + before;
            const uint32_t tb = (uint32_t)t0;
            while (m) {
                const int r = __builtin_ctz(m);
                m &= m - 1;
                L.qidx[jl][pos++] = tb + (uint32_t)row_of(r);
            }
            cntr += total;
        }
        // ---- flush queries whose queue could overflow on the next tile ----
        if (__builtin_amdgcn_ballot_w64(lane < QPW && cntr > (uint32_t)kFlushAt)) {
            if (lane < QPW) L.thr[lane] = fminf(L.thr[lane], thr);
            MLRS_FLUSH();
            thr = L.thr[jl];
        }
        // ---- pick up thresholds tightened by other strips of these queries ----
        rotate_wave_priority((uint32_t)tiles + 1u, gram_f32_wgs_per_cu(NG));
        if (SHARED_R && (++tiles % kShareEvery) == 0) {
            if (lane < QPW && qvalid) {
                const float R = __uint_as_float(SHARED_R[qmine]);
                L.thr[lane] = fminf(fminf(L.thr[lane], thr), screen_threshold(R, L.qs[lane], L.eps[lane]));
            }
            thr = L.thr[jl];
        }
    };
    for (int64_t t0 = t_begin; t0 < t_end; t0 += 2 * kBn) {
        tile_step(tileA, tnA, t0);
        if (t0 + kBn < t_end) tile_step(tileB, tnB, t0 + kBn);
    }

    // ---- final flush of every non-empty queue ----
    if (__builtin_amdgcn_ballot_w64(lane < QPW && cntr > 0u)) MLRS_FLUSH();
#undef MLRS_FLUSH
#undef MLRS_PREFETCH
#undef MLRS_PF_SRC
#undef MLRS_PF_ROW
#undef MLRS_PF_ON

    // ---- the kept pair is this segment's ----
    if (lane < QPW && qvalid) {
        const unsigned long long b = L.best[lane];
        LV[qmine] = __uint_as_float((uint32_t)(b >> 32));
        LI[qmine] = (uint32_t)b;
    }
    u += tile1 - tile0;
    __syncthreads();  // LDS state and tile buffers are reused by the next segment
    }
}

// The strip merge, one lane per query: the segment lists are one pair each, so
// the merge is a (value, index) minimum.
__global__ __launch_bounds__(256) void knn_merge1_f32_kernel(GramArgs32 a) {
    const int64_t qg = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (qg >= a.nq) return;
    float lv = a.part_val[qg];
    uint32_t li = a.part_idx[qg];
    const StreamSplit sp(a.nq, a.nt, a.qpb, kBn, a.grid_wgs);
    const int64_t nsl = sp.slots_of(qg / a.qpb);
    for (int64_t s = 1; s < nsl; ++s) {
        const float v = a.part_val[s * a.nq + qg];
        const uint32_t ix = a.part_idx[s * a.nq + qg];
        if (pair_less<float>(v, ix, lv, li)) {
            lv = v;
            li = ix;
        }
    }
    emit_pair(a.mode, a.q, a.x, a.qsq, a.xsq, a.d, 1, qg, 0, lv, li, a.out_val, a.out_idx);
}

// The shared per-query threshold words start at +inf (as float bits).
__global__ void fill_inf_bits_kernel(unsigned int* p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0x7F800000u;
}

template <int NG, bool VEC4>
hipError_t launch_ng(const GramArgs32& a, int arm, hipStream_t s) {
    dim3 grid((unsigned)StreamSplit(a.nq, a.nt, a.qpb, kBn, a.grid_wgs).G);
    const dim3 block(GramShape<(NG > 16)>::threads);
    if (arm == ARM_EUCLID_MULADD)
        hipLaunchKernelGGL((knn_gram_f32_kernel<NG, ARM_EUCLID_MULADD, VEC4>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((knn_gram_f32_kernel<NG, ARM_EUCLID_FMA, VEC4>), grid, block, 0, s, a);
    return hipGetLastError();
}

template <bool VEC4>
hipError_t launch_d(const GramArgs32& a, int arm, hipStream_t s) {
    const int ng = (int)((a.d + 7) / 8);
    // the split and the merge must see the query-block size of the shape
    if (a.qpb != (ng > 16 ? kQpbWide : kQpbNarrow)) return hipErrorInvalidValue;
    if (ng <= 2) return launch_ng<2, VEC4>(a, arm, s);
    if (ng <= 4) return launch_ng<4, VEC4>(a, arm, s);
    if (ng <= 8) return launch_ng<8, VEC4>(a, arm, s);
    if (ng <= 12) return launch_ng<12, VEC4>(a, arm, s);
    if (ng <= 16) return launch_ng<16, VEC4>(a, arm, s);
    if (ng <= 24) return launch_ng<24, VEC4>(a, arm, s);
    return launch_ng<32, VEC4>(a, arm, s);
}

}  // namespace

int gram_f32_queries_per_block(int64_t d) { return d > 128 ? kQpbWide : kQpbNarrow; }


void gram_f32_split(int64_t nq, int64_t nt, int64_t d, int cus, int64_t* grid_wgs, int* nslots) {
    const int64_t qpb = gram_f32_queries_per_block(d);
    const StreamSplit full(nq, nt, qpb, kBn, 1);
    // one resident round (gram_f32_wgs_per_cu workgroups per CU), but at
    // least 16 tiles each
    int64_t g0 = gram_f32_wgs_per_cu((int)((d + 7) / 8)) * (int64_t)(cus > 0 ? cus : 1);
    if (g0 > full.T / 16) g0 = full.T / 16;
    if (g0 < 1) g0 = 1;
    *grid_wgs = g0;
    *nslots = (int)StreamSplit(nq, nt, qpb, kBn, g0).nslots();
}

int gram_f32_max_d() { return 256; }

hipError_t launch_gram_f32_prep(const GramArgs32& a, hipStream_t s) {
    if (!a.shared_r) return hipSuccess;
    hipLaunchKernelGGL(fill_inf_bits_kernel, dim3((unsigned)((a.nq + 255) / 256)), dim3(256), 0, s, a.shared_r, a.nq);
    return hipGetLastError();
}

hipError_t launch_gram_f32_merge(const GramArgs32& a, hipStream_t s) {
    hipLaunchKernelGGL(knn_merge1_f32_kernel, dim3((unsigned)((a.nq + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_gram_f32(const GramArgs32& a, int arm, hipStream_t s) {
    if (a.k != 1 || (arm != ARM_EUCLID_MULADD && arm != ARM_EUCLID_FMA)) return hipErrorInvalidValue;
    const bool vec4 = (a.d % 4 == 0) && ((reinterpret_cast<uintptr_t>(a.q) & 15) == 0) &&
                      ((reinterpret_cast<uintptr_t>(a.x) & 15) == 0);
    return vec4 ? launch_d<true>(a, arm, s) : launch_d<false>(a, arm, s);
}

}  // namespace mlrs
