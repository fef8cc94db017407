// Fused f64 Gram-MFMA nearest row with exact rescoring (gfx950): the k-means
// assignment (argmin_dist_rows, crates/mlrs-kernels/src/kmeans.rs:284-310) in
// f64, d <= 256.
//
// Shape of one workgroup: 4 waves x 16 queries = 64 queries, walking one
// segment of index rows 16 at a time with v_mfma_f64_16x16x4f64.
//  * Lane l of a wave owns query l%16 and lane group g = l/16.  The K
//    dimension is split into four contiguous quarters of NS columns: at
//    k-step s, group g supplies column g*NS + s of both operands, so each
//    lane's A operand is a contiguous run of its tile row (ds_read_b128
//    feeds two k-steps) and its B operand (the query, pre-scaled by -2) is
//    held in VGPRs for the whole segment.
//  * The MFMA result layout is D[l/16 + 4r][l%16], r = 0..3: lane l scores
//    tile rows g, g+4, g+8, g+12 against its query.
//  * The screen, the per-query queues, the exact rescoring in the arm's
//    operation order and the stream-K split with a shared per-query bound are
//    those of the f32 kernel, in double; the bound starts from a sample of the
//    rows (knn_seed_f64_kernel).
// The thresholds are computed in double with a margin for their own
// rounding folded into the error bound (the f32 kernel rounds up in double
// instead).
#include "knn_common.hpp"
#include "knn_kernels.hpp"

namespace mlrs {

namespace {

constexpr int kWaves = 4;
constexpr int kQpw = 16;               // queries per wave (MFMA N dimension)
constexpr int kQpb = kWaves * kQpw;    // queries per workgroup
constexpr int kBn = 16;                // index rows per tile (MFMA M dimension)
constexpr int kQcap = 48;              // queued candidates per query (two workgroups still fit a CU's LDS)
constexpr int kFlushAt = kQcap - kBn;  // flush when a queue may overflow on the next tile
constexpr int kShareEvery = 32;        // tiles between reads of the shared bound
constexpr int kMaxD = 256;

typedef double f64x4 __attribute__((ext_vector_type(4)));

struct WaveLds64 {
    uint32_t qidx[kQpw][kQcap];
    double thr[kQpw];
    double qs[kQpw];   // ||q||^2
    double eps[kQpw];  // screen error bound
};

__device__ __forceinline__ double screen_threshold64(double R, double qs, double eps) {
    const double inf = __builtin_huge_val();
    if (!(R < inf)) return inf;
    return ((R + __builtin_fabs(R) * 0x1p-48) - qs) + eps;
}

// Exact value of one (query, row) pair in the arm's operation order; loads
// issued two 16-byte pairs at a time when rows are 16-byte aligned (the d = 256
// kernel holds 128 VGPRs of query operand).
template <bool VEC2>
__device__ __forceinline__ double exact_f64(const double* __restrict__ q, const double* __restrict__ y, int64_t d) {
    if (!VEC2) return exact_pair<double, ARM_EUCLID_MULADD>(q, y, d, 0.0, 0.0);
    constexpr int U = 2;
    const double2* q2 = reinterpret_cast<const double2*>(q);
    const double2* y2 = reinterpret_cast<const double2*>(y);
    const int n2 = (int)(d >> 1);
    double acc = 0.0;
    int c = 0;
    for (; c < n2; c += U) {
        double2 a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (c + u < n2) {
                a[u] = q2[c + u];
                b[u] = y2[c + u];
            } else {
                a[u] = make_double2(0.0, 0.0);
                b[u] = make_double2(0.0, 0.0);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (c + u >= n2) break;
            const double e0a = a[u].x, e1a = a[u].y, e0b = b[u].x, e1b = b[u].y;
            const double d0 = e0a - e0b, d1 = e1a - e1b;
            acc = acc + d0 * d0;
            acc = acc + d1 * d1;
        }
    }
    return acc;
}

template <int NS, bool VEC2>
__global__ __launch_bounds__(256, 2) void knn_gram_f64_kernel(GramArgs64 a) {
    constexpr int DP = 4 * NS;             // padded feature count
    constexpr int STRIDE = DP + 2;         // LDS row stride (doubles): rows 16 bytes apart in the banks
    constexpr int CPT = DP / 2;            // 16-byte column pairs per tile row
    constexpr int RPG = 256 / CPT;         // tile rows one pass of the workgroup loads
    constexpr int PF = kBn / RPG;          // passes per tile
    static_assert(RPG >= 1 && kBn % RPG == 0, "tile fill shape");
    // Rows of whole kilobytes (d padded to 128 or 256) with 16-byte aligned
    // operands load the next tile straight into LDS (global_load_lds_dwordx4:
    // each wave instruction fills one contiguous kilobyte, half or all of a
    // row), so no registers hold it in flight; other shapes stage it through
    // registers.
    constexpr bool DIRECT = VEC2 && (DP % 128 == 0);
    constexpr int KB_PER_ROW = DP >= 128 ? DP / 128 : 1;  // 1 KB wave loads per tile row (DIRECT)
    constexpr int LOADS_PER_WAVE = kBn * KB_PER_ROW / kWaves;

    // The two tile buffers are distinct objects, so the compiler can tell the
    // direct loads into one from the reads of the other.
    __shared__ __attribute__((aligned(16))) double tileA[kBn][STRIDE];
    __shared__ __attribute__((aligned(16))) double tileB[kBn][STRIDE];
    __shared__ __attribute__((aligned(16))) double tnA[kBn];
    __shared__ __attribute__((aligned(16))) double tnB[kBn];
    __shared__ WaveLds64 wl[kWaves];

    const double* __restrict__ Q = a.q;
    const double* __restrict__ X = a.x;
    const double* __restrict__ QSQ = a.qsq;
    const double* __restrict__ XSQ = a.xsq;
    unsigned long long* __restrict__ SHARED_R = a.shared_r;
    const int64_t nq = a.nq, nt = a.nt, d = a.d;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: tile rows and LDS slots in SGPRs
    const int g = lane >> 4;   // lane group: K quarter / first tile row of the lane
    const int jl = lane & 15;  // query of the lane within the wave
    WaveLds64& L = wl[w];
    const double inf = __builtin_huge_val();
    // ---- work split (StreamSplit), as in the f32 kernel ----
    const StreamSplit sp(nq, nt, kQpb, kBn, a.grid_wgs);
    const int64_t wg = xcd_grouped_wg(blockIdx.x, gridDim.x);
    const int64_t u_hi = ((wg + 1) * sp.P < sp.T) ? (wg + 1) * sp.P : sp.T;
    for (int64_t u = wg * sp.P; u < u_hi;) {
    int64_t panel, qblock, tile0, left;
    sp.decode(u, panel, qblock, tile0, left);
    const int64_t tile1 = tile0 + ((left < u_hi - u) ? left : (u_hi - u));
    const int64_t slot = sp.slot(wg, panel, qblock);
    double* __restrict__ LV = a.part_val + slot * nq;
    uint32_t* __restrict__ LI = a.part_idx + slot * nq;

    const int64_t qwave = qblock * kQpb + w * kQpw;
    const int64_t qmine = qwave + jl;
    const bool qvalid = qmine < nq;
    const int64_t t_begin = tile0 * kBn;
    int64_t t_end = tile1 * kBn;
    if (t_end > nt) t_end = nt;
    const uint32_t t_end32 = (uint32_t)t_end;

    uint32_t cntr = 0u;  // queued candidates of query jl (equal in the four lanes of the query)
    if (lane < kQpw) {
        const double qsq = qvalid ? QSQ[qmine] : 0.0;
        L.thr[lane] = qvalid ? inf : -inf;
        L.qs[lane] = qsq;
        L.eps[lane] = a.eps_rel * (qsq + a.stats->xsq_max64) + a.eps_abs;
        if (qvalid) {
            LV[qmine] = inf;
            LI[qmine] = kSentinelIdx;
        }
    }
    if (SHARED_R && lane < kQpw && qvalid) {
        const double R0 = __longlong_as_double((long long)SHARED_R[qmine]);
        L.thr[lane] = fmin(L.thr[lane], screen_threshold64(R0, L.qs[lane], L.eps[lane]));
    }

    // ---- query operand: qreg[s] = scale * q[g*NS + s] ----
    double qreg[NS];
    {
        const double scale = -2.0;
        const double* qp = Q + qmine * d;
        if (VEC2) {  // 16-byte loads, all issued before use (NS and d even)
#pragma unroll
            for (int s = 0; s < NS; s += 2) {
                const int64_t c = (int64_t)g * NS + s;
                const double2 v = (qvalid && c < d) ? *reinterpret_cast<const double2*>(qp + c) : make_double2(0.0, 0.0);
                qreg[s] = v.x;
                qreg[s + 1] = v.y;
            }
#pragma unroll
            for (int s = 0; s < NS; ++s) qreg[s] *= scale;
        } else {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const int64_t c = (int64_t)g * NS + s;
                qreg[s] = (qvalid && c < d) ? qp[c] * scale : 0.0;
            }
        }
    }

    // ---- tile prefetch into registers.  Thread tid owns column pair c2 =
    //      tid % CPT of rows r0 + RPG*p (r0 = tid / CPT), p < PF: one walking
    //      row pointer, constant row and LDS offsets. ----
    const int pc2 = tid % CPT;
    const int pr0 = tid / CPT;
    const bool pon = (pr0 < RPG) && (2 * pc2 < d);
    const double* pfp = X + (t_begin + pr0) * d + 2 * pc2;
    const int64_t prow = (int64_t)RPG * d;  // elements between a thread's rows
    double2 pf[PF];
    double pfn = 0.0;
#define MLRS_PREFETCH64(T0)                                                                  \
    do {                                                                                     \
        const uint32_t t0_ = (uint32_t)(T0);                                                 \
        _Pragma("unroll") for (int p = 0; p < PF; ++p) {                                     \
            double2 v = make_double2(0.0, 0.0);                                              \
            const uint32_t t = t0_ + (uint32_t)(pr0 + RPG * p);                              \
            if (pon && t < t_end32) {                                                        \
                const double* src = pfp + p * prow;                                          \
                if (VEC2) {                                                                  \
                    v = *reinterpret_cast<const double2*>(src);                              \
                } else {                                                                     \
                    v.x = src[0];                                                            \
                    v.y = (2 * pc2 + 1 < d) ? src[1] : 0.0;                                  \
                }                                                                            \
            }                                                                                \
            pf[p] = v;                                                                       \
        }                                                                                    \
        pfp += kBn * d;                                                                      \
        if (tid < kBn) {                                                                     \
            const uint32_t t = t0_ + (uint32_t)tid;                                          \
            pfn = (t < t_end32) ? XSQ[t] : inf;                                              \
        }                                                                                    \
    } while (0)

// Flush: one query's queued rows evaluated exactly, the best of them against
// the segment's best pair (in memory).
#define MLRS_FLUSH64(J)                                                                      \
    do {                                                                                     \
        const int j_ = (J);                                                                  \
        const int64_t qg_ = qwave + j_;                                                      \
        const uint32_t n_ = bcast_u(cntr, j_);                                               \
        double e_ = inf;                                                                     \
        uint32_t t_ = kSentinelIdx;                                                          \
        if ((uint32_t)lane < n_) {                                                           \
            t_ = L.qidx[j_][lane];                                                           \
            e_ = exact_f64<VEC2>(Q + qg_ * d, X + (int64_t)t_ * d, d);                       \
            if (e_ != e_) { /* NaN is never admitted */                                      \
                e_ = inf;                                                                    \
                t_ = kSentinelIdx;                                                           \
            }                                                                                \
        }                                                                                    \
        wave_sort64<double>(e_, t_, lane);                                                   \
        if (lane == 0) {                                                                     \
            double R_ = LV[qg_];                                                             \
            if (pair_less<double>(e_, t_, R_, LI[qg_])) {                                    \
                LV[qg_] = R_ = e_;                                                           \
                LI[qg_] = t_;                                                                \
            }                                                                                \
            if (SHARED_R && R_ < inf) {                                                      \
                const unsigned long long old_ =                                              \
                    atomicMin(&SHARED_R[qg_], (unsigned long long)__double_as_longlong(R_)); \
                R_ = fmin(R_, __longlong_as_double((long long)old_));                        \
            }                                                                                \
            L.thr[j_] = fmin(L.thr[j_], screen_threshold64(R_, L.qs[j_], L.eps[j_]));        \
        }                                                                                    \
        if (jl == j_) cntr = 0u;                                                             \
    } while (0)

#define MLRS_STORE64(DST, TN)                                                                \
    do {                                                                                     \
        if (pr0 < RPG) {                                                                     \
            double* dst_ = &(DST)[pr0][2 * pc2];                                             \
            _Pragma("unroll") for (int p = 0; p < PF; ++p)                                   \
                *reinterpret_cast<double2*>(dst_ + p * RPG * STRIDE) = pf[p];                \
        }                                                                                    \
        if (tid < kBn) (TN)[tid] = pfn;                                                      \
    } while (0)

    // Direct loads of tile T0's rows into DST: wave w fills kilobytes
    // w*LOADS_PER_WAVE + i of the tile (row kb / KB_PER_ROW, its half kb %
    // KB_PER_ROW); a row past the segment is not loaded (its values are masked
    // out of the screen).  The row norms go through a register as in the
    // staged path.
    auto direct_load = [&](double (&dst)[kBn][STRIDE], uint32_t t0) {
        if constexpr (DIRECT) {
            // the row (and kilobyte) of each load is wave-uniform: a scalar
            // base plus the lane's 16-byte offset.  A whole tile of rows
            // without padded columns loads unconditionally (t0 + kBn could
            // wrap, so the rows left are compared).
            if (t_end32 - t0 >= (uint32_t)kBn && d == DP) {
#pragma unroll
                for (int i = 0; i < LOADS_PER_WAVE; ++i) {
                    const int kb = w * LOADS_PER_WAVE + i;
                    const int r = kb / KB_PER_ROW, half = kb % KB_PER_ROW;
                    const double* row = X + ((int64_t)(t0 + (uint32_t)r) * d + half * 128);
                    global_to_lds16(row + 2 * lane, &dst[r][half * 128]);
                }
            } else {
#pragma unroll
                for (int i = 0; i < LOADS_PER_WAVE; ++i) {
                    const int kb = w * LOADS_PER_WAVE + i;
                    const int r = kb / KB_PER_ROW, half = kb % KB_PER_ROW;
                    const double* row = X + ((int64_t)(t0 + (uint32_t)r) * d + half * 128);
                    if (t0 + (uint32_t)r < t_end32 && half * 128 + 2 * lane < d)
                        global_to_lds16(row + 2 * lane, &dst[r][half * 128]);
                }
            }
        }
        if (tid < kBn) {
            const uint32_t t = t0 + (uint32_t)tid;
            pfn = (t < t_end32) ? XSQ[t] : inf;
        }
    };
    if (DIRECT && d < DP) {
        // columns past d are never loaded: zero them once in both buffers
        // (they meet the query operand's zeros, and garbage could be NaN)
        const int pad = (int)(DP - d);
        for (int e = tid; e < kBn * pad; e += 256) {
            tileA[e / pad][d + e % pad] = 0.0;
            tileB[e / pad][d + e % pad] = 0.0;
        }
    }

    // The next tile is loaded (into registers, or straight into the other LDS
    // buffer) before this tile's MFMAs; staged registers are stored into the
    // other buffer right after them, so they are free again during the screen
    // and the rescoring.
    if (t_begin < t_end) {
        if (DIRECT) {
            direct_load(tileA, (uint32_t)t_begin);
            if (tid < kBn) tnA[tid] = pfn;
        } else {
            MLRS_PREFETCH64(t_begin);
            MLRS_STORE64(tileA, tnA);
        }
    }

    double thr = L.thr[jl];
    int tiles = 0;
    auto tile_step = [&](double (&cur)[kBn][STRIDE], double* tncur, double (&nxt)[kBn][STRIDE], double* tnnxt,
                         int64_t t0) {
        // this wave's direct loads into cur are done; the barrier makes every
        // wave's visible and ends every wave's reads of nxt
        if (DIRECT) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
        __syncthreads();
        const bool more = t0 + kBn < t_end;
        if (more) {
            if (DIRECT)
                direct_load(nxt, (uint32_t)(t0 + kBn));
            else
                MLRS_PREFETCH64(t0 + kBn);
        }

        // two accumulator chains (even and odd k-steps): one dependent chain
        // of f64 MFMAs leaves the matrix unit idle between its instructions
        f64x4 acc0, acc1;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            acc0[r] = tncur[g + 4 * r];
            acc1[r] = 0.0;
        }
        // A operand: this lane's tile row jl, columns g*NS + s; one 16-byte
        // read feeds two k-steps, the next pair is read one step ahead.
        const double* arow = &cur[jl][g * NS];
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
        f64x4 acc;
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = acc0[r] + acc1[r];
        if (more) {
            if (DIRECT) {
                if (tid < kBn) tnnxt[tid] = pfn;
            } else {
                MLRS_STORE64(nxt, tnnxt);
            }
        }

        // ---- screen: lane holds tile rows g + 4r for query jl ----
        uint32_t m = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) m |= (uint32_t)!(acc[r] > thr) << r;
        if (!qvalid) m = 0;
        if (t0 + kBn > t_end) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if ((uint32_t)t0 + (uint32_t)(g + 4 * r) >= t_end32) m &= ~(1u << r);
        }
        if (__builtin_amdgcn_ballot_w64(m != 0)) {
            // the query's four lanes (groups 0..3) append in group order
            const uint32_t c = (uint32_t)__builtin_popcount(m);
            // the counts of the query's other three lanes: groups g^1, g^2, g^3
            const uint32_t x1 = shfl_xor_u(c, 16), x2 = shfl_xor_u(c, 32), x3 = shfl_xor_u(x1, 32);
            const uint32_t c0 = (g == 0) ? c : (g == 1) ? x1 : (g == 2) ? x2 : x3;
            const uint32_t c1 = (g == 1) ? c : (g == 0) ? x1 : (g == 3) ? x2 : x3;
            const uint32_t c2 = (g == 2) ? c : (g == 3) ? x1 : (g == 0) ? x2 : x3;
            const uint32_t c3 = (g == 3) ? c : (g == 2) ? x1 : (g == 1) ? x2 : x3;
            uint32_t pos = cntr + (g > 0 ? c0 : 0u) + (g > 1 ? c1 : 0u) + (g > 2 ? c2 : 0u);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (m & (1u << r)) {
                    L.qidx[jl][pos] = (uint32_t)t0 + (uint32_t)(g + 4 * r);
                    ++pos;
                }
            }
            cntr += c0 + c1 + c2 + c3;
        }
        uint64_t mask = __builtin_amdgcn_ballot_w64(lane < kQpw && cntr > (uint32_t)kFlushAt);
        if (mask) {
            if (lane < kQpw) L.thr[lane] = fmin(L.thr[lane], thr);
            // the queued rows were stored by other lanes of this wave
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            while (mask) {
                const int j = __builtin_ctzll(mask);
                mask &= mask - 1;
                MLRS_FLUSH64(j);
            }
            thr = L.thr[jl];
        }
        rotate_wave_priority((uint32_t)tiles + 1u, 2);
        if (SHARED_R && (++tiles % kShareEvery) == 0) {
            if (lane < kQpw && qvalid) {
                const double R = __longlong_as_double((long long)SHARED_R[qmine]);
                L.thr[lane] = fmin(fmin(L.thr[lane], thr), screen_threshold64(R, L.qs[lane], L.eps[lane]));
            }
            thr = L.thr[jl];
        }
    };
    for (int64_t t0 = t_begin; t0 < t_end;) {
        tile_step(tileA, tnA, tileB, tnB, t0);
        t0 += kBn;
        if (t0 >= t_end) break;
        tile_step(tileB, tnB, tileA, tnA, t0);
        t0 += kBn;
    }
    {
        uint64_t mask = __builtin_amdgcn_ballot_w64(lane < kQpw && cntr > 0u);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        while (mask) {
            const int j = __builtin_ctzll(mask);
            mask &= mask - 1;
            MLRS_FLUSH64(j);
        }
    }
#undef MLRS_FLUSH64
#undef MLRS_STORE64
#undef MLRS_PREFETCH64
    u += tile1 - tile0;
    __syncthreads();  // LDS state and tile buffers are reused by the next segment
    }
}

// A query's best pair over its segments, and the output transform: the k-means
// pair with the centre-0 NaN rule of argmin_dist_rows
// (crates/mlrs-kernels/src/kmeans.rs:284-310), the boundary sqrt or identity.
__global__ __launch_bounds__(256) void knn_merge_f64_kernel(GramArgs64 a) {
    const int64_t qg = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (qg >= a.nq) return;
    const double inf = __builtin_huge_val();
    const StreamSplit sp(a.nq, a.nt, kQpb, kBn, a.grid_wgs);
    const int64_t nsl = sp.slots_of(qg / kQpb);
    double lv = a.part_val[qg];
    uint32_t li = a.part_idx[qg];
    for (int64_t s = 1; s < nsl; ++s) {
        const double v = a.part_val[s * a.nq + qg];
        const uint32_t ix = a.part_idx[s * a.nq + qg];
        if (pair_less<double>(v, ix, lv, li)) {
            lv = v;
            li = ix;
        }
    }
    if (a.mode == EMIT_KMEANS) {
        if (!(a.qsq[qg] < inf) || !(a.xsq[0] < inf)) {
            const double e0 = exact_pair<double, ARM_EUCLID_MULADD>(a.q + qg * a.d, a.x, a.d, 0.0, 0.0);
            if (e0 != e0) {
                lv = e0;
                li = 0;
            }
        }
        a.out_val[qg] = lv;
    } else {
        a.out_val[qg] = (a.mode == EMIT_SQRT) ? __builtin_sqrt(lv) : lv;
    }
    a.out_idx[qg] = (li == kSentinelIdx) ? 0u : li;
}

// Initial per-query bound: the smallest exact value over an evenly spaced
// sample of index rows (seed_kth_block), so that each segment's screen starts
// tight instead of at +inf.
__global__ __launch_bounds__(256) void knn_seed_f64_kernel(GramArgs64 a, int64_t nsamp) {
    seed_kth_block<double, ARM_EUCLID_MULADD, unsigned long long, 1>(a.q, a.x, a.nq, a.nt, a.d, 1, nsamp, nullptr,
                                                                     nullptr, a.shared_r);
}

template <int NS>
hipError_t launch_ns(const GramArgs64& a, bool vec2, hipStream_t s) {
    dim3 grid((unsigned)StreamSplit(a.nq, a.nt, kQpb, kBn, a.grid_wgs).G);
    if (vec2)
        hipLaunchKernelGGL((knn_gram_f64_kernel<NS, true>), grid, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((knn_gram_f64_kernel<NS, false>), grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

bool rows_vec2(const GramArgs64& a) {
    return (a.d % 2 == 0) && ((reinterpret_cast<uintptr_t>(a.q) & 15) == 0) &&
           ((reinterpret_cast<uintptr_t>(a.x) & 15) == 0);
}

}  // namespace

void gram_f64_split(int64_t nq, int64_t nt, int cus, int64_t* grid_wgs, int* nslots) {
    const StreamSplit full(nq, nt, kQpb, kBn, 1);
    // one resident round (two workgroups per CU), but at least 16 tiles each
    int64_t g0 = 2 * (int64_t)(cus > 0 ? cus : 1);
    if (g0 > full.T / 16) g0 = full.T / 16;
    if (g0 < 1) g0 = 1;
    *grid_wgs = g0;
    *nslots = (int)StreamSplit(nq, nt, kQpb, kBn, g0).nslots();
}

int gram_f64_max_d() { return kMaxD; }

hipError_t launch_gram_f64_prep(const GramArgs64& a, hipStream_t s) {
    // 512 rows, or the whole index
    const int64_t nsamp = a.nt < 512 ? a.nt : 512;
    hipLaunchKernelGGL(knn_seed_f64_kernel, dim3((unsigned)((a.nq + kSeedQpb - 1) / kSeedQpb)), dim3(256), 0, s, a,
                       nsamp);
    return hipGetLastError();
}

hipError_t launch_gram_f64(const GramArgs64& a, int arm, hipStream_t s) {
    if (arm != ARM_EUCLID_MULADD) return hipErrorInvalidValue;
    const bool vec2 = rows_vec2(a);
    // k-steps per lane group, even (one 16-byte LDS read feeds two)
    const int64_t ns = ((a.d + 3) / 4 + 1) / 2 * 2;
    if (ns <= 8) return launch_ns<8>(a, vec2, s);
    if (ns <= 16) return launch_ns<16>(a, vec2, s);
    if (ns <= 32) return launch_ns<32>(a, vec2, s);
    if (ns <= 48) return launch_ns<48>(a, vec2, s);
    return launch_ns<64>(a, vec2, s);
}

hipError_t launch_gram_f64_merge(const GramArgs64& a, hipStream_t s) {
    hipLaunchKernelGGL(knn_merge_f64_kernel, dim3((unsigned)((a.nq + 255) / 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace mlrs
