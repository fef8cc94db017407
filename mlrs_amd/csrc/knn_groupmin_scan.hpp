// The scan of the group-minimum search (knn_groupmin.hpp): screen values on
// the f16 matrix cores, one minimum per (query, 16 index rows).
//
// A screen value is the f32 norm plus a contraction whose operands are split
// into two f16 halves each (gm_prep): x q = xh qh + xh ql + xl qh, three
// v_mfma_f32_32x32x16_f16 per 16 columns where eight v_mfma_f32_32x32x2f32 of
// twice the cycles stood, 96 cycles for 512.  Every row is scaled by its own
// power of two before the split, so that the halves lie within f16's range and
// hold 22 bits of every element that counts; the products accumulate in f32,
// about half as many roundings as the f32 chain made.  A workgroup is 4 waves of 32 queries; each wave
// holds its queries in VGPRs as the B operand (d / 2 registers: two halves of 16 bits per column), and the index
// is walked in 32-row tiles through two LDS buffers with one barrier per tile.
// A lane ends a tile with 16 values of one query (its half of the tile's rows),
// unscales them (a multiplication and a multiply-add each, 32 instructions per
// query block) and keeps their minimum (eight v_min3), beside 3 / 16 MFMAs a
// column and query block, 48 at most.  Four tiles'
// minima make one 16-byte store.  No state outlives a tile, so the (query
// block, four tiles) units are cut into equal ranges, one per resident
// workgroup, panel by panel (StreamSplit) so that workgroups of an XCD stream
// the same rows together.
#pragma once

#include "knn_common.hpp"
#include "knn_groupmin.hpp"

namespace mlrs {

namespace {

// A tile reaches LDS one tile ahead of its use, straight from global memory
// (global_load_lds_dwordx4).  The rows lie back to back there, and chunk c
// of row r is kept at chunk c ^ gm_swizzle(r), so that the 16-byte A-operand
// reads of eight rows fall on distinct banks.
//
// Rows are 2 NK chunks apart (NK is even): with NK a multiple of 4 all rows
// share a bank group and three bits of the row number spread them, else two.
template <int NK>
__device__ __forceinline__ int gm_swizzle(int r) {
    return NK % 4 == 0 ? (r & 7) : ((r >> 1) & 3);
}

// Waves per SIMD (workgroups per CU) the kernel is compiled for: a wave's 32 QB
// queries take 4 NK QB registers beside 16 QB accumulators and about 60 others.
constexpr int gm_waves(int nk, int qb) {
    return 4 * nk * qb + 16 * qb + 60 <= 96    ? 5
           : 4 * nk * qb + 16 * qb + 60 <= 128 ? 4
           : 4 * nk * qb + 16 * qb + 60 <= 168 ? 3
                                               : 2;
}

typedef float gm_f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 gm_f16x8 __attribute__((ext_vector_type(8)));

template <int NK, int QB>
__global__ __launch_bounds__(256, gm_waves(NK, QB)) void knn_groupmin_kernel(GmScanArgs a) {
    constexpr int DP = NK * 8;
    constexpr int CPR = DP / 4;           // 16-byte chunks per tile row
    constexpr int PF = (NK + 3) / 4;      // loads per wave: NK a tile, 64 chunks each
    __shared__ __attribute__((aligned(16))) float tileA[kGmRows * DP];
    __shared__ __attribute__((aligned(16))) float tileB[kGmRows * DP];
    __shared__ __attribute__((aligned(16))) float tnA[2 * kGmRows];  // the rows' norms, then their scales
    __shared__ __attribute__((aligned(16))) float tnB[2 * kGmRows];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, jl = lane & 31;
    const float* __restrict__ X = a.x;
    const float* __restrict__ NORM = tid < kGmRows ? a.bias : a.xinv;
    const int d = (int)a.d;
    const uint32_t row_bytes = 4u * (uint32_t)a.ldx;
    // rows past the index: their bias leaves them out, so their loads only
    // have to stay inside it -- the tile base stops at the last tile and each
    // offset at the last chunk of the last row
    const int last_tile = (int)((a.nt + kGmRows - 1) / kGmRows) - 1;
    const uint32_t last_bytes = (uint32_t)(a.nt - (int64_t)last_tile * kGmRows) * row_bytes;

    // The lane's chunks of a tile, as byte offsets.  Chunks past d repeat the
    // row's first one: the query operand is zero there and the copy is finite.
    float pfn = 0.0f;
    uint32_t src[PF];
#pragma unroll
    for (int p = 0; p < PF; ++p) {
        const int f = (w * PF + p) * 64 + lane;
        const int r = f / CPR;
        int c = (f % CPR) ^ gm_swizzle<NK>(r);
        if (4 * c >= d) c = 0;
        src[p] = (uint32_t)r * row_bytes + 16u * (uint32_t)c;
    }
    auto load_tile = [&](float* buf, int t) {
        if (tid < 2 * kGmRows)
            pfn = *(const __attribute__((address_space(1))) float*)(NORM + ((int64_t)t * kGmRows + (tid & (kGmRows - 1))));
        const int tc = t < last_tile ? t : last_tile;
        const char* base = reinterpret_cast<const char*>(X) + (int64_t)tc * kGmRows * row_bytes;
        const uint32_t lim = (tc < last_tile ? kGmRows * row_bytes : last_bytes) - 16u;
#pragma unroll
        for (int p = 0; p < PF; ++p) {
            if (NK % 4 != 0 && w * PF + p >= NK) break;  // uniform
            const uint32_t o = src[p] < lim ? src[p] : lim;
            global_to_lds16(base + o, buf + (w * PF + p) * 256);
        }
    };
    auto publish = [&](float* tn) {
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the tile's loads have landed
        if (tid < 2 * kGmRows) tn[tid] = pfn;
        __syncthreads();
    };

    // Chunk 2 g + h of row jl, kept at (2 g + h) ^ swizzle: only the low three
    // bits move, so four lane offsets serve every g.
    int aoff[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) aoff[j] = jl * DP + 4 * (((2 * j) | h) ^ gm_swizzle<NK>(jl));
    auto a_chunk = [&](const float* buf, int g) -> gm_f16x8 {
        return *reinterpret_cast<const gm_f16x8*>(buf + aoff[g & 3] + 32 * (g >> 2));
    };

    const StreamSplit sp(a.nq, a.tiles * kGmRows, kGmQpb * QB, kGmRows * kGmQuad, a.grid_wgs);
    const int64_t wg = xcd_grouped_wg(blockIdx.x, gridDim.x);
    const int64_t u_hi = ((wg + 1) * sp.P < sp.T) ? (wg + 1) * sp.P : sp.T;
    for (int64_t u = wg * sp.P; u < u_hi;) {
        int64_t panel, qblock, quad0, left;
        sp.decode(u, panel, qblock, quad0, left);
        const int64_t quads = left < u_hi - u ? left : u_hi - u;
        u += quads;
        const int t0 = (int)quad0 * kGmQuad, t_end = (int)(quad0 + quads) * kGmQuad;
        load_tile(tileA, t0);
        // the wave's query blocks lie 128 queries apart
        const int64_t q = qblock * (kGmQpb * QB) + w * 32 + jl;
        gm_f16x8 qreg[QB][NK];  // of 16-column step g: high halves at 2 g, low halves at 2 g + 1
        float qi[QB];
#pragma unroll
        for (int b = 0; b < QB; ++b) {
            const float* qp = a.q + (q + b * kGmQpb) * DP + 4 * h;
#pragma unroll
            for (int g = 0; g < NK; ++g) qreg[b][g] = __builtin_bit_cast(gm_f16x8, gload4(qp + 8 * g));
            qi[b] = a.qinv[q + b * kGmQpb < a.nq ? q + b * kGmQpb : 0];
        }
        float* __restrict__ out = a.gmin + (q * 2 + h) * a.ntp;
        for (int t = t0; t < t_end; t += kGmQuad) {
            float m[QB][kGmQuad];
#pragma unroll
            for (int i = 0; i < kGmQuad; ++i) {
                float* cur = (i & 1) ? tileB : tileA;
                float* tn = (i & 1) ? tnB : tnA;
                publish(tn);
                if (i + 1 < kGmQuad || t + kGmQuad < t_end) load_tile((i & 1) ? tileA : tileB, t + i + 1);
                gm_f32x16 acc[QB] = {};
                gm_f16x8 hi = a_chunk(cur, 0), lo = a_chunk(cur, 1);
#pragma unroll
                for (int g = 0; g < NK; g += 2) {
                    gm_f16x8 hn = hi, ln = lo;
                    if (g + 2 < NK) {
                        hn = a_chunk(cur, g + 2);
                        ln = a_chunk(cur, g + 3);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int b = 0; b < QB; ++b)
                        acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, qreg[b][g], acc[b], 0, 0, 0);
#pragma unroll
                    for (int b = 0; b < QB; ++b)
                        acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, qreg[b][g + 1], acc[b], 0, 0, 0);
#pragma unroll
                    for (int b = 0; b < QB; ++b)
                        acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, qreg[b][g], acc[b], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    hi = hn;
                    lo = ln;
                }
                // rows left out have norm +inf; no value is NaN
                float v[QB];
#pragma unroll
                for (int b = 0; b < QB; ++b) v[b] = __builtin_huge_valf();
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    const float4 n4 = *reinterpret_cast<const float4*>(tn + 8 * g4 + 4 * h);
                    const float4 s4 = *reinterpret_cast<const float4*>(tn + kGmRows + 8 * g4 + 4 * h);
#pragma unroll
                    for (int b = 0; b < QB; ++b) {
                        v[b] = fminf(v[b], __builtin_fmaf(acc[b][4 * g4 + 0] * s4.x, qi[b], n4.x));
                        v[b] = fminf(v[b], __builtin_fmaf(acc[b][4 * g4 + 1] * s4.y, qi[b], n4.y));
                        v[b] = fminf(v[b], __builtin_fmaf(acc[b][4 * g4 + 2] * s4.z, qi[b], n4.z));
                        v[b] = fminf(v[b], __builtin_fmaf(acc[b][4 * g4 + 3] * s4.w, qi[b], n4.w));
                    }
                }
#pragma unroll
                for (int b = 0; b < QB; ++b) {
                    // an empty statement that reads and returns v: without it the
                    // compiler sinks the minimum to the store and keeps all four
                    // tiles' accumulators until then
                    asm volatile("" : "+v"(v[b]));
                    m[b][i] = v[b];
                }
            }
#pragma unroll
            for (int b = 0; b < QB; ++b)
                if (q + b * kGmQpb < a.nq)
                    *reinterpret_cast<float4*>(out + b * (2 * kGmQpb) * a.ntp + t) =
                        make_float4(m[b][0], m[b][1], m[b][2], m[b][3]);
        }
    }
}

template <int NK, int QB>
void gm_launch_nk(GmScanArgs a, hipStream_t s) {
    a.grid_wgs *= gm_waves(NK, QB);
    const StreamSplit sp(a.nq, a.tiles * kGmRows, kGmQpb * QB, kGmRows * kGmQuad, a.grid_wgs);
    hipLaunchKernelGGL((knn_groupmin_kernel<NK, QB>), dim3((unsigned)sp.G), dim3(256), 0, s, a);
}

// a.grid_wgs: the CU count; one resident round of workgroups is launched.
hipError_t gm_launch(const GmScanArgs& a, hipStream_t s) {
    const int nk = gm_chunks(a.d);
    if (gm_two_blocks(nk, a.nq, a.nt)) {
        switch (nk) {
#define MLRS_GM_CASE(N) \
    case N: gm_launch_nk<N, 2>(a, s); break;
        MLRS_GM_CASE(2)
        MLRS_GM_CASE(4)
        MLRS_GM_CASE(6)
        MLRS_GM_CASE(8)
        MLRS_GM_CASE(10)
        MLRS_GM_CASE(12)
        MLRS_GM_CASE(14)
        MLRS_GM_CASE(16)
#undef MLRS_GM_CASE
        default: return hipErrorInvalidValue;
        }
    } else {
        switch (nk) {
#define MLRS_GM_CASE(N) \
    case N: gm_launch_nk<N, 1>(a, s); break;
        MLRS_GM_CASE(2)
        MLRS_GM_CASE(4)
        MLRS_GM_CASE(6)
        MLRS_GM_CASE(8)
        MLRS_GM_CASE(10)
        MLRS_GM_CASE(12)
        MLRS_GM_CASE(14)
        MLRS_GM_CASE(16)
        MLRS_GM_CASE(20)
        MLRS_GM_CASE(24)
        MLRS_GM_CASE(28)
        MLRS_GM_CASE(32)
#undef MLRS_GM_CASE
        default: return hipErrorInvalidValue;
        }
    }
    return hipGetLastError();
}

}  // namespace

}  // namespace mlrs
