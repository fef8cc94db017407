// The scan of the group-minimum search (knn_groupmin.hpp): screen values on
// the f32 matrix cores, one minimum per (query, 16 index rows).  Included once
// per arm family so that they compile side by side.
//
// Bound by the f32 MFMA rate.  A workgroup is 4 waves of 32 queries; each wave
// holds its queries in VGPRs as the B operand (d / 2 registers), and the index
// is walked in 32-row tiles through two LDS buffers with one barrier per tile.
// A lane ends a tile with 16 values of one query (its half of the tile's rows)
// and keeps their minimum: eight v_min3 for up to 128 MFMAs, where a screen
// with per-row admission issued about 110 vector instructions.  Four tiles'
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
// (global_load_lds_dwordx4; the rows are 16-byte aligned, gm_prep makes them so
// where the caller's are not).  The rows lie back to back there, and chunk c
// of row r is kept at chunk c ^ gm_swizzle(r), so that the 16-byte A-operand
// reads of eight rows fall on distinct banks.
//
// Rows are 2 NK chunks apart: with NK a multiple of 4 all rows share a bank
// group and three bits of the row number spread them, else two bits or one.
template <int NK>
__device__ __forceinline__ int gm_swizzle(int r) {
    return NK % 4 == 0 ? (r & 7) : NK % 2 == 0 ? ((r >> 1) & 3) : ((r >> 2) & 1);
}

// Waves per SIMD (workgroups per CU) the kernel is compiled for: the query
// operand is 4 NK registers beside 16 accumulators and about 48 others.
constexpr int gm_waves(int nk) { return nk <= 4 ? 6 : nk <= 8 ? 5 : nk <= 16 ? 4 : nk <= 24 ? 3 : 2; }

typedef float gm_f32x16 __attribute__((ext_vector_type(16)));

template <int NK, bool COS>
__global__ __launch_bounds__(256, gm_waves(NK)) void knn_groupmin_kernel(GmScanArgs a) {
    constexpr int DP = NK * 8;
    constexpr int CPR = DP / 4;           // 16-byte chunks per tile row
    constexpr int PF = (NK + 3) / 4;      // loads per wave: NK a tile, 64 chunks each
    __shared__ __attribute__((aligned(16))) float tileA[kGmRows * DP];
    __shared__ __attribute__((aligned(16))) float tileB[kGmRows * DP];
    __shared__ __attribute__((aligned(16))) float tnA[kGmRows];
    __shared__ __attribute__((aligned(16))) float tnB[kGmRows];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, jl = lane & 31;
    const float* __restrict__ X = a.x;
    const float* __restrict__ BIAS = a.bias;
    const int d = (int)a.d;
    const uint32_t row_bytes = 4u * (uint32_t)a.ldx;
    // rows past the index: their bias leaves them out, so their loads only
    // have to stay inside it -- the tile base stops at the last tile and each
    // offset at the last chunk of the last row
    const int last_tile = (int)((a.nt + kGmRows - 1) / kGmRows) - 1;
    const uint32_t last_bytes = (uint32_t)(a.nt - (int64_t)last_tile * kGmRows) * row_bytes;

    // The lane's chunks of a tile, as byte offsets.  Chunks past d repeat the
    // row's first one: the operand is zero there, and a NaN or infinity in it
    // is in the row anyway.
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
        if (tid < kGmRows)
            pfn = *(const __attribute__((address_space(1))) float*)(reinterpret_cast<const char*>(BIAS + (int64_t)t * kGmRows) +
                                                                   4u * (uint32_t)tid);
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
        if (tid < kGmRows) tn[tid] = pfn;
        __syncthreads();
    };

    // Chunk 2 g + h of row jl, kept at (2 g + h) ^ swizzle: only the low three
    // bits move, so four lane offsets serve every g.
    int aoff[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) aoff[j] = jl * DP + 4 * (((2 * j) | h) ^ gm_swizzle<NK>(jl));
    auto a_chunk = [&](const float* buf, int g) -> float4 {
        return *reinterpret_cast<const float4*>(buf + aoff[g & 3] + 32 * (g >> 2));
    };

    const StreamSplit sp(a.nq, a.tiles * kGmRows, kGmQpb, kGmRows * kGmQuad, a.grid_wgs);
    const int64_t wg = xcd_grouped_wg(blockIdx.x, gridDim.x);
    const int64_t u_hi = ((wg + 1) * sp.P < sp.T) ? (wg + 1) * sp.P : sp.T;
    for (int64_t u = wg * sp.P; u < u_hi;) {
        int64_t panel, qblock, quad0, left;
        sp.decode(u, panel, qblock, quad0, left);
        const int64_t quads = left < u_hi - u ? left : u_hi - u;
        u += quads;
        const int t0 = (int)quad0 * kGmQuad, t_end = (int)(quad0 + quads) * kGmQuad;
        load_tile(tileA, t0);
        const int64_t q = qblock * kGmQpb + w * 32 + jl;
        float4 qreg[NK];
        {
            const float* qp = a.q + q * DP + 4 * h;
#pragma unroll
            for (int g = 0; g < NK; ++g) qreg[g] = gload4(qp + 8 * g);
        }
        float* __restrict__ out = a.gmin + (q * 2 + h) * a.ntp;
        const bool qvalid = q < a.nq;
        for (int t = t0; t < t_end; t += kGmQuad) {
            float m[kGmQuad];
#pragma unroll
            for (int i = 0; i < kGmQuad; ++i) {
                float* cur = (i & 1) ? tileB : tileA;
                float* tn = (i & 1) ? tnB : tnA;
                publish(tn);
                if (i + 1 < kGmQuad || t + kGmQuad < t_end) load_tile((i & 1) ? tileA : tileB, t + i + 1);
                gm_f32x16 acc;
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    const float4 n4 = *reinterpret_cast<const float4*>(tn + 8 * g4 + 4 * h);
                    acc[4 * g4 + 0] = COS ? 0.0f : n4.x;
                    acc[4 * g4 + 1] = COS ? 0.0f : n4.y;
                    acc[4 * g4 + 2] = COS ? 0.0f : n4.z;
                    acc[4 * g4 + 3] = COS ? 0.0f : n4.w;
                }
                float4 av = a_chunk(cur, 0);
#pragma unroll
                for (int g = 0; g < NK; ++g) {
                    float4 an = av;
                    if (g + 1 < NK) an = a_chunk(cur, g + 1);
                    __builtin_amdgcn_sched_barrier(0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.x, qreg[g].x, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.y, qreg[g].y, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.z, qreg[g].z, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.w, qreg[g].w, acc, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    av = an;
                }
                if (COS) {
#pragma unroll
                    for (int g4 = 0; g4 < 4; ++g4) {
                        const float4 s4 = *reinterpret_cast<const float4*>(tn + 8 * g4 + 4 * h);
                        acc[4 * g4 + 0] *= s4.x;
                        acc[4 * g4 + 1] *= s4.y;
                        acc[4 * g4 + 2] *= s4.z;
                        acc[4 * g4 + 3] *= s4.w;
                    }
                }
                // NaN (rows left out) is ignored by the minimum
                float v = __builtin_huge_valf();
#pragma unroll
                for (int r = 0; r < 16; ++r) v = fminf(v, acc[r]);
                // an empty statement that reads and returns v: without it the
                // compiler sinks the minimum to the store and keeps all four
                // tiles' accumulators (48 registers) until then
                asm volatile("" : "+v"(v));
                m[i] = v;
            }
            if (qvalid) *reinterpret_cast<float4*>(out + t) = make_float4(m[0], m[1], m[2], m[3]);
        }
    }
}

// a.grid_wgs: the CU count; one resident round of workgroups is launched.
template <bool COS>
hipError_t gm_launch(GmScanArgs a, hipStream_t s) {
    const int nk = gm_chunks(a.d);
    a.grid_wgs *= gm_waves(nk);
    const StreamSplit sp(a.nq, a.tiles * kGmRows, kGmQpb, kGmRows * kGmQuad, a.grid_wgs);
    const dim3 grid((unsigned)sp.G);
    switch (nk) {
#define MLRS_GM_CASE(N) \
    case N: hipLaunchKernelGGL((knn_groupmin_kernel<N, COS>), grid, dim3(256), 0, s, a); break;
        MLRS_GM_CASE(1)
        MLRS_GM_CASE(2)
        MLRS_GM_CASE(3)
        MLRS_GM_CASE(4)
        MLRS_GM_CASE(5)
        MLRS_GM_CASE(6)
        MLRS_GM_CASE(7)
        MLRS_GM_CASE(8)
        MLRS_GM_CASE(9)
        MLRS_GM_CASE(10)
        MLRS_GM_CASE(11)
        MLRS_GM_CASE(12)
        MLRS_GM_CASE(13)
        MLRS_GM_CASE(14)
        MLRS_GM_CASE(15)
        MLRS_GM_CASE(16)
        MLRS_GM_CASE(20)
        MLRS_GM_CASE(24)
        MLRS_GM_CASE(28)
        MLRS_GM_CASE(32)
#undef MLRS_GM_CASE
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

}  // namespace mlrs
