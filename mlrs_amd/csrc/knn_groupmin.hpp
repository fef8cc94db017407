// Group-minimum search: the k nearest rows of every query for the Euclidean
// and cosine arms (d <= 256, k <= 128), f32 and f64, in two passes.
//
//  scan    (knn_groupmin_scan.hpp) every (query, row) pair gets a screen value
//          on v_mfma_f32_32x32x2f32, and only the minimum over each group of
//          16 index rows is written: 4 bytes for 16 pairs.
//  select  (knn_groupmin.hip) per query: T, the k-th smallest group minimum,
//          bounds the k-th screen value (k groups hold k distinct rows at or
//          below it), so with |screen - exact| <= eps every row of the answer
//          lies in a group whose minimum is at most T + 2 eps.  The rows of
//          those groups (about k of them) are evaluated exactly, in the
//          reference arm's operation order, and ranked by (value, index).
//
// The screen is f32 whatever the element type: it only decides which pairs are
// evaluated, never a result.  It works on an f32 copy of the index, made per
// search: rows around a centre (Euclidean; a common shift leaves distances
// alone, and the screen's error grows with the norms) or unit rows (cosine),
// 16-byte aligned.  eps carries the rounding.
//
// Against the searches this one replaced (per-row admission into per-segment
// lists behind f32 or f64 MFMA tiles; exact tiles and a selection for small
// searches), ms per call: 1M x 10k, d = 128, k = 32, f32: 20.8 -> 19.1 (the
// scan 17.5, 93% of the f32 MFMA peak); 200k x 5k, d = 256, k = 16, f64 cosine:
// 9.40 -> 4.18; 60k-row f32 graph, d = 50, k = 15: 14.2 -> 3.76; 50k x 5k, d =
// 50, k = 15, f32: 1.33 -> 0.32; 10k x 1k, d = 64, k = 10, f32: 0.090 -> 0.056.
// What it is bad at: points whose neighbours the screen cannot tell apart
// (clusters a hundredth of their spacing wide and less, where every row of a
// query's cluster is evaluated): 200k x 5k, d = 128 in 100 such clusters take
// 10.7 ms in f32 and 20 in f64.
//
// Rows whose screen value cannot be trusted (norms near the ends of the f32
// range, NaN under the fold arm) are "forced": their screen value is +inf and
// a short list hands them to every query.  Queries of that kind, and every
// query when the list overflows, evaluate all rows.
#pragma once

#include "knn_kernels.hpp"

namespace mlrs {

constexpr int kGmRows = 32;        // index rows per MFMA tile
constexpr int kGmQuad = 4;         // tiles between stores of the minima
constexpr int kGmQpb = 128;        // queries per workgroup: 4 waves of 32
constexpr int kGmMaxD = 256;
constexpr int kGmMaxK = 128;
constexpr int kGmForced = 256;     // forced rows listed before every query evaluates all rows

// Written by the preparation launches.
struct GmStats {
    unsigned int xmax_bits;  // largest trusted ||x||^2 (f32 bits, non-negative)
    unsigned int nforced;    // rows not trusted (kGmForced of them are listed)
};

struct GmScanArgs {
    const float* q;     // [nqb * 128][DP] query operand: -2 q (Euclidean) or -q / ||q||; zeros past nq
    const float* x;     // index rows, 16-byte aligned, row stride ldx (a multiple of 4)
    const float* bias;  // [tiles * 32] Euclidean ||x||^2, cosine in place 1 / ||x||, unit rows 0;
                        // +inf (cosine in place: NaN) for rows left out
    int64_t ldx, d;     // d: columns read per row (<= DP, a multiple of 4)
    int64_t nq, nt;     // queries and index rows of this launch
    int64_t tiles;      // ceil(nt / 32), rounded up to kGmQuad
    int64_t ntp;        // tiles of the whole index: stride of gmin
    float* gmin;        // [nq][2][ntp]: minima of group (tile, half), from this launch's first tile
    int64_t grid_wgs;   // launch: the CU count; kernel: workgroups of one resident round
};

// Padded row width of the query operand: the 8-column steps the scan is
// compiled for (every multiple of 8 up to 128, of 32 up to 256).
inline int gm_chunks(int64_t d) {
    const int c = (int)((d + 7) / 8);
    return c <= 16 ? c : (c + 3) / 4 * 4;
}
inline int64_t gm_tiles(int64_t nt) { return ((nt + kGmRows - 1) / kGmRows + kGmQuad - 1) / kGmQuad * kGmQuad; }
// Index rows of group (tile, half): row 8 (j / 4) + 4 half + j % 4 of the tile, j < 16.
__host__ __device__ inline int gm_group_row(int half, int j) { return 8 * (j >> 2) + 4 * half + (j & 3); }

// Rows of one kind, as given (T) to the scan's f32 operands.
struct GmPrepArgs {
    const void* rows;    // [n][d] of T
    int64_t n, d;
    const void* centre;  // Euclidean copies: the index, whose first, middle and last rows give the centre
    int64_t centre_n;
    int64_t row0;        // index: number of the first row here (the forced list holds row numbers)
    float* out;          // the f32 copy, row stride ldo (zeros past d), or null
    int64_t ldo;
    int64_t n_out;       // rows of out (zeros past n)
    float* norm;         // index: bias; queries: ||q||^2 (0 for cosine), NaN where the screen is not trusted
    int64_t n_norm;      // entries of norm (index: ntp * 32, +inf / NaN past n; queries: n)
    float scale;         // queries: -2 (Euclidean) or -1 (cosine); index: 1
    int queries;         // 1: query operand; 0: index rows
    int cosine;
    int unit;            // cosine: out holds unit rows and bias is 0; else bias is 1 / ||x|| (rows in place)
    GmStats* stats;      // filled from the index rows
    int reset;           // zero stats (the launch before the index's)
    uint32_t* forced;    // [kGmForced]
};
template <typename T>
hipError_t launch_gm_prep(const GmPrepArgs& a, hipStream_t s);

hipError_t launch_gm_scan_euclid(const GmScanArgs& a, hipStream_t s);
hipError_t launch_gm_scan_cosine(const GmScanArgs& a, hipStream_t s);

template <typename TS>
struct GmSelectArgs {
    const TS* q;         // [nq][d] queries as given
    const TS* x;         // [nt][d] index rows as given
    int64_t nq, nt, d;
    int k, mode;
    const float* gmin;   // [nq][2][ntp]
    int64_t ntp;
    const float* bias;
    const float* qnorm;  // [nq], NaN: evaluate every row
    const GmStats* stats;  // null: the minima are of the arm's own values (launch_groupmin_tile), no row is left out
    const uint32_t* forced;
    double eps_rel, eps_abs;  // eps = eps_rel (||q||^2 + max ||x||^2) + eps_abs
    double eps_t;        // relative error of a minimum (values rounded to f32)
    int bias_nan;        // rows left out carry NaN (cosine in place) instead of +inf
    double pexp, root_exp;  // Minkowski: the exponent and (EMIT_ROOT_RANKED) its root's
    int pint;               // its integer exponent
    void* out_val;       // [nq][k] of T
    uint32_t* out_idx;
};
// T: the arithmetic of the arm; TS: the rows' element type (float rows are
// widened for T = double).
template <typename T, typename TS>
hipError_t launch_gm_select(const GmSelectArgs<TS>& a, int arm, hipStream_t s);

// The Manhattan, Chebyshev and Minkowski arms (knn_groupmin_metric.hip); T = TS.
template <typename T>
hipError_t launch_gm_select_metric(const GmSelectArgs<T>& a, int arm, hipStream_t s);

}  // namespace mlrs
