// Group-minimum search: the k nearest rows of every query for the Euclidean
// and cosine arms (d <= 256, k <= 128), f32 and f64, in two passes.
//
//  scan    (knn_groupmin_scan.hpp) every (query, row) pair gets a screen value
//          on the f16 matrix cores from operands of two halves, and only the
//          minimum over each group of 16 index rows is written: 4 bytes for 16
//          pairs.
//  select  (knn_groupmin.hip) per query: T, the k-th smallest group minimum,
//          bounds the k-th screen value (k groups hold k distinct rows at or
//          below it), so with the screen's error bounded (gm_bound) every row
//          of the answer lies in a group whose minimum is not far above T.
//          The rows of those groups (about k of them) are evaluated exactly, in
//          the reference arm's operation order, and ranked by (value, index).
//  precise (knn_groupmin_precise.hip) f64 values only: the queries whose
//          candidates the screen leaves too many, scanned again in f64 and
//          selected for by those minima.  Usually there are none.
//
// The screen is the same whatever the element type: it only decides which pairs
// are evaluated, never a result.  It works on a copy of the index, made per
// search: f32 rows around a centre (Euclidean; a common shift leaves distances
// alone, and the screen's error grows with the norms) or unit rows (cosine),
// each scaled by a power of two and split into two f16 halves per element, 22
// bits.  eps carries the rounding.
//
// ms per call of the searches this one replaced (per-row admission into
// per-segment lists behind f32 or f64 MFMA tiles; exact tiles and a selection
// for small searches), of this one with an f32 MFMA scan at 93% of that peak, and
// now: 1M x 10k, d = 128, k = 32, f32: 20.8, 19.0, 8.1 (scan 6.3, selection 1.3);
// 200k x 5k, d = 256, k = 16, f64 cosine: 9.41, 4.17, 1.84; 60k-row f32 graph, d =
// 50, k = 15: 14.1, 3.69, 2.13; 50k x 5k, d = 50, k = 15, f32: 1.33, 0.32, 0.19; 10k
// x 1k, d = 64, k = 10, f32: 0.090, 0.056, 0.049.
// What it is bad at: points whose neighbours the screen cannot tell apart
// (clusters a fiftieth of their spacing wide and less).  f32 searches, and f64
// ones too small for the precise scan, evaluate every row of a query's cluster:
// 20k x 2k, d = 64, k = 10 in five clusters take 0.57 and 0.79 ms, where exact tiles
// and a selection took 0.22 and 0.42; 100k x 10k, k = 15, f32 15.7 (13.8 with
// per-row admission).
//
// Rows whose screen value cannot be trusted (norms near the ends of the f32
// range, NaN under the fold arm) are "forced": their screen value is +inf and
// a short list hands them to every query.  More rows than it holds are found by
// a mark in the rows' scales.  Queries of that kind evaluate all rows.
#pragma once

#include "knn_kernels.hpp"

namespace mlrs {

constexpr int kGmRows = 32;        // index rows per MFMA tile
constexpr int kGmQuad = 4;         // tiles between stores of the minima
constexpr int kGmQpb = 128;        // queries of one block: 4 waves of 32; a workgroup takes one block or two
constexpr int kGmMaxD = 256;
constexpr int kGmMaxK = 128;
constexpr int kGmForced = 256;     // forced rows listed; more are found by their mark

// Written by the preparation launches.
struct GmStats {
    unsigned int xmax_bits;  // largest trusted ||x||^2 (f32 bits, non-negative)
    unsigned int nforced;    // forced rows (kGmForced of them are listed)
    unsigned int nflag;      // queries the selection leaves to the precise scan
};

struct GmScanArgs {
    // Operand rows hold, per 16 columns, the high halves of the first and the
    // last eight, then the low halves: 64 bytes, counted as 16 floats.
    const float* q;     // [queries, rounded up to the launch's 128 or 256][DP] query operand:
                        // -q or -q / ||q||, scaled and split; zeros past nq
    const float* x;     // index rows, scaled and split, row stride ldx (a multiple of 16)
    const float* bias;  // [tiles * 32] Euclidean ||x||^2 less its share of the error, cosine 0; +inf for rows left out
    const float* xinv;  // [tiles * 32] what undoes the row's scale
    const float* qinv;  // [nq] the same for the queries, times 2 (Euclidean)
    int64_t ldx, d;     // d: columns read per row (<= DP, a multiple of 16)
    int64_t nq, nt;     // queries and index rows of this launch
    int64_t tiles;      // ceil(nt / 32), rounded up to kGmQuad
    int64_t ntp;        // the same: stride of gmin
    float* gmin;        // [nq][2][ntp]: minima of group (tile, half)
    int64_t grid_wgs;   // launch: the CU count; kernel: workgroups of one resident round
};

// Padded row width of the query operand: the 8-column steps the scan is
// compiled for (every multiple of 16 columns up to 128, of 32 up to 256).
inline int gm_chunks(int64_t d) {
    const int c = (int)((d + 7) / 8);
    return c <= 16 ? (c + 1) / 2 * 2 : (c + 3) / 4 * 4;
}
// Two query blocks per workgroup read every LDS tile for twice the products
// (one block keeps the LDS at about 80% of its rate), but leave half the
// workgroups.  One block / two, us per f32 search of k = 10 at d = 32, 64, 128:
// 2^25.6 pairs: 71.9 / 70.8, 87.8 / 87.4, 127.6 / 128.3; 10k x 10k (2^26.6):
// 103.1 / 104.4, 135.0 / 133.0, 206.5 / 210.6; 50k x 5k (2^27.9): 142.5 / 133.6,
// 187.8 / 179.8, 287.3 / 281.5; 200k x 5k (2^29.9): 463 / 398, 588 / 527, 883 / 842:
// the line stands where they are equal.  Past 128 columns two blocks' operands do
// not fit the registers.
inline bool gm_two_blocks(int nk, int64_t nq, int64_t nt) {
    return nk <= 16 && nq > kGmQpb && (double)nq * (double)nt >= 0x1p26;
}
inline int64_t gm_tiles(int64_t nt) { return ((nt + kGmRows - 1) / kGmRows + kGmQuad - 1) / kGmQuad * kGmQuad; }
// Index rows of group (tile, half): row 8 (j / 4) + 4 half + j % 4 of the tile, j < 16.
__host__ __device__ inline int gm_group_row(int half, int j) { return 8 * (j >> 2) + 4 * half + (j & 3); }

// Rows of one kind, as given (T) to the scan's operands.
struct GmPrepArgs {
    const void* rows;    // [n][d] of T
    int64_t n, d;
    const void* centre;  // Euclidean copies: the index, whose first, middle and last rows give the centre
    int64_t centre_n;
    float* out;          // the split copy, row stride ldo (a multiple of 16; zeros past d)
    int64_t ldo;
    int64_t n_out;       // rows of out (zeros past n)
    float* norm;         // index: bias; queries: ||q||^2 (0 for cosine), NaN where the screen is not trusted
    float* inv;          // undoes the rows' scales (queries, Euclidean: times 2); -1: a forced row (its operand is zero)
    int64_t n_norm;      // entries of norm and inv (index: ntp * 32, +inf past n; queries: n)
    int queries;         // 1: query operand; 0: index rows
    int cosine;
    float eps_rel;       // index: the share of ||x||^2 the bias is lowered by
    GmStats* stats;      // filled from the index rows
    int reset;           // zero the index's stats (the launch before the index's; the queries' always zeroes nflag)
    uint32_t* forced;    // [kGmForced]
};
template <typename T>
hipError_t launch_gm_prep(const GmPrepArgs& a, hipStream_t s);

hipError_t launch_gm_scan(const GmScanArgs& a, hipStream_t s);

// The precise scan (knn_groupmin_precise.hip): the same minima on the f64
// matrix cores, of the rows as given, for the queries whose candidates were too
// many to evaluate.  How many those are is known on the device only, so the launch
// is made whenever the search is large enough for it not to show.
template <typename TS>
struct GmPreciseArgs {
    const TS* q;           // [..][d] queries as given
    const TS* x;           // [nt][d] index rows of this part, as given
    int64_t nt, d;
    const TS* centre;      // the index, as the preparation takes its centre
    int64_t centre_n;
    const float* bias;     // +inf for rows left out
    const uint32_t* list;  // [stats->nflag] queries
    const GmStats* stats;
    int64_t tiles, ntp;    // as GmScanArgs
    float* gmin;           // [stats->nflag][2][ntp]: distances (Euclidean: squared), rounded down
    int64_t grid_wgs;      // the CU count
};
template <typename TS>
hipError_t launch_gm_precise(const GmPreciseArgs<TS>& a, bool cosine, hipStream_t s);

// What the minima are.
enum GmKind {
    GM_SCREEN,   // launch_gm_scan's
    GM_PRECISE,  // launch_gm_precise's
    GM_EXACT,    // the arm's own values (launch_groupmin_tile): no statistics, no row left out
};

template <typename TS>
struct GmSelectArgs {
    const TS* q;         // [nq][d] queries as given
    const TS* x;         // [nt][d] index rows of this part, as given
    int64_t nq, nt, d;
    int64_t row0;        // the part's first row in the index
    int first, last;     // the index's first / last part: between them the lists wait in the outputs, untransformed
    int k, mode, kind;
    const float* gmin;   // [nq][2][ntp], GM_PRECISE: rows as list
    int64_t ntp;
    const uint32_t* list;  // GM_PRECISE: the stats->nflag queries to select for (null: all)
    uint32_t* flag;        // where to list queries for the precise scan, or null
    uint32_t flag_above;   // at once with more candidate groups than this
    const float* bias;
    const float* xinv;   // below 0: a forced row
    const float* xcopy;  // the part's operand rows, stride ldx
    const float* qop;    // the queries', stride dp
    const float* qinv;
    int64_t ldx, dp;
    const float* qnorm;  // [nq], NaN: evaluate every row
    GmStats* stats;        // GM_EXACT: null
    const uint32_t* forced;
    // |minimum's value - exact| <= eps_rel (||q||^2 + ||x||^2) + eps_abs + eps_t |value|
    double eps_rel, eps_abs, eps_t;
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
