// normal.h -- the level-space form of the LSMR iteration: the normal matrix
// M = A'A of the scaled fixed-effect map (unit diagonal but for rounding) as one
// sparse matrix over the levels, and the launches of an iteration that reads M instead of
// the observations.
#pragma once

#include <vector>

#include "fehip_common.h"

struct fehip_solver;

namespace fehip {

// A tile is what one wave takes at a time: consecutive entries, and the rows
// that begin among them.
constexpr int kNfTile = 512;    // entries + kNfRow per row that a tile aims at
constexpr int kNfSlack = 128;   // a row with at most this many units left at a tile's end is finished in it
constexpr int kNfCap = kNfTile + kNfSlack;
constexpr int kNfRow = 8;       // tile units of one row beside its entries (its vector elements)
constexpr int kNfRows = kNfCap / kNfRow + 2;  // rows one tile owns, at most

// a tile: its number (ascending with its entries), first entry and the row it
// is in (the first that begins there, or after it), entries | rows that begin
// in it << 16
struct NfTileAt {
    int32_t k, e0, r0, len_nr;
};

// a row whose entries lie in several tiles: [t0, t1) hold its later parts,
// tile t0 - 1 its first
struct NfItem {
    int32_t row, t0, t1;
};

// cells (distinct level pairs) of one pair of FEs
struct NfPair {
    int a = 0, b = 0;              // cells sorted by (level of a, level of b)
    int64_t ncell = 0;
    int32_t *order = nullptr;      // internal positions sorted by (a, b); nullptr: the internal order itself
    int32_t *start = nullptr;      // ncell + 1: first position (in that order) of each cell
    int32_t *dsta = nullptr, *dstb = nullptr;  // the cell's entry in row a and in row b
    int32_t *big = nullptr;        // cells of more than kNfBigCell observations
    int32_t nbig = 0;
};
constexpr int kNfBigCell = 32;
constexpr int64_t kNfFarLevels = 1 << 18;  // 2 MB of one column

struct NormalMat {
    int64_t p = 0, nnz = 0;
    int64_t far = 0;  // entries whose column is of an FE of more than kNfFarLevels levels
    int32_t *off = nullptr, *col = nullptr;  // p + 1, nnz
    double *val = nullptr;                   // nnz: sum over the cell of cache_a * cache_b
    std::vector<NfPair> pairs;
    int32_t ntile = 0, ts0 = 0, ts1 = 0;     // [ts0, ts1): the tiles of FE s's rows
    NfTileAt *tiles = nullptr;               // in the order of the launches (FE s's stay in [ts0, ts1))
    NfItem *items = nullptr;
    int32_t nitem = 0, is0 = 0, is1 = 0;     // [is0, is1): the items of FE s's rows
    uint32_t *split = nullptr;               // bit per row: its sum comes from its item
    // entries on the diagonal, one per large level (NfInput::big_rows)
    int32_t ndiag = 0;
    int32_t *dpos = nullptr;                 // their places in col and val
    bool projected = false;                  // val is the projected iteration's
};

// *all_done when every column has stopped: 1 + the state's copy, or this + the
// copy where rounding has reached the betas of some (bad), which start over on
// the observations (see kNfLost).
constexpr int32_t kNfStartOver = 4;

// per-column coefficients of the step, written by the scalar launch
struct NfCols {
    double ia[kMaxK], iold[kMaxK];            // v = ia * w, the one before = iold * wold
    double cq[kMaxK], cv[kMaxK], co[kMaxK];   // w' = cq q + cv w + co wold
    double chb[kMaxK], cx[kMaxK], ch[kMaxK];  // the h / hbar / x update
    double beta1[kMaxK];                      // beta of the iteration before
    double err[kMaxK];                        // error bound of beta^2
    int32_t on[kMaxK], upd[kMaxK];            // the column runs; an update goes with the step
    int32_t due[kMaxK];                       // alpha and the rotations are due
    int32_t test[kMaxK];                      // the stopping rules are due
    // updates in pairs: the second one, the column's last iteration is reached,
    // and x takes the second one back
    double chb2[kMaxK], cx2[kMaxK], ch2[kMaxK];
    int32_t upd2[kMaxK], last[kMaxK], undo[kMaxK];
    int32_t bad[kMaxK];   // the column has to start over (kNfStartOver)
};

struct NfApply {
    const int32_t *off, *col;
    const double *val;
    const NfTileAt *tiles;
    int32_t t0, n0, t1, nt;   // positions t0 .. t0+n0-1, then t1 .. (nt tiles in all)
    const double *w;          // p x K
    double *q;                // p x K: M w
    double *pa;               // partials [block * K + c]: w'q
    double *head, *tail;      // [tile * K + c]
    const int32_t *all_done;
    double *neg;              // projected, FE s rows: neg[row] = -sum (into w), nothing else
};

// The scalar step between a product and the step after it.
struct NfScalars {
    const double *pa, *pw, *px, *px2;
    int32_t na, nw;           // their lengths (px and px2 have pw's)
    const void *sin;          // LsmrState<double>, K
    void *sout;               // the same copy in a launch of its own, the other one when folded
    const NfCols *cin;
    NfCols *cout;
    int32_t copy;             // which copy sout is
    int32_t *all_done;
    void *snap;               // updates in pairs: the state after the rotations of each, 2 x K
    int32_t even;             // updates in pairs: 1 in iterations 2, 4, ..
};
struct NfStep {
    NfScalars fold;           // kNfFolded
    int64_t p;
    int64_t row0, rown;       // rows [row0, row0 + rown) are left alone (the eliminated FE)
    const double *q, *w;
    double *wold;             // in: the vector before w; out: the next one
    double *h, *hbar, *x;
    const NfCols *cols;
    const NfItem *items;
    int32_t nitem;
    const uint32_t *split;
    const double *head, *tail;
    double *pw, *px, *px2;    // partials ||w'||^2, ||x||^2 (after the first and the second update)
    const int32_t *all_done;
    unsigned fix_blocks;
    int mode;
};
// What a step does beside w'.
enum NfMode { kNfFolded, kNfLight, kNfHeavy };

// launches (normal.hip); K in {1, 2, 4, 8, 16, 32}
unsigned nf_apply_blocks(int K, int32_t ntiles);
bool nf_folds(int K, unsigned apply_blocks, unsigned step_blocks);  // the step does the scalar step (kNfFolded)
void nf_apply(int K, const NfApply &a, unsigned blocks, hipStream_t st);
void nf_fix_neg(int K, const NfItem *items, int32_t n, const double *head, const double *tail, double *neg,
                const int32_t *all_done, hipStream_t st);
void nf_scalars(int K, const NfScalars &s, hipStream_t st);
void nf_step(int K, const NfStep &s, unsigned blocks, hipStream_t st);
void nf_init_cols(int K, const void *state, NfCols *cols, hipStream_t st);

// construction (normal.hip), on the handle's stream through its allocator and sort
struct NfInput {
    int64_t N = 0;
    int G = 0, s = 0, t_sec = -1;
    const int64_t *n = nullptr, *off = nullptr;
    const int32_t *ref[kMaxG] = {};
    const double *cache[kMaxG] = {};
    const int32_t *by_level[kMaxG] = {};  // positions sorted (stably) by level, where a handle has them
    // levels of many observations, FE after FE, and the exact sums of z^2 w over
    // them; every level's scale (p)
    int32_t nbig[kMaxG] = {}, big0_s = 0;  // of each FE; FE s's first
    const int32_t *big_rows = nullptr;
    const double *big_sum = nullptr;
    const double *scale = nullptr;
    hipStream_t stream = nullptr;
};
// the form is taken up to nnz_max entries (*fits = 1; else 0) of which far_max
// are far (else -1); m is left empty where it is not
int nf_build(fehip_solver *h, const NfInput &in, int64_t nnz_max, int64_t far_max, NormalMat &m, int *fits);
int nf_values(const NfInput &in, NormalMat &m, bool projected);
void nf_free(fehip_solver *h, NormalMat &m);

}  // namespace fehip
