// normal.hip -- the LSMR iteration in level space.
//
// The iteration of src/utils/lsmr.jl:103-215 needs u only through A'u and
// ||u||.  With v_k and s_k = A'u_k in the span of the levels,
//   A'u_{k+1} beta_{k+1} = M v_k - alpha_k s_k,   M = A'A,
//   alpha_{k+1} beta_{k+1} v_{k+1} = M v_k - (v_k'M v_k) v_k - alpha_k beta_k v_{k-1},
//   beta_{k+1}^2 = v_k'M v_k - alpha_k^2,
// the same bidiagonalization, with the same alpha and beta, and no vector over
// the observations.  M has a unit diagonal but for scale!'s rounding
// (src/SolverCPU.jl:78-89; large levels have an entry for what it leaves, see
// k_nf_diag) and one entry per pair of levels that meet: a worker/firm/year panel of 1e7
// observations (1e6 workers, 1e5 firms, 20 years) has 1.19e7 entries, 142 MB,
// where the pass over the observations reads and writes 470 MB per column.
//
// One iteration is three launches, k counting iterations from 1:
//   k_nf_apply    q = M w, w'q for the raw next vector w (v_k = w / ||w||)
//   k_nf_scalars  stopping rules of iteration k-2 (||x|| came with the last
//                 step), alpha and the plane rotations of k-1 (||w|| did too),
//                 beta of k
//   k_nf_step     x, hbar, h of iteration k-1; the next w; ||x||, ||w||
// A column that stops does so one product and one scalar launch later than it
// might; x is the stopping iteration's.  That is the form with two launches
// (kNfFolded); with three, x, hbar and h of k-2 and k-1 are updated together in
// the steps of odd k, and the rules of both are looked at in k+1.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <vector>

#include "../../include/fehip.h"
#include "fehip_common.h"
#include "linmap.h"
#include "normal.h"

namespace fehip {

// of the solver (fehip.hip)
int set_error(int code, const std::string &msg);
int solver_alloc(fehip_solver *h, void **ptr, size_t bytes);
void solver_free(fehip_solver *h, void *ptr);
int solver_sort(fehip_solver *h, const int32_t *keys, int64_t n, int64_t nlev, int32_t *keys_out, int32_t *vals_out,
                const int32_t *vals_in);
int solver_scan(fehip_solver *h, const uint32_t *in, int64_t n, uint32_t *out);

#define NCHK(expr)                                                                                          \
    do {                                                                                                    \
        hipError_t e_ = (expr);                                                                             \
        if (e_ != hipSuccess) return set_error(FEHIP_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)
#define NRC(expr)                 \
    do {                          \
        int rc_ = (expr);         \
        if (rc_ != 0) return rc_; \
    } while (0)

static inline unsigned blocks_for(int64_t n, int64_t per) {
    return (unsigned)std::max<int64_t>((n + per - 1) / per, 1);
}

// ---------------------------------------------------------------------------
// the product with M
// ---------------------------------------------------------------------------

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) v += __shfl_xor(v, d, kWave);
    return v;
}

// Tiles of a launch over nt: workgroup b's j-th round takes kWavesPerBlock
// neighbouring tiles, one per wave.  Groups of neighbouring rounds go to one
// XCD (workgroup number mod 8), so rows that gather the same levels share its
// L2, and the groups alternate over the XCDs, so none of them gets all the
// tiles of one kind.
struct TileMap {
    int32_t grp, end;  // in rounds
    __device__ __forceinline__ explicit TileMap(int32_t nt) {
        const int32_t nq = (nt + kWavesPerBlock - 1) / kWavesPerBlock;
        grp = nq >= 2048 ? 32 : (nq >= 64 ? nq / 64 : 1);
        end = (nq + 8 * grp - 1) / (8 * grp) * (8 * grp);
    }
    __device__ __forceinline__ int32_t at(int32_t j) const {
        const int32_t x = j & 7, l = j >> 3;
        return ((l / grp) * 8 + x) * grp + l % grp;
    }
};

// one tile of a launch
struct TileDesc {
    int32_t k, e0, r0;
    int len, nr;
};

// the wave's next tile from launch position j on (j is moved to it)
__device__ __forceinline__ bool next_tile(const NfApply &p, const TileMap &tm, int wave, int32_t &j, TileDesc &d) {
    int32_t ti = p.nt;
    for (; j < tm.end; j += gridDim.x) {
        ti = tm.at(j) * kWavesPerBlock + wave;
        if (ti < p.nt) break;
    }
    if (ti >= p.nt) return false;
    const int32_t at = __builtin_amdgcn_readfirstlane(ti < p.n0 ? p.t0 + ti : p.t1 + ti - p.n0);
    const int32_t *q = (const int32_t *)p.tiles;
    d.k = ld_const(q, 4 * at);
    d.e0 = ld_const(q, 4 * at + 1);
    d.r0 = ld_const(q, 4 * at + 2);
    const int32_t ln = ld_const(q, 4 * at + 3);
    d.len = ln & 0xffff;
    d.nr = ln >> 16;
    return true;
}

// two adjacent doubles at a 32-bit element offset from a uniform base (p * K * 8
// < 2^32: one address register instead of two)
__device__ __forceinline__ double2 ld2(const double *base, uint32_t i) {
    return *(const double2 *)((const char *)base + (i << 3));
}
__device__ __forceinline__ void st2(double *base, uint32_t i, double2 v) {
    *(double2 *)((char *)base + (i << 3)) = v;
}

// LDS written by a wave and read by it: its operations complete in order, only
// the compiler has to keep them so
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

constexpr int kSerial1 = 64;  // K = 1: a row of more entries in the tile is summed by the wave
constexpr int kSerialK = 48;  // K > 1: ... by the wave instead of one group of its lanes
constexpr int kNfPer = kNfCap / kWave;  // entries of a tile per lane
static_assert(kNfPer * kWave == kNfCap, "a tile is kNfPer entries per lane");

// sum of prod[s, t) in order, eight LDS reads in flight
__device__ __forceinline__ double serial_sum(const double *prod, int s, int t) {
    double sum = 0.0;
    for (; s + 8 <= t; s += 8) {
        double x[8];
#pragma unroll
        for (int u = 0; u < 8; u++) x[u] = prod[s + u];
#pragma unroll
        for (int u = 0; u < 8; u++) sum += x[u];
    }
    double x[8];
#pragma unroll
    for (int u = 0; u < 8; u++) x[u] = prod[s + u < t ? s + u : s];
#pragma unroll
    for (int u = 0; u < 8; u++) sum += s + u < t ? x[u] : 0.0;
    return sum;
}

// q = M v of one column.  A wave forms the products of its tile's entries in
// its own part of LDS (every load of the tile in flight together, none depends
// on a row's length), and adds each row's run of them: a lane per row, the
// wave per long row.  The next tile's entries are loaded while the rows of
// this one are summed; no wave waits for another.  A row cut by a tile
// boundary leaves its parts in head / tail.
// NEG: the rows of the eliminated FE in the projected iteration, -sum into neg.
template <bool NEG>
__global__ __launch_bounds__(kBlock) void k_nf_apply1(NfApply p) {
    if (*p.all_done) return;
    __shared__ double prods[kWavesPerBlock][kNfCap + 8];
    __shared__ double red[kWavesPerBlock];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    double *prod = prods[wave];
    double acc = 0.0;
    const TileMap tm(p.nt);
    constexpr int H = kNfPer / 2, U = kNfPer;
    int32_t c[U];
    double a[U];
    auto load_entries = [&](const TileDesc &d) {
#pragma unroll
        for (int u = 0; u < H; u++) {
            const int e = u * kWave + lane;
            const int32_t ee = e < d.len ? d.e0 + e : 0;
            c[u] = p.col[ee];
            a[u] = p.val[ee];
        }
        if (d.len > H * kWave) {
#pragma unroll
            for (int u = H; u < U; u++) {
                const int e = u * kWave + lane;
                const int32_t ee = e < d.len ? d.e0 + e : 0;
                c[u] = p.col[ee];
                a[u] = p.val[ee];
            }
        }
    };
    int32_t j = blockIdx.x;
    TileDesc d;
    bool more = next_tile(p, tm, wave, j, d);
    if (more) load_entries(d);
    while (more) {
        const int32_t k = d.k, r0 = d.r0, e0 = d.e0, e1 = d.e0 + d.len;
        const int len = d.len, nr = d.nr;
        // the first rows' starts and vector elements, the entries' elements of v
        double wv = 0.0;
        int s = 0, t = 0;
        const int32_t first = ld_const(p.off, r0);
        const bool cut = nr > 0 && ld_const(p.off, r0 + nr) > e1;  // the last row goes on in the next tile
        if (lane < nr) {
            s = p.off[r0 + lane];
            t = p.off[r0 + lane + 1];
            if (!NEG) wv = p.w[r0 + lane];
        }
        {
            double x[U];
#pragma unroll
            for (int u = 0; u < H; u++) x[u] = p.w[c[u]];
            if (len > H * kWave) {
#pragma unroll
                for (int u = H; u < U; u++) x[u] = p.w[c[u]];
#pragma unroll
                for (int u = H; u < U; u++) prod[u * kWave + lane] = a[u] * x[u];
            }
#pragma unroll
            for (int u = 0; u < H; u++) prod[u * kWave + lane] = a[u] * x[u];
        }
        TileDesc dn;
        j += gridDim.x;
        const bool more_n = next_tile(p, tm, wave, j, dn);
        wave_lds_sync();
        if (more_n) load_entries(dn);
        const int hl = min(first, e1) - e0;
        if (hl > 0) {  // the row that began before this tile
            double h = 0.0;
            for (int i = lane; i < hl; i += kWave) h += prod[i];
            h = wave_sum(h);
            if (lane == 0) {
                p.head[k] = h;
                if (!NEG) acc += p.w[r0 - 1] * h;
            }
        }
        for (int i0 = 0; i0 < nr; i0 += kWave) {
            const int i = i0 + lane;
            const bool own = i < nr;
            const int32_t r = r0 + (own ? i : 0);
            if (i0 && own) {
                s = p.off[r];
                t = p.off[r + 1];
                if (!NEG) wv = p.w[r];
            }
            const int ls = own ? s - e0 : 0, lt = own ? min(t, e1) - e0 : 0;
            const bool big = lt - ls > kSerial1;
            double sum = big ? 0.0 : serial_sum(prod, ls, lt);
            for (uint64_t m = __ballot(big); m; m &= m - 1) {
                const int b = __builtin_ctzll(m);
                const int bs = __builtin_amdgcn_readlane(ls, b), bt = __builtin_amdgcn_readlane(lt, b);
                double q = 0.0;
                for (int e = bs + lane; e < bt; e += kWave) q += prod[e];
                q = wave_sum(q);
                if (lane == b) sum = q;
            }
            if (own) {
                const bool part = cut && i == nr - 1;
                if (part) p.tail[k] = sum;
                if (NEG) {
                    if (!part) p.neg[r] = -sum;
                } else {
                    const double qv = wv + sum;  // (the diagonal's 1; k_nf_diag)
                    acc += wv * qv;
                    if (!part) p.q[r] = qv;
                }
            }
        }
        wave_lds_sync();
        d = dn;
        more = more_n;
    }
    if (NEG) return;
    acc = wave_sum(acc);
    if (lane == 0) red[wave] = acc;
    __syncthreads();
    if (tid == 0) p.pa[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// q = M V of K columns.  A wave takes a tile; a group of K/2 of its lanes holds
// two adjacent columns per lane and takes a row at a time: the entries come
// from the wave's part of LDS (staged coalesced, the next tile's loaded
// meanwhile), each entry's row of V as one 16-byte load per lane, four entries
// in flight.  Longer rows are shared by the groups.
template <int K, bool NEG>
__global__ __launch_bounds__(kBlock) void k_nf_apply(NfApply p) {
    if (*p.all_done) return;
    constexpr int KL = K / 2, GW = kWave / KL, U = 4;
    constexpr int RW = (kNfRows + kWave) / kWave;  // rounds that load a tile's row starts
    __shared__ double lvs[kWavesPerBlock][kNfCap];
    __shared__ int32_t lcs[kWavesPerBlock][kNfCap];
    __shared__ int32_t ros[kWavesPerBlock][RW * kWave];
    __shared__ double red[kWavesPerBlock * K];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int gw = lane / KL, cg = lane % KL, c0 = 2 * cg;
    double *lv = lvs[wave];
    int32_t *lc = lcs[wave], *ro = ros[wave];
    double aq0 = 0.0, aq1 = 0.0;
    const TileMap tm(p.nt);

    struct Sum {
        double s0, s1;
    };
    // entries first, first + step, ... of [s, t)
    auto row_sum = [&](int s, int t, int first, int step) {
        Sum r{0.0, 0.0};
        for (int e = s + first; e < t; e += U * step) {
            double a[U];
            double2 x[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const bool in = e + u * step < t;
                const int ee = in ? e + u * step : e;
                a[u] = in ? lv[ee] : 0.0;
                x[u] = ld2(p.w, (uint32_t)lc[ee] * (uint32_t)K + (uint32_t)c0);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                r.s0 += a[u] * x[u].x;
                r.s1 += a[u] * x[u].y;
            }
        }
        return r;
    };
    auto over_groups = [&](Sum &s) {
#pragma unroll
        for (int q = KL; q < kWave; q <<= 1) {
            s.s0 += __shfl_xor(s.s0, q, kWave);
            s.s1 += __shfl_xor(s.s1, q, kWave);
        }
    };
    // what a row's sum is for; q not written when the row goes on (part)
    auto emit = [&](int32_t k, int32_t r, bool part, const Sum &s, const double2 &w) {
        const uint32_t at = (uint32_t)r * (uint32_t)K + (uint32_t)c0;
        if (part) *(double2 *)(p.tail + (int64_t)k * K + c0) = make_double2(s.s0, s.s1);
        if (NEG) {
            if (!part) st2(p.neg, at, make_double2(-s.s0, -s.s1));
            return;
        }
        const double q0 = w.x + s.s0, q1 = w.y + s.s1;  // (the diagonal's 1; k_nf_diag)
        aq0 += w.x * q0;
        aq1 += w.y * q1;
        if (!part) st2(p.q, at, make_double2(q0, q1));
    };
    // a tile's first entries and its row starts, in registers until the tile
    // before it is done (the rest of a tile of long rows is read when it is due)
    constexpr int PF = 4;
    int32_t ec[PF], er[RW];
    double ea[PF];
    auto load_tile = [&](const TileDesc &d) {
#pragma unroll
        for (int u = 0; u < PF; u++) {
            const int e = u * kWave + lane;
            const int32_t ee = e < d.len ? d.e0 + e : 0;
            ec[u] = p.col[ee];
            ea[u] = p.val[ee];
        }
#pragma unroll
        for (int u = 0; u < RW; u++) {
            const int i = u * kWave + lane;
            er[u] = p.off[d.r0 + (i <= d.nr ? i : 0)];
        }
    };

    int32_t j = blockIdx.x;
    TileDesc d;
    bool more = next_tile(p, tm, wave, j, d);
    if (more) load_tile(d);
    while (more) {
        const int32_t k = d.k, r0 = d.r0, e1 = d.e0 + d.len;
        const int nr = d.nr;
#pragma unroll
        for (int u = 0; u < PF; u++) {
            lc[u * kWave + lane] = ec[u];
            lv[u * kWave + lane] = ea[u];
        }
        if (d.len > PF * kWave) {
            constexpr int R = kNfPer - PF;
            int32_t c[R];
            double a[R];
#pragma unroll
            for (int u = 0; u < R; u++) {
                const int e = (PF + u) * kWave + lane;
                const int32_t ee = e < d.len ? d.e0 + e : 0;
                c[u] = p.col[ee];
                a[u] = p.val[ee];
            }
#pragma unroll
            for (int u = 0; u < R; u++) {
                lc[(PF + u) * kWave + lane] = c[u];
                lv[(PF + u) * kWave + lane] = a[u];
            }
        }
#pragma unroll
        for (int u = 0; u < RW; u++) ro[u * kWave + lane] = min(er[u], e1) - d.e0;
        const bool cut = nr > 0 && ld_const(p.off, r0 + nr) > e1;
        const int hl = min(ld_const(p.off, r0), e1) - d.e0;
        TileDesc dn;
        j += gridDim.x;
        const bool more_n = next_tile(p, tm, wave, j, dn);
        wave_lds_sync();
        if (more_n) load_tile(dn);
        if (hl > 0) {  // the row that began before this tile
            Sum s = row_sum(0, hl, gw, GW);
            over_groups(s);
            if (gw == 0) {
                *(double2 *)(p.head + (int64_t)k * K + c0) = make_double2(s.s0, s.s1);
                if (!NEG) {
                    const double2 wv = *(const double2 *)(p.w + (int64_t)(r0 - 1) * K + c0);
                    aq0 += wv.x * s.s0;
                    aq1 += wv.y * s.s1;
                }
            }
        }
        for (int i0 = 0; i0 < nr; i0 += GW) {
            const int i = i0 + gw;
            const bool own = i < nr;
            const int s = own ? ro[i] : 0, t = own ? ro[i + 1] : 0;
            const bool big = t - s > kSerialK;
            if (own && !big) {
                double2 w{0.0, 0.0};
                if (!NEG) w = ld2(p.w, (uint32_t)(r0 + i) * (uint32_t)K + (uint32_t)c0);
                const Sum a = row_sum(s, t, 0, 1);
                emit(k, r0 + i, cut && i == nr - 1, a, w);
            }
            for (uint64_t m = __ballot(big); m; ) {
                const int b = __builtin_ctzll(m) / KL;  // its group
                m &= ~(((KL < 64 ? 1ull << (KL & 63) : 0ull) - 1ull) << (b * KL));
                const int bs = ro[i0 + b], bt = ro[i0 + b + 1];
                double2 w{0.0, 0.0};
                if (!NEG) w = ld2(p.w, (uint32_t)(r0 + i0 + b) * (uint32_t)K + (uint32_t)c0);
                Sum a = row_sum(bs, bt, gw, GW);
                over_groups(a);
                if (gw == 0) emit(k, r0 + i0 + b, cut && i0 + b == nr - 1, a, w);
            }
        }
        wave_lds_sync();
        d = dn;
        more = more_n;
    }
    if (NEG) return;
    Sum s{aq0, aq1};
    over_groups(s);
    if (gw == 0) {
        red[wave * K + c0] = s.s0;
        red[wave * K + c0 + 1] = s.s1;
    }
    __syncthreads();
    if (tid < K) p.pa[(int64_t)blockIdx.x * K + tid] = (red[tid] + red[K + tid]) + (red[2 * K + tid] + red[3 * K + tid]);
}

// sum of a cut row's parts by the workgroup: thread = t * K + c; threads c < K
// get column c's (red: kWavesPerBlock * K doubles)
template <int K>
__device__ __forceinline__ double item_sum(const NfItem &it, const double *head, const double *tail, double *red) {
    const int c = threadIdx.x % K, t = threadIdx.x / K;
    constexpr int TP = kBlock / K;
    double s = 0.0;
    int32_t k = it.t0 + t;
    for (; k + 3 * TP < it.t1; k += 4 * TP) {
        const double a0 = head[(int64_t)k * K + c], a1 = head[(int64_t)(k + TP) * K + c];
        const double a2 = head[(int64_t)(k + 2 * TP) * K + c], a3 = head[(int64_t)(k + 3 * TP) * K + c];
        s += (a0 + a1) + (a2 + a3);
    }
    for (; k < it.t1; k += TP) s += head[(int64_t)k * K + c];
    if (t == 0) s += tail[(int64_t)(it.t0 - 1) * K + c];
    return block_column_sum<K>(s, red);
}

// projected iteration: the cut rows of the eliminated FE, before the other rows read them
template <int K>
__global__ __launch_bounds__(kBlock) void k_nf_fix_neg(const NfItem *items, int32_t n, const double *head,
                                                       const double *tail, double *neg, const int32_t *all_done) {
    if (*all_done) return;
    __shared__ double red[kWavesPerBlock * K];
    for (int32_t i = blockIdx.x; i < n; i += gridDim.x) {
        const NfItem it = items[i];
        const double s = item_sum<K>(it, head, tail, red);
        if (threadIdx.x < K) neg[(int64_t)it.row * K + threadIdx.x] = -s;
    }
}

// one column's entry of NfCols
struct ColCoef {
    double ia, iold, cq, cv, co, chb, cx, ch, beta1, chb2, cx2, ch2, err;
    int32_t on, upd, due, test, upd2, last, undo, bad;
};
__device__ __forceinline__ ColCoef load_coef(const NfCols *n, int c) {
    return {n->ia[c],   n->iold[c], n->cq[c],  n->cv[c],   n->co[c],   n->chb[c],  n->cx[c],   n->ch[c],  n->beta1[c],
            n->chb2[c], n->cx2[c],  n->ch2[c], n->err[c],  n->on[c],   n->upd[c],  n->due[c],  n->test[c], n->upd2[c], n->last[c],
            n->undo[c], n->bad[c]};
}
__device__ __forceinline__ void store_coef(NfCols *n, int c, const ColCoef &f) {
    n->ia[c] = f.ia;
    n->iold[c] = f.iold;
    n->cq[c] = f.cq;
    n->cv[c] = f.cv;
    n->co[c] = f.co;
    n->chb[c] = f.chb;
    n->cx[c] = f.cx;
    n->ch[c] = f.ch;
    n->beta1[c] = f.beta1;
    n->err[c] = f.err;
    n->chb2[c] = f.chb2;
    n->cx2[c] = f.cx2;
    n->ch2[c] = f.ch2;
    n->on[c] = f.on;
    n->upd[c] = f.upd;
    n->due[c] = f.due;
    n->test[c] = f.test;
    n->upd2[c] = f.upd2;
    n->last[c] = f.last;
    n->undo[c] = f.undo;
    n->bad[c] = f.bad;
}

// beta^2 = v'Mv - alpha^2 with alpha = ||w'|| / beta of the iteration before: v'Mv
// carries rounding of a few eps (|v| = 1; the diagonal's 1 is off by up to n eps / 8
// for n = 128 equal observations, the largest level without an entry of its own),
// and an error of beta^2 goes on times alpha^2 / beta^2.  A column with noise keeps
// err / beta^2 below 1e-10 (condition numbers to 1e4, 1700 iterations).  It grows to 1
// where the FEs explain a column in full, once ||r|| is between 1e-6 and 1e-8 of ||b||, and is
// there at once for a v in the null space of A (an FE collinear with the
// eliminated one) or an exhausted Krylov space.  ||A'r|| hangs on the product
// alpha beta, which stays right, but ||r|| on the betas alone.  A column whose
// err / beta^2 passes kNfLost before it stops is left out from there, and starts
// over on the observations when the others have stopped; there beta =
// ||A v - alpha u|| comes from the vectors.
constexpr double kNfErr = 16.0 * 2.220446049250313e-16, kNfLost = 1e-2;

// alpha and the rotations of the last iteration, from ||w||^2
__device__ __forceinline__ void rotate_step(LsmrState<double> &s, ColCoef &f, double wsq, int c, ColOps *ops) {
    const double nw = sqrt(wsq);
    f.iold = f.ia;
    s.alpha = nw / s.beta;
    f.ia = nw > 0.0 ? 1.0 / nw : 1.0;
    s.inv_alpha = 1.0;
    fin_rotate<double>(s, c, ops);
}
// A stopping rule holds whatever ||x|| is (src/utils/lsmr.jl:192-215; ||x||
// only loosens the two rules on ||r||).
__device__ __forceinline__ bool stops_anyway(const LsmrState<double> &s) {
    const double test1 = s.normr / s.normb, test2 = s.normAr / (s.normA * s.normr), test3 = 1.0 / s.condA;
    return s.iter >= s.maxiter || 1.0 + test3 <= 1.0 || 1.0 + test2 <= 1.0 || 1.0 + test1 <= 1.0 ||
           test3 <= s.ctol || test2 <= s.atol || test1 <= s.btol;
}

// beta of this iteration from w'Mw, and w'
__device__ __forceinline__ void beta_step(LsmrState<double> &s, ColCoef &f, double wMw, int c, ColOps *ops) {
    const double alpha = s.alpha, beta = s.beta;
    const double vMv = wMw * f.ia * f.ia;
    const double co = s.iter == 0 ? 0.0 : -(alpha * beta) * f.iold;
    double b2 = fma(-alpha, alpha, vMv);
    f.err = kNfErr + (f.due ? f.err * (alpha / beta) * (alpha / beta) : 0.0);
    if (!(f.err < kNfLost * b2)) {
        if (!f.due || !stops_anyway(s)) {
            s.done = f.bad = 1;
            f.upd = f.upd2 = 0;
            return;
        }
        b2 = b2 > kNfErr ? b2 : kNfErr;  // (it stops where ||x|| is known: nothing hangs on beta)
    }
    fin_after_db<double>(s, b2, MODE_ITER, c, ops);
    f.beta1 = beta;
    f.cq = f.ia;
    f.cv = -vMv * f.ia;
    f.co = co;
    f.on = f.due = 1;
}

// The scalar step of one column, from w'Mw, ||w||^2 and ||x||^2: the stopping
// rules of the iteration before last, alpha and the rotations of the last,
// beta of this one.
__device__ __forceinline__ void scalar_step(LsmrState<double> &s, ColCoef &f, double wMw, double wsq, double xsq,
                                            int c, ColOps *ops) {
    if (!s.done && f.test) {
        // (beta of the iteration after it has been formed: its count and beta
        // are put back if the column stops)
        s.iter -= 1;
        fin_after_update<double>(s, xsq, c, ops);
        if (s.done) s.beta = f.beta1;
        else s.iter += 1;
    }
    f.test = f.on = f.upd = 0;
    if (s.done) return;
    if (f.due) {
        rotate_step(s, f, wsq, c, ops);
        f.chb = s.c_hbar;
        f.cx = s.c_x;
        f.ch = s.c_h;
        f.upd = f.test = 1;
    }
    beta_step(s, f, wMw, c, ops);
}

// The same with the updates of iterations j and j + 1 (j odd) in one step,
// that of iteration j + 2, which leaves h, hbar and x alone in every other
// step: 14 vectors read and written in two iterations instead of 20 (32
// columns, 1.1e6 levels: 198 and 568 us in turn, at 5.6 - 6.4 TB/s, instead of
// 575 each time; a solve 361 -> 291 ms).  ||x||
// after both, xsq and xsq2, is known in iteration j + 3 (even): the rules of
// both are looked at there, on the states a and b kept after their rotations.
// A column for which a rule holds without ||x|| (nearly always one of these is
// the first) goes no further (last); where one that needs ||x|| held after j,
// x takes the update of j + 1 back (undo).  That update is finite then: a
// rotation breaks down only where alpha = 0, and there stops_anyway held.
__device__ __forceinline__ void scalar_step_pair(LsmrState<double> &s, ColCoef &f, LsmrState<double> &a,
                                                 LsmrState<double> &b, bool even, double wMw, double wsq, double xsq,
                                                 double xsq2, int c, ColOps *ops) {
    f.on = f.undo = 0;
    if (s.done) {
        f.upd = f.upd2 = 0;
        return;
    }
    if (even) {
        if (f.upd) {
            fin_after_update<double>(a, xsq, c, ops);
            bool second = false;
            if (!a.done && f.upd2) {
                second = true;
                fin_after_update<double>(b, xsq2, c, ops);
            }
            LsmrState<double> &t = second ? b : a;
            if (t.done || f.last) {
                s = t;
                s.done = 1;
                f.undo = !second && f.upd2;
                f.upd = f.upd2 = 0;
                return;
            }
        }
        f.upd = f.upd2 = 0;
    }
    if (f.last) {
        f.iold = f.ia;  // (its w is the step's wold by now)
        return;
    }
    if (f.due) {
        rotate_step(s, f, wsq, c, ops);
        if (even) {
            f.chb = s.c_hbar;
            f.cx = s.c_x;
            f.ch = s.c_h;
            f.upd = 1;
            a = s;
        } else {
            f.chb2 = s.c_hbar;
            f.cx2 = s.c_x;
            f.ch2 = s.c_h;
            f.upd2 = 1;
            b = s;
        }
        if (stops_anyway(s)) {
            f.last = 1;
            return;
        }
    }
    beta_step(s, f, wMw, c, ops);
}

// Sum of partials [i * K + c] over a thread's share (NT threads, column
// threadIdx.x % K), four chains of loads in flight
template <int K, int NT>
__device__ __forceinline__ double thread_sum(const double *p, int32_t n) {
    constexpr int R = NT / K;
    const int c = threadIdx.x % K;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int32_t j = threadIdx.x / K;
    for (; j + 3 * R < n; j += 4 * R) {
        s0 += p[(int64_t)j * K + c];
        s1 += p[(int64_t)(j + R) * K + c];
        s2 += p[(int64_t)(j + 2 * R) * K + c];
        s3 += p[(int64_t)(j + 3 * R) * K + c];
    }
    for (; j < n; j += R) s0 += p[(int64_t)j * K + c];
    return (s0 + s1) + (s2 + s3);
}

// The scalar step of K columns by NT threads: the column sums of the
// partials (lanes, then waves), and thread c < K steps column c in LDS.
template <int K, int NT, bool PAIR>
struct ScalarMem {
    double red[4][NT / kWave][K];
    LsmrState<double> state[K], snap[PAIR ? 2 : 1][PAIR ? K : 1];
    ColCoef coef[K];
    ColOps ops;
};
template <int K, int NT, bool PAIR>
__device__ __forceinline__ void scalar_block(const NfScalars &p, ScalarMem<K, NT, PAIR> &m) {
    constexpr int W = NT / kWave;
    const int c = threadIdx.x, lane = c & (kWave - 1), wave = c / kWave;
    const bool even = PAIR && p.even, needx = !PAIR || even;
    if (c < K) {
        m.state[c] = ((const LsmrState<double> *)p.sin)[c];
        m.coef[c] = load_coef(p.cin, c);
    }
    if constexpr (PAIR)
        if (even && c >= kWave && c < kWave + 2 * K)
            m.snap[(c - kWave) / K][(c - kWave) % K] = ((const LsmrState<double> *)p.snap)[c - kWave];
    const double a = column_allreduce<K>(thread_sum<K, NT>(p.pa, p.na));
    const double wsq = column_allreduce<K>(thread_sum<K, NT>(p.pw, p.nw));
    const double xsq = needx ? column_allreduce<K>(thread_sum<K, NT>(p.px, p.nw)) : 0.0;
    const double xsq2 = PAIR && even ? column_allreduce<K>(thread_sum<K, NT>(p.px2, p.nw)) : 0.0;
    if (lane < K) {
        m.red[0][wave][lane] = a;
        m.red[1][wave][lane] = wsq;
        m.red[2][wave][lane] = xsq;
        m.red[3][wave][lane] = xsq2;
    }
    __syncthreads();
    if (c < K) {
        double t[4];
        for (int q = 0; q < (PAIR ? 4 : 3); q++) {
            double x[4] = {0.0, 0.0, 0.0, 0.0};
            for (int w = 0; w < W; w += 4)
#pragma unroll
                for (int u = 0; u < 4; u++) x[u] += m.red[q][w + u][c];
            t[q] = (x[0] + x[1]) + (x[2] + x[3]);
        }
        if constexpr (PAIR)
            scalar_step_pair(m.state[c], m.coef[c], m.snap[0][c], m.snap[1][c], even, t[0], t[1], t[2], t[3], c,
                             &m.ops);
        else scalar_step(m.state[c], m.coef[c], t[0], t[1], t[2], c, &m.ops);
    }
    __syncthreads();
}
// the result of the launch's workgroup 0, and *all_done
template <int K, int NT, bool PAIR>
__device__ __forceinline__ void scalar_keep(const NfScalars &p, const ScalarMem<K, NT, PAIR> &m) {
    const int c = threadIdx.x;
    if (c < K) {
        ((LsmrState<double> *)p.sout)[c] = m.state[c];
        store_coef(p.cout, c, m.coef[c]);
        if constexpr (PAIR) {
            const int i = p.even ? 0 : 1;
            ((LsmrState<double> *)p.snap)[i * K + c] = m.snap[i][c];
        }
    }
    if (c == 0) {
        int all = 1, bad = 0;
        for (int q = 0; q < K; q++) {
            all &= m.state[q].done && !m.coef[q].undo ? 1 : 0;
            bad |= m.coef[q].bad;
        }
        if (all) *p.all_done = (bad ? kNfStartOver : 1) + p.copy;
    }
}

// The step's workgroups do the scalar step themselves while each of the
// partials has at most kNfFold values: two launches an iteration then beat
// three (N = 1e4 to 3.6e4: 20.6 -> 17.5 us an iteration; 24 such panels at once
// 27.5 -> 24.7 ms). Past it every workgroup reads too much: with 20000 values
// (N = 1e7) the step took 22 us, against 7.4 + 5.0 us as two launches. And past
// kNfFoldStep workgroups of the step the updates in pairs, which need the
// launch, save more than it costs (1.1e6 levels, 1150 workgroups: a solve 23.8
// folded, 22.4 ms; 2.2e5 levels, 216: 14.4 both).
constexpr int64_t kNfFold = 2048;
constexpr unsigned kNfFoldStep = 512;

// w' = cq q + cv w + co wold over wold, ||w'||^2, and by MODE
//  kNfFolded  the update of hbar, x and h with v = ia w, and ||x||^2.  Every
//             workgroup does the scalar step itself first, from the partials of
//             the product and of the step before (a launch less; see kNfFold),
//             and reads and writes alternate copies of the state and of the
//             step's partials.
//  kNfHeavy   two updates, with v = iold wold and v = ia w, and ||x||^2 after each
//  kNfLight   x takes back its last update in columns that stopped before it
// The first fix_blocks workgroups have the cut rows (split), one at a time.
template <int K, int MODE>
__global__ __launch_bounds__(kBlock) void k_nf_step(NfStep p) {
    if (*p.all_done) return;
    constexpr bool FOLD = MODE == kNfFolded, HEAVY = MODE == kNfHeavy;
    __shared__ double red[kWavesPerBlock * K];
    __shared__ ScalarMem<FOLD ? K : 1, kBlock, false> sm;
    const int tid = threadIdx.x;
    if constexpr (FOLD) {
        scalar_block<K, kBlock, false>(p.fold, sm);
        if (blockIdx.x == 0) scalar_keep<K, kBlock, false>(p.fold, sm);
    }
    auto coef = [&](int c) -> ColCoef {
        if constexpr (FOLD) return sm.coef[c];
        else return load_coef(p.cols, c);
    };
    // whether x, hbar and h (kNfLight: x and hbar) of the column are touched
    auto touched = [](const ColCoef &f) { return MODE == kNfLight ? f.undo != 0 : f.upd != 0; };
    // the updates of one element; w, o = its w and wold; adds to the sums of x^2
    auto update = [](const ColCoef &f, double &h, double &hb, double &x, double w, double o, double &sx, double &sx2) {
        if constexpr (MODE == kNfLight) {
            x -= f.cx2 * hb;
        } else {
            hb = hb * f.chb + h;
            x = x + f.cx * hb;
            h = h * f.ch + (HEAVY ? o * f.iold : w * f.ia);
            sx += x * x;
            if (HEAVY && f.upd2) {
                hb = hb * f.chb2 + h;
                x = x + f.cx2 * hb;
                h = h * f.ch2 + w * f.ia;
                sx2 += x * x;
            }
        }
    };
    if (blockIdx.x < p.fix_blocks) {
        const int c = tid % K;
        const ColCoef f = coef(c);
        const bool on = f.on != 0, touch = touched(f);
        double acc = 0.0, accx = 0.0, accx2 = 0.0;
        for (int32_t i = blockIdx.x; i < p.nitem; i += p.fix_blocks) {
            const NfItem it = p.items[i];
            if (it.row >= p.row0 && it.row < p.row0 + p.rown) continue;
            const int64_t e = (int64_t)it.row * K + c;
            double w = 0.0, o = 0.0, h = 0.0, hb = 0.0, x = 0.0;
            if (tid < K) {
                w = p.w[e];
                o = p.wold[e];
                if (touch) {
                    if (MODE != kNfLight) h = p.h[e];
                    hb = p.hbar[e];
                    x = p.x[e];
                }
            }
            const double s = item_sum<K>(it, p.head, p.tail, red);
            if (tid < K && touch) {
                update(f, h, hb, x, w, o, accx, accx2);
                p.x[e] = x;
                if (MODE != kNfLight) {
                    p.hbar[e] = hb;
                    p.h[e] = h;
                }
            }
            if (tid < K && on) {
                const double n = f.cq * (w + s) + f.cv * w + f.co * o;
                p.wold[e] = n;
                acc += n * n;
            }
        }
        if (tid < K) {
            p.pw[(int64_t)blockIdx.x * K + tid] = acc;
            if (MODE != kNfLight) p.px[(int64_t)blockIdx.x * K + tid] = accx;
            if (HEAVY) p.px2[(int64_t)blockIdx.x * K + tid] = accx2;
        }
        return;
    }
    // V adjacent columns of a row per thread (16-byte accesses), U of them in flight
    constexpr int V = K == 1 ? 1 : 2, KV = K / V, U = 4 / V;
    using Vec = VecC<double, V>;
    const int c0 = tid % KV * V;
    ColCoef f[V];
    bool on[V], touch[V], any = false, anyu = false;
#pragma unroll
    for (int v = 0; v < V; v++) {
        f[v] = coef(c0 + v);
        on[v] = f[v].on != 0;
        touch[v] = touched(f[v]);
        any |= on[v];
        anyu |= touch[v];
    }
    double acc[V] = {}, accx[V] = {}, accx2[V] = {};
    if (any || anyu) {
        const int64_t n = (p.p - p.rown) * KV, skip0 = p.row0 * KV, skipn = p.rown * KV;
        const int64_t stride = (int64_t)(gridDim.x - p.fix_blocks) * kBlock;
        for (int64_t b = (int64_t)(blockIdx.x - p.fix_blocks) * kBlock + tid; b < n; b += U * stride) {
            uint32_t ee[U];
            Vec q[U], w[U], o[U], h[U], hb[U], x[U];
            bool in[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                in[u] = b + u * stride < n;
                const int64_t e = in[u] ? b + u * stride : b;
                const uint32_t at = (uint32_t)(e < skip0 ? e : e + skipn), r = at / KV;
                ee[u] = at * V;
                if ((p.split[r >> 5] >> (r & 31)) & 1) in[u] = false;
                q[u] = ldv<V>(p.q, ee[u]);
                w[u] = ldv<V>(p.w, ee[u]);
                o[u] = ldv<V>((const double *)p.wold, ee[u]);
                if (anyu) {
                    if (MODE != kNfLight) h[u] = ldv<V>((const double *)p.h, ee[u]);
                    hb[u] = ldv<V>((const double *)p.hbar, ee[u]);
                    x[u] = ldv<V>((const double *)p.x, ee[u]);
                }
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (!in[u]) continue;
                if (anyu) {
#pragma unroll
                    for (int v = 0; v < V; v++)
                        if (touch[v])
                            update(f[v], h[u].v[v], hb[u].v[v], x[u].v[v], w[u].v[v], o[u].v[v], accx[v], accx2[v]);
                    stv<V>(p.x, ee[u], x[u]);
                    if (MODE != kNfLight) {
                        stv<V>(p.hbar, ee[u], hb[u]);
                        stv<V>(p.h, ee[u], h[u]);
                    }
                }
                if (!any) continue;
#pragma unroll
                for (int v = 0; v < V; v++) {
                    if (!on[v]) continue;
                    o[u].v[v] = f[v].cq * q[u].v[v] + f[v].cv * w[u].v[v] + f[v].co * o[u].v[v];
                    acc[v] += o[u].v[v] * o[u].v[v];
                }
                stv<V>(p.wold, ee[u], o[u]);
            }
        }
    }
#pragma unroll
    for (int v = 0; v < V; v++) {
        const double s = block_column_sum<KV>(acc[v], red);
        if (tid < KV) p.pw[(int64_t)blockIdx.x * K + tid * V + v] = s;
        if (MODE != kNfLight) {
            const double sx = block_column_sum<KV>(accx[v], red);
            if (tid < KV) p.px[(int64_t)blockIdx.x * K + tid * V + v] = sx;
        }
        if (HEAVY) {
            const double sx = block_column_sum<KV>(accx2[v], red);
            if (tid < KV) p.px2[(int64_t)blockIdx.x * K + tid * V + v] = sx;
        }
    }
}

// the scalar step as a launch of its own
template <int K>
__global__ __launch_bounds__(kFinBlock) void k_nf_scalars(NfScalars p) {
    if (*p.all_done) return;
    __shared__ ScalarMem<K, kFinBlock, true> sm;
    scalar_block<K, kFinBlock, true>(p, sm);
    scalar_keep<K, kFinBlock, true>(p, sm);
}

__global__ void k_nf_init_cols(const LsmrState<double> *st, int K, NfCols *cols) {
    const int c = threadIdx.x;
    if (c >= kMaxK) return;
    cols->ia[c] = 1.0;  // k_init_vectors left v normalized
    cols->iold[c] = 0.0;
    cols->cq[c] = cols->cv[c] = cols->co[c] = 0.0;
    cols->chb[c] = cols->cx[c] = cols->ch[c] = 0.0;
    cols->beta1[c] = 0.0;
    cols->on[c] = c < K && !st[c].done ? 1 : 0;
    cols->upd[c] = cols->due[c] = cols->test[c] = 0;
    cols->chb2[c] = cols->cx2[c] = cols->ch2[c] = cols->err[c] = 0.0;
    cols->upd2[c] = cols->last[c] = cols->undo[c] = cols->bad[c] = 0;
}

template <int K>
static const void *apply_kernel() {
    if constexpr (K == 1) return (const void *)k_nf_apply1<false>;
    else return (const void *)k_nf_apply<K, false>;
}

template <int K>
static void apply_launch(const NfApply &a, unsigned nb, hipStream_t st) {
    if constexpr (K == 1) {
        if (a.neg) hipLaunchKernelGGL(k_nf_apply1<true>, dim3(nb), dim3(kBlock), 0, st, a);
        else hipLaunchKernelGGL(k_nf_apply1<false>, dim3(nb), dim3(kBlock), 0, st, a);
    } else {
        if (a.neg) hipLaunchKernelGGL((k_nf_apply<K, true>), dim3(nb), dim3(kBlock), 0, st, a);
        else hipLaunchKernelGGL((k_nf_apply<K, false>), dim3(nb), dim3(kBlock), 0, st, a);
    }
}

template <typename F>
static void for_width(int K, F &&f) {
    switch (K) {
        case 1: f(std::integral_constant<int, 1>{}); break;
        case 2: f(std::integral_constant<int, 2>{}); break;
        case 4: f(std::integral_constant<int, 4>{}); break;
        case 8: f(std::integral_constant<int, 8>{}); break;
        case 16: f(std::integral_constant<int, 16>{}); break;
        default: f(std::integral_constant<int, 32>{}); break;
    }
}

static unsigned resident_blocks(const void *kernel) {
    int dev = 0, cus = 0, nb = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, kBlock, 0) != hipSuccess || nb < 1 || cus < 1) {
        (void)hipGetLastError();
        return 1024;
    }
    return (unsigned)(nb * cus);
}

unsigned nf_apply_blocks(int K, int32_t ntiles) {
    unsigned r = 1024;
    for_width(K, [&](auto k) { r = resident_blocks(apply_kernel<decltype(k)::value>()); });
    // a multiple of 8 (TileMap spreads a launch over the XCDs by j mod 8)
    const unsigned rounds = (unsigned)(ntiles + kWavesPerBlock - 1) / kWavesPerBlock;
    return std::max(8u, std::min(r, (rounds + 7) / 8 * 8) / 8 * 8);
}

void nf_apply(int K, const NfApply &a, unsigned blocks, hipStream_t st) {
    for_width(K, [&](auto k) { apply_launch<decltype(k)::value>(a, blocks, st); });
}

void nf_fix_neg(int K, const NfItem *items, int32_t n, const double *head, const double *tail, double *neg,
                const int32_t *all_done, hipStream_t st) {
    if (n <= 0) return;
    const unsigned nb = std::min((unsigned)n, 2048u);
    for_width(K, [&](auto k) {
        hipLaunchKernelGGL((k_nf_fix_neg<decltype(k)::value>), dim3(nb), dim3(kBlock), 0, st, items, n, head, tail,
                           neg, all_done);
    });
}

bool nf_folds(int K, unsigned apply_blocks, unsigned step_blocks) {
    return (int64_t)std::max(apply_blocks, step_blocks) * K <= kNfFold && step_blocks <= kNfFoldStep;
}
void nf_scalars(int K, const NfScalars &a, hipStream_t st) {
    for_width(K, [&](auto k) {
        hipLaunchKernelGGL((k_nf_scalars<decltype(k)::value>), dim3(1), dim3(kFinBlock), 0, st, a);
    });
}

void nf_step(int K, const NfStep &s, unsigned blocks, hipStream_t st) {
    for_width(K, [&](auto k) {
        constexpr int W = decltype(k)::value;
        auto kernel = s.mode == kNfFolded  ? k_nf_step<W, kNfFolded>
                      : s.mode == kNfHeavy ? k_nf_step<W, kNfHeavy>
                                           : k_nf_step<W, kNfLight>;
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kBlock), 0, st, s);
    });
}

void nf_init_cols(int K, const void *state, NfCols *cols, hipStream_t st) {
    hipLaunchKernelGGL(k_nf_init_cols, dim3(1), dim3(kWave), 0, st, (const LsmrState<double> *)state, K, cols);
}

// ---------------------------------------------------------------------------
// construction of M
// ---------------------------------------------------------------------------
constexpr int kHeadItems = 8;
constexpr int kHeadTile = kBlock * kHeadItems;

__global__ void k_nf_gather(const int32_t *__restrict__ in, const int32_t *__restrict__ perm, int64_t n,
                            int32_t *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = in[perm[i]];
}

__device__ __forceinline__ bool cell_head(const int32_t *ka, const int32_t *kb, int64_t i, int64_t n) {
    return i < n && (i == 0 || ka[i] != ka[i - 1] || kb[i] != kb[i - 1]);
}

// cells begin where the sorted pair changes: their count per chunk of
// positions, then (after a scan) their levels and first positions
__global__ __launch_bounds__(kBlock) void k_nf_count_cells(const int32_t *__restrict__ ka,
                                                           const int32_t *__restrict__ kb, int64_t n,
                                                           uint32_t *__restrict__ cnt) {
    __shared__ uint32_t ws[kWavesPerBlock];
    const int64_t base = (int64_t)blockIdx.x * kHeadTile;
    uint32_t s = 0;
#pragma unroll
    for (int q = 0; q < kHeadItems; q++) {
        const uint64_t m = __ballot(cell_head(ka, kb, base + q * kBlock + threadIdx.x, n));
        s += (uint32_t)__popcll(m);
    }
    if ((threadIdx.x & (kWave - 1)) == 0) ws[threadIdx.x / kWave] = s;
    __syncthreads();
    if (threadIdx.x == 0) cnt[blockIdx.x] = ws[0] + ws[1] + ws[2] + ws[3];
}

__global__ __launch_bounds__(kBlock) void k_nf_write_cells(const int32_t *__restrict__ ka,
                                                           const int32_t *__restrict__ kb, int64_t n,
                                                           const uint32_t *__restrict__ first, int64_t ncell,
                                                           int32_t *__restrict__ ca, int32_t *__restrict__ cb,
                                                           int32_t *__restrict__ start) {
    __shared__ uint32_t ws[kHeadItems][kWavesPerBlock];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const int64_t base = (int64_t)blockIdx.x * kHeadTile;
    uint64_t m[kHeadItems];
#pragma unroll
    for (int q = 0; q < kHeadItems; q++) {
        m[q] = __ballot(cell_head(ka, kb, base + q * kBlock + threadIdx.x, n));
        if (lane == 0) ws[q][wave] = (uint32_t)__popcll(m[q]);
    }
    __syncthreads();
    uint32_t at = first[blockIdx.x];
#pragma unroll
    for (int q = 0; q < kHeadItems; q++) {
        uint32_t o = at;
        for (int v = 0; v < kWavesPerBlock; v++) {
            if (v < wave) o += ws[q][v];
            at += ws[q][v];
        }
        if ((m[q] >> lane) & 1) {
            const int64_t i = base + q * kBlock + threadIdx.x;
            o += (uint32_t)__popcll(m[q] & lanes_lt(lane));
            ca[o] = ka[i];
            cb[o] = kb[i];
            start[o] = (int32_t)i;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) start[ncell] = (int32_t)n;
}

// off[k] = first position whose (sorted) key is >= k
__global__ void k_nf_offsets(const int32_t *__restrict__ keys, int64_t n, int32_t nlev, int32_t *__restrict__ off) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j > n) return;
    const int32_t prev = j == 0 ? -1 : keys[j - 1], cur = j == n ? nlev : keys[j];
    for (int32_t k = prev + 1; k <= cur; k++) off[k] = (int32_t)j;
}

// rows[k] += entries of level k
__global__ void k_nf_add_counts(const int32_t *__restrict__ off, int64_t nlev, uint32_t *__restrict__ rows) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nlev) rows[k] += (uint32_t)(off[k + 1] - off[k]);
}

__global__ void k_nf_zero(uint32_t *a, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = 0;
}

// entries of one orientation of a pair: e-th in row order is cell perm[e] (or e)
__global__ void k_nf_place(const int32_t *__restrict__ rowlev, const int32_t *__restrict__ collev,
                           const int32_t *__restrict__ perm, int64_t ncell, const int32_t *__restrict__ off,
                           const uint32_t *__restrict__ cur, int32_t coloff, int32_t *__restrict__ dst,
                           int32_t *__restrict__ col) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ncell) return;
    const int64_t cell = perm ? perm[e] : e;
    const int32_t row = rowlev[cell];
    const int32_t d = (int32_t)cur[row] + (int32_t)(e - off[row]);
    dst[cell] = d;
    col[d] = coloff + collev[cell];
}

__global__ void k_nf_big_cells(const int32_t *__restrict__ start, int64_t ncell, int32_t *__restrict__ list,
                               uint32_t *__restrict__ count) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < ncell && start[i + 1] - start[i] > kNfBigCell) list[atomicAdd(count, 1u)] = (int32_t)i;
}

// M's entry of a cell: the sum of cache_a * cache_b over its observations, in
// their order (a thread per cell; a workgroup per cell of many)
__global__ __launch_bounds__(kBlock) void k_nf_cell_values(const int32_t *__restrict__ start, int64_t ncell,
                                                           const int32_t *__restrict__ order,
                                                           const double *__restrict__ ca, const double *__restrict__ cb,
                                                           const int32_t *__restrict__ dsta,
                                                           const int32_t *__restrict__ dstb, double *__restrict__ val) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= ncell) return;
    const int32_t s = start[i], t = start[i + 1];
    if (t - s > kNfBigCell) return;
    double sum = 0.0;
    for (int32_t e = s; e < t; e++) {
        const int32_t o = order ? order[e] : e;
        sum += ca[o] * cb[o];
    }
    val[dsta[i]] = sum;
    val[dstb[i]] = sum;
}

__global__ __launch_bounds__(kBlock) void k_nf_big_values(const int32_t *__restrict__ list,
                                                          const int32_t *__restrict__ start,
                                                          const int32_t *__restrict__ order,
                                                          const double *__restrict__ ca, const double *__restrict__ cb,
                                                          const int32_t *__restrict__ dsta,
                                                          const int32_t *__restrict__ dstb, double *__restrict__ val) {
    __shared__ double red[kWavesPerBlock];
    const int32_t i = list[blockIdx.x], s = start[i], t = start[i + 1];
    double sum = 0.0;
    for (int32_t e = s + threadIdx.x; e < t; e += kBlock) {
        const int32_t o = order ? order[e] : e;
        sum += ca[o] * cb[o];
    }
    sum = wave_sum(sum);
    if ((threadIdx.x & (kWave - 1)) == 0) red[threadIdx.x / kWave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        sum = (red[0] + red[1]) + (red[2] + red[3]);
        val[dsta[i]] = sum;
        val[dstb[i]] = sum;
    }
}

// What scale!'s sum leaves on M's diagonal, per large level: its sum rounds once
// per observation (1e6 weights of 0.1: d = 1 + 1.3e-11), too much for beta^2 =
// v'Mv - alpha^2 to carry.  An entry at the row's end holds d - 1; levels of fewer
// observations are within kNfErr.
__global__ void k_nf_add_diag(const int32_t *__restrict__ rows, int32_t n, uint32_t *__restrict__ cnt) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) cnt[rows[i]] += 1;
}

// (after every pair's entries: cur is at the row's last)
__global__ void k_nf_place_diag(const int32_t *__restrict__ rows, int32_t n, const uint32_t *__restrict__ cur,
                                int32_t *__restrict__ dpos, int32_t *__restrict__ col) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t d = (int32_t)cur[rows[i]];
    dpos[i] = d;
    col[d] = rows[i];
}

// scale^2 times the sum, less 1
__device__ __forceinline__ double diag_rest(double s, double r) {
    return s > 0.0 && s <= 1.7976931348623157e308 ? fma(r, r * s, -1.0) : 0.0;  // (not a sum that overflowed)
}

// all but the levels [skip0, skip1) of the list
__global__ void k_nf_diag(const int32_t *__restrict__ rows, int32_t n, int32_t skip0, int32_t skip1,
                          const double *__restrict__ sum, const double *__restrict__ scale,
                          const int32_t *__restrict__ dpos, int32_t *__restrict__ col, double *__restrict__ val) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || (i >= skip0 && i < skip1)) return;
    col[dpos[i]] = rows[i];
    val[dpos[i]] = diag_rest(sum[i], scale[rows[i]]);
}

// The rows of FE s in the projected iteration, a workgroup per large level: they
// form (A_s'A_s)^-1 A_s'A_o v, so their entries are divided by d; the one on the
// diagonal is taken out (its element of v is being written by the same launch).
__global__ __launch_bounds__(kBlock) void k_nf_project_rows(const int32_t *__restrict__ rows,
                                                            const double *__restrict__ sum,
                                                            const double *__restrict__ scale,
                                                            const int32_t *__restrict__ off,
                                                            int32_t *__restrict__ col, double *__restrict__ val) {
    const int32_t i = blockIdx.x, k = rows[i], e0 = off[k], e1 = off[k + 1] - 1;
    const double f = 1.0 / (1.0 + diag_rest(sum[i], scale[k]));
    for (int32_t e = e0 + threadIdx.x; e < e1; e += kBlock) val[e] *= f;
    if (threadIdx.x == 0) {
        col[e1] = col[e0];
        val[e1] = 0.0;
    }
}

// Tile starts of rows [ra, rb): every T units (an entry is one, a row kNfRow
// more).  A boundary goes to the end of the row it falls into when at most
// kNfSlack units of it are left, else it cuts the row (in[k] = that row).
__global__ void k_nf_tiles(const int32_t *__restrict__ off, int32_t ra, int32_t rb, int32_t T, int32_t nt,
                           int32_t *__restrict__ te, int32_t *__restrict__ tr, int32_t *__restrict__ in) {
    const int32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nt) return;
    const int64_t u = (int64_t)k * T;
    auto f = [&](int32_t r) { return (int64_t)(off[r] - off[ra]) + (int64_t)kNfRow * (r - ra); };
    int32_t lo = ra, hi = rb;
    while (lo < hi) {
        const int32_t mid = lo + (hi - lo) / 2;
        if (f(mid) >= u) hi = mid;
        else lo = mid + 1;
    }
    int32_t r = lo, e = off[lo], cut = -1;
    if (lo > ra && f(lo) - u > kNfSlack) {
        const int64_t inside = u - f(lo - 1) - kNfRow;
        if (inside > 0) {
            e = (int32_t)(off[lo - 1] + inside);
            cut = lo - 1;
        } else {
            r = lo - 1;
            e = off[lo - 1];
        }
    }
    te[k] = e;
    tr[k] = r;
    in[k] = cut;
}

// first column of each tile
__global__ void k_nf_tile_cols(const int32_t *__restrict__ te, int32_t nt, const int32_t *__restrict__ col,
                               int32_t nnz, int32_t *__restrict__ out) {
    const int32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nt) out[k] = te[k] < nnz ? col[te[k]] : 0;
}

// order == nullptr: the tiles' own
__global__ void k_nf_tile_list(const int32_t *__restrict__ te, const int32_t *__restrict__ tr, int32_t nt,
                               const int32_t *__restrict__ order, NfTileAt *__restrict__ out) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nt) return;
    const int32_t k = order ? order[i] : i;
    out[i] = {k, te[k], tr[k], (te[k + 1] - te[k]) | (tr[k + 1] - tr[k]) << 16};
}

__global__ void k_nf_split_bits(const NfItem *__restrict__ items, int32_t n, uint32_t *__restrict__ split) {
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) atomicOr(&split[items[i].row >> 5], 1u << (items[i].row & 31));
}

namespace {
template <typename P>
int alloc(fehip_solver *h, P **ptr, int64_t n) {
    void *q = nullptr;
    const int rc = solver_alloc(h, &q, sizeof(P) * (size_t)std::max<int64_t>(n, 1));
    *ptr = (P *)q;
    return rc;
}

// construction scratch of one pair, freed when the build ends
struct PairScratch {
    int32_t *ca = nullptr, *cb = nullptr, *offa = nullptr, *offb = nullptr, *permb = nullptr;
};

struct Scratch {
    fehip_solver *h;
    std::vector<void *> v;
    ~Scratch() {
        for (void *q : v) solver_free(h, q);
    }
    template <typename P>
    int get(P **ptr, int64_t n) {
        NRC(alloc(h, ptr, n));
        v.push_back(*ptr);
        return 0;
    }
    void drop(void *q) {
        auto it = std::find(v.begin(), v.end(), q);
        if (it != v.end()) v.erase(it);
        solver_free(h, q);
    }
};
}  // namespace

void nf_free(fehip_solver *h, NormalMat &m) {
    for (NfPair &q : m.pairs)
        for (void *x : {(void *)q.order, (void *)q.start, (void *)q.dsta, (void *)q.dstb, (void *)q.big})
            solver_free(h, x);
    for (void *x : {(void *)m.off, (void *)m.col, (void *)m.val, (void *)m.tiles, (void *)m.items,
                    (void *)m.split, (void *)m.dpos})
        solver_free(h, x);
    m = NormalMat{};
}

// The order in which launches visit the tiles.  A row of many tiles (a year)
// reads all of v; a few of them one after another read it that often from
// memory.  Tiles inside such rows are visited by their first column instead, so
// that the rows' tiles over the same levels run side by side and share an
// XCD's L2; the others come first, in their own order.  Group after group
// (bounds), each within itself.
// Measured (N = 1e7, 20 years): K = 1 48.2 -> 38.2 us a product, K = 32 452 -> 394;
// 50 years of N = 2e7, K = 16: 357 -> 302.
constexpr int32_t kNfReorder = 2048;  // fewer tiles: the vectors stay in the L2s anyway
static std::vector<int32_t> tile_order(const std::vector<int32_t> &in, const std::vector<int32_t> &col, int64_t p,
                                       const std::vector<int32_t> &bounds) {
    const int32_t nt = (int32_t)in.size();
    std::vector<int32_t> order(nt);
    int shift = 0;
    while ((p >> shift) >= 1 << 16) shift++;
    for (size_t g = 0; g + 1 < bounds.size(); g++) {
        const int32_t a = bounds[g], b = bounds[g + 1];
        // inside a row: it began before the tile and goes on after it
        auto inside = [&](int32_t k) { return in[k] >= 0 && k + 1 < b && in[k + 1] == in[k]; };
        std::vector<int32_t> at((size_t)(p >> shift) + 2, 0);
        int32_t n = 0;
        for (int32_t k = a; k < b; k++) {
            if (inside(k)) at[(col[k] >> shift) + 1]++;
            else order[a + n++] = k;
        }
        at[0] = a + n;
        for (size_t i = 1; i < at.size(); i++) at[i] += at[i - 1];
        for (int32_t k = a; k < b; k++)
            if (inside(k)) order[at[col[k] >> shift]++] = k;
    }
    return order;
}

static int build(fehip_solver *h, const NfInput &in, int64_t nnz_max, int64_t far_max, NormalMat &m, int *fits) {
    const int64_t N = in.N;
    const hipStream_t st = in.stream;
    const int64_t p = in.off[in.G];
    Scratch tmp{h, {}};
    std::vector<PairScratch> ps;
    m.p = p;
    const int64_t nchunk = (N + kHeadTile - 1) / kHeadTile;
    uint32_t *cnt = nullptr, *count = nullptr;
    NRC(tmp.get(&cnt, nchunk + 1));
    NRC(tmp.get(&count, 1));
    int64_t cells = 0;
    std::vector<int64_t> fe_nnz(in.G, 0);
    for (int g = 0; g < in.G; g++) {
        fe_nnz[g] = in.nbig[g];
        m.ndiag += in.nbig[g];
    }
    for (int x = 0; x < in.G; x++)
        for (int y = x + 1; y < in.G; y++) {
            // a: FE s where it is one of the two (the internal order keeps its levels together), else the larger
            int a = x, b = y;
            if (y == in.s || (x != in.s && in.n[y] > in.n[x])) std::swap(a, b);
            m.pairs.emplace_back();
            NfPair &q = m.pairs.back();
            ps.emplace_back();
            PairScratch &w = ps.back();
            q.a = a;
            q.b = b;
            const int32_t *ka = in.ref[a], *kb = in.ref[b];
            int32_t *ska = nullptr, *skb = nullptr;
            if (!(a == in.s && b == in.t_sec)) {
                int32_t *own = nullptr, *k1 = nullptr;
                const int32_t *p1 = in.by_level[b];
                NRC(alloc(h, &q.order, N));
                if (!p1) NRC(tmp.get(&own, N));
                NRC(tmp.get(&k1, N));
                NRC(tmp.get(&ska, N));
                NRC(tmp.get(&skb, N));
                if (!p1) {
                    NRC(solver_sort(h, in.ref[b], N, in.n[b], ska, own, nullptr));
                    p1 = own;
                }
                hipLaunchKernelGGL(k_nf_gather, dim3(blocks_for(N, kBlock)), dim3(kBlock), 0, st, in.ref[a], p1, N, k1);
                NRC(solver_sort(h, k1, N, in.n[a], ska, q.order, p1));
                hipLaunchKernelGGL(k_nf_gather, dim3(blocks_for(N, kBlock)), dim3(kBlock), 0, st, in.ref[b], q.order,
                                   N, skb);
                NCHK(hipGetLastError());
                if (own) tmp.drop(own);
                tmp.drop(k1);
                ka = ska;
                kb = skb;
            }
            hipLaunchKernelGGL(k_nf_count_cells, dim3((unsigned)nchunk), dim3(kBlock), 0, st, ka, kb, N, cnt);
            NCHK(hipGetLastError());
            NRC(solver_scan(h, cnt, nchunk, cnt));
            uint32_t nc = 0;
            NCHK(hipMemcpyAsync(&nc, cnt + nchunk, sizeof(nc), hipMemcpyDeviceToHost, st));
            NCHK(hipStreamSynchronize(st));
            q.ncell = nc;
            cells += nc;
            fe_nnz[a] += nc;
            fe_nnz[b] += nc;
            m.far += (in.n[a] > kNfFarLevels ? nc : 0) + (in.n[b] > kNfFarLevels ? nc : 0);
            if (2 * cells > nnz_max || 2 * cells + m.ndiag + (int64_t)kNfRow * p > INT32_MAX) {
                *fits = 0;
                return 0;
            }
            if (m.far > far_max) {
                *fits = -1;
                return 0;
            }
            NRC(tmp.get(&w.ca, nc));
            NRC(tmp.get(&w.cb, nc));
            NRC(alloc(h, &q.start, (int64_t)nc + 1));
            hipLaunchKernelGGL(k_nf_write_cells, dim3((unsigned)nchunk), dim3(kBlock), 0, st, ka, kb, N,
                               (const uint32_t *)cnt, (int64_t)nc, w.ca, w.cb, q.start);
            NCHK(hipGetLastError());
            if (ska) tmp.drop(ska);
            if (skb) tmp.drop(skb);
            // row offsets of both orientations; b's entries in the order of its levels
            int32_t *sk = nullptr;
            NRC(tmp.get(&w.offa, in.n[a] + 1));
            NRC(tmp.get(&w.offb, in.n[b] + 1));
            NRC(tmp.get(&w.permb, nc));
            NRC(tmp.get(&sk, nc));
            hipLaunchKernelGGL(k_nf_offsets, dim3(blocks_for((int64_t)nc + 1, kBlock)), dim3(kBlock), 0, st,
                               (const int32_t *)w.ca, (int64_t)nc, (int32_t)in.n[a], w.offa);
            NRC(solver_sort(h, w.cb, nc, in.n[b], sk, w.permb, nullptr));
            hipLaunchKernelGGL(k_nf_offsets, dim3(blocks_for((int64_t)nc + 1, kBlock)), dim3(kBlock), 0, st,
                               (const int32_t *)sk, (int64_t)nc, (int32_t)in.n[b], w.offb);
            NCHK(hipGetLastError());
            tmp.drop(sk);
            // cells of many observations
            int32_t *list = nullptr;
            NRC(tmp.get(&list, N / (kNfBigCell + 1) + 1));
            hipLaunchKernelGGL(k_nf_zero, dim3(1), dim3(kWave), 0, st, count, (int64_t)1);
            hipLaunchKernelGGL(k_nf_big_cells, dim3(blocks_for(nc, kBlock)), dim3(kBlock), 0, st,
                               (const int32_t *)q.start, (int64_t)nc, list, count);
            NCHK(hipGetLastError());
            uint32_t nb = 0;
            NCHK(hipMemcpyAsync(&nb, count, sizeof(nb), hipMemcpyDeviceToHost, st));
            NCHK(hipStreamSynchronize(st));
            q.nbig = (int32_t)nb;
            if (nb) {
                NRC(alloc(h, &q.big, nb));
                NCHK(hipMemcpyAsync(q.big, list, sizeof(int32_t) * nb, hipMemcpyDeviceToDevice, st));
            }
            tmp.drop(list);
        }
    // rows: the entries of every pair a level takes part in, pair after pair, and a large level's diagonal
    m.nnz = 2 * cells + m.ndiag;
    uint32_t *cur = nullptr;
    NRC(tmp.get(&cur, p + 1));
    NRC(alloc(h, &m.off, p + 1));
    NRC(alloc(h, &m.col, m.nnz));
    NRC(alloc(h, &m.val, m.nnz));
    hipLaunchKernelGGL(k_nf_zero, dim3(blocks_for(p + 1, kBlock)), dim3(kBlock), 0, st, cur, p + 1);
    auto add = [&](const int32_t *off, int g) {
        hipLaunchKernelGGL(k_nf_add_counts, dim3(blocks_for(in.n[g], kBlock)), dim3(kBlock), 0, st, off, in.n[g],
                           cur + in.off[g]);
    };
    for (size_t i = 0; i < ps.size(); i++) {
        add(ps[i].offa, m.pairs[i].a);
        add(ps[i].offb, m.pairs[i].b);
    }
    if (m.ndiag)
        hipLaunchKernelGGL(k_nf_add_diag, dim3(blocks_for(m.ndiag, kBlock)), dim3(kBlock), 0, st, in.big_rows,
                           m.ndiag, cur);
    NCHK(hipGetLastError());
    NRC(solver_scan(h, cur, p, (uint32_t *)m.off));
    NCHK(hipMemcpyAsync(cur, m.off, sizeof(uint32_t) * p, hipMemcpyDeviceToDevice, st));
    for (size_t i = 0; i < ps.size(); i++) {
        NfPair &q = m.pairs[i];
        const PairScratch &w = ps[i];
        NRC(alloc(h, &q.dsta, q.ncell));
        NRC(alloc(h, &q.dstb, q.ncell));
        const dim3 gr(blocks_for(q.ncell, kBlock));
        hipLaunchKernelGGL(k_nf_place, gr, dim3(kBlock), 0, st, (const int32_t *)w.ca, (const int32_t *)w.cb,
                           (const int32_t *)nullptr, q.ncell, (const int32_t *)w.offa,
                           (const uint32_t *)cur + in.off[q.a], (int32_t)in.off[q.b], q.dsta, m.col);
        add(w.offa, q.a);
        hipLaunchKernelGGL(k_nf_place, gr, dim3(kBlock), 0, st, (const int32_t *)w.cb, (const int32_t *)w.ca,
                           (const int32_t *)w.permb, q.ncell, (const int32_t *)w.offb,
                           (const uint32_t *)cur + in.off[q.b], (int32_t)in.off[q.a], q.dstb, m.col);
        add(w.offb, q.b);
        NCHK(hipGetLastError());
    }
    if (m.ndiag) {
        NRC(alloc(h, &m.dpos, m.ndiag));
        hipLaunchKernelGGL(k_nf_place_diag, dim3(blocks_for(m.ndiag, kBlock)), dim3(kBlock), 0, st, in.big_rows,
                           m.ndiag, (const uint32_t *)cur, m.dpos, m.col);
        NCHK(hipGetLastError());
    }
    // tiles: of the FEs before s, of s, of those after it
    // (small problems: shorter tiles, down to a wave's two loads per lane, so that
    // every CU has some)
    const int64_t units = m.nnz + (int64_t)kNfRow * p;
    const int32_t T = (int32_t)std::min<int64_t>(kNfTile, std::max<int64_t>(kNfSlack, units / 4096));
    int64_t ends[4] = {0, in.off[in.s], in.off[in.s + 1], p}, nt[3];
    for (int g3 = 0; g3 < 3; g3++) {
        int64_t un = (int64_t)kNfRow * (ends[g3 + 1] - ends[g3]);
        for (int g = 0; g < in.G; g++)
            if (in.off[g] >= ends[g3] && in.off[g] < ends[g3 + 1]) un += fe_nnz[g];
        nt[g3] = (un + T - 1) / T;
    }
    m.ntile = (int32_t)(nt[0] + nt[1] + nt[2]);
    m.ts0 = (int32_t)nt[0];
    m.ts1 = (int32_t)(nt[0] + nt[1]);
    int32_t *tin = nullptr;
    int32_t *te = nullptr, *tr = nullptr, *tcol = nullptr;
    const bool reorder = m.ntile >= kNfReorder;
    NRC(tmp.get(&te, m.ntile + 1));
    NRC(tmp.get(&tr, m.ntile + 1));
    NRC(tmp.get(&tin, m.ntile + 1));
    NRC(alloc(h, &m.tiles, m.ntile));
    int64_t at = 0;
    for (int g3 = 0; g3 < 3; g3++) {
        if (nt[g3])
            hipLaunchKernelGGL(k_nf_tiles, dim3(blocks_for(nt[g3], kBlock)), dim3(kBlock), 0, st,
                               (const int32_t *)m.off, (int32_t)ends[g3], (int32_t)ends[g3 + 1], T, (int32_t)nt[g3],
                               te + at, tr + at, tin + at);
        at += nt[g3];
    }
    NCHK(hipGetLastError());
    const int32_t last[2] = {(int32_t)m.nnz, (int32_t)p};
    NCHK(hipMemcpyAsync(te + m.ntile, &last[0], sizeof(int32_t), hipMemcpyHostToDevice, st));
    NCHK(hipMemcpyAsync(tr + m.ntile, &last[1], sizeof(int32_t), hipMemcpyHostToDevice, st));
    std::vector<int32_t> hin(m.ntile), hcol(reorder ? m.ntile : 0);
    if (reorder) {
        NRC(tmp.get(&tcol, m.ntile));
        hipLaunchKernelGGL(k_nf_tile_cols, dim3(blocks_for(m.ntile, kBlock)), dim3(kBlock), 0, st,
                           (const int32_t *)te, m.ntile, (const int32_t *)m.col, (int32_t)m.nnz, tcol);
        NCHK(hipMemcpyAsync(hcol.data(), tcol, sizeof(int32_t) * m.ntile, hipMemcpyDeviceToHost, st));
    }
    NCHK(hipMemcpyAsync(hin.data(), tin, sizeof(int32_t) * m.ntile, hipMemcpyDeviceToHost, st));
    NCHK(hipStreamSynchronize(st));
    std::vector<int32_t> order;
    if (reorder) {
        order = tile_order(hin, hcol, p, {0, m.ts0, m.ts1, m.ntile});
        NCHK(hipMemcpyAsync(tcol, order.data(), sizeof(int32_t) * m.ntile, hipMemcpyHostToDevice, st));
    }
    hipLaunchKernelGGL(k_nf_tile_list, dim3(blocks_for(m.ntile, kBlock)), dim3(kBlock), 0, st, (const int32_t *)te,
                       (const int32_t *)tr, m.ntile, (const int32_t *)tcol, m.tiles);
    NCHK(hipGetLastError());
    std::vector<NfItem> items;
    for (int32_t k = 0; k < m.ntile; k++) {
        if (k == m.ts0) m.is0 = (int32_t)items.size();
        if (k == m.ts1) m.is1 = (int32_t)items.size();
        if (hin[k] < 0) continue;
        if (!items.empty() && items.back().row == hin[k] && items.back().t1 == k) items.back().t1 = k + 1;
        else items.push_back({hin[k], k, k + 1});
    }
    m.nitem = (int32_t)items.size();
    if (m.ts0 >= m.ntile) m.is0 = m.nitem;
    if (m.ts1 >= m.ntile) m.is1 = m.nitem;
    const int64_t nw = p / 32 + 1;
    NRC(alloc(h, &m.items, m.nitem));
    NRC(alloc(h, &m.split, nw));
    hipLaunchKernelGGL(k_nf_zero, dim3(blocks_for(nw, kBlock)), dim3(kBlock), 0, st, m.split, nw);
    if (m.nitem) {
        NCHK(hipMemcpyAsync(m.items, items.data(), sizeof(NfItem) * m.nitem, hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL(k_nf_split_bits, dim3(blocks_for(m.nitem, kBlock)), dim3(kBlock), 0, st,
                           (const NfItem *)m.items, m.nitem, m.split);
    }
    NCHK(hipGetLastError());
    NCHK(hipStreamSynchronize(st));
    *fits = 1;
    return 0;
}

int nf_build(fehip_solver *h, const NfInput &in, int64_t nnz_max, int64_t far_max, NormalMat &m, int *fits) {
    *fits = 0;
    const int rc = build(h, in, nnz_max, far_max, m, fits);
    if (rc || *fits <= 0) nf_free(h, m);
    return rc;
}

int nf_values(const NfInput &in, NormalMat &m, bool projected) {
    for (const NfPair &q : m.pairs) {
        const double *ca = in.cache[q.a], *cb = in.cache[q.b];
        hipLaunchKernelGGL(k_nf_cell_values, dim3(blocks_for(q.ncell, kBlock)), dim3(kBlock), 0, in.stream,
                           (const int32_t *)q.start, q.ncell, (const int32_t *)q.order, ca, cb,
                           (const int32_t *)q.dsta, (const int32_t *)q.dstb, m.val);
        if (q.nbig)
            hipLaunchKernelGGL(k_nf_big_values, dim3((unsigned)q.nbig), dim3(kBlock), 0, in.stream,
                               (const int32_t *)q.big, (const int32_t *)q.start, (const int32_t *)q.order, ca, cb,
                               (const int32_t *)q.dsta, (const int32_t *)q.dstb, m.val);
    }
    if (m.ndiag) {
        const int32_t s0 = in.big0_s, ns = projected ? in.nbig[in.s] : 0;
        hipLaunchKernelGGL(k_nf_diag, dim3(blocks_for(m.ndiag, kBlock)), dim3(kBlock), 0, in.stream, in.big_rows,
                           m.ndiag, s0, s0 + ns, in.big_sum, in.scale, (const int32_t *)m.dpos, m.col, m.val);
        if (ns)
            hipLaunchKernelGGL(k_nf_project_rows, dim3((unsigned)ns), dim3(kBlock), 0, in.stream, in.big_rows + s0,
                               in.big_sum + s0, in.scale, (const int32_t *)m.off, m.col, m.val);
    }
    m.projected = projected;
    NCHK(hipGetLastError());
    return 0;
}

}  // namespace fehip
