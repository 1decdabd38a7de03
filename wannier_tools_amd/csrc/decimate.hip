// Batched Lopez-Sancho decimation on gfx950: the FP32-with-FP64-accumulation
// rounds and the persistent schedules up to order 80, and the FP64 rounds
// beyond order 112 (the FP64 rounds up to there are in mid.hip).
//
// Restates surfgreen_1985 (src/surfgreen.f90:74-134) for many (k, omega)
// instances.  Per iteration:
//
//   g = (z - eps_i)^-1                 blocked Gauss-Jordan in LDS (MFMA updates)
//   [m1 ; m2]     = [alpha ; beta] g   dual GEMM
//   [m1 b ; m2 b] -> eps_s += m1 b ; beta'  = m2 b    (b = beta)
//   [m2 a ; m1 a] -> eps_t += m2 a ; alpha' = m1 a    (a = alpha)
//   stop when sum_ij |alpha'_ij| <= accuracy
//
// the reference's 1 inverse + 6 GEMMs, grouped into three products that each
// stage one shared operand through LDS.  The reference adds both products to
// eps_i as well; since every iteration adds m1 b to eps_s, m2 a to eps_t and
// both to eps_i, starting from H00 for all three, eps_i = eps_s + eps_t - H00
// at every step, and it is formed that way where it is read instead of being
// stored (a third fewer FP64 read-modify-writes per iteration; the sum adds
// two roundings of eps, it does not accumulate them).  R is the working precision of the
// inverse and the GEMMs: double reproduces the reference; float runs them on
// the FP32 MFMA while the eps accumulators, the convergence sum, the three
// final inverses and the traces stay in FP64.
//
// Schedule.  The Gauss-Jordan inverse is a chain of pivot steps run by one
// wave: its time is set by latency, not arithmetic, and it holds the whole
// matrix in LDS (100 KB at order 80).  The GEMMs are arithmetic-bound and
// need only a small LDS stage.  The two halves therefore run as two kernels
// sized to share every CU:
//   gj_round_kernel    one inverse per instance slot      (4 waves, large LDS)
//   gemm_round_kernel  the three dual GEMMs per slot      (8 waves, small LDS)
// Instance slots come in two sets, one per stream; each stream alternates its
// set between the two kernels (a "round" is one launch of each), so one set's
// pivot chains run beside the other set's GEMMs.  A slot keeps its decimation
// state in global memory between rounds and takes the next (k, omega)
// instance from a device counter once its previous one is written out.
#include "wtsurf_device.h"
#include <type_traits>
#include "wtsurf_internal.h"
#include "decimate_common.h"

namespace wtsurf {

template <typename T>
constexpr T cmax(T a, T b) { return a > b ? a : b; }

constexpr int kGjBlock = 256;  // Gauss-Jordan kernel: 4 waves, one per SIMD
// One workgroup of each kernel shares a CU: per SIMD one Gauss-Jordan wave
// (at most 144 VGPRs at order 80) and two GEMM waves of at most 184 VGPRs,
// 144 + 2 x 184 = 512.  amdgpu_num_vgpr counts half the unified register
// file on this target, hence 92.
constexpr int kGemmVgprHalf = 92;

// Slot phases (SlotState::phase); zero-filled state is kEmpty.
enum : int { kEmpty = 0, kLoop = 1, kGemm = 2, kFinal0 = 3, kFinal1 = 4, kFinal2 = 5, kDone = 6 };

// LDS of the Gauss-Jordan kernel: the matrix S (NP x LD, precision R) and the
// panel pivot rows T; the final inverses reuse it in FP64.
template <int Q, typename R>
struct GjLay {
    using C = typename Prec<R>::C;
    static constexpr int NP = 16 * Q, LD = NP + 1;
    static constexpr size_t S = (size_t)NP * LD * sizeof(C);
    static constexpr size_t fin = (size_t)NP * LD * 16 + (size_t)kPanel * NP * 16;
    static constexpr size_t bytes = cmax(S + (size_t)kPanel * NP * sizeof(C), fin);
};

// LDS of the GEMM kernel: one K-chunk of B (rows, padded) and of the two A
// column panels.
template <int Q, typename R>
struct GemmLay {
    using C = typename Prec<R>::C;
    static constexpr int NP = 16 * Q;
    static constexpr size_t B = (size_t)kChunk * (NP + 1) * sizeof(C);
    static constexpr size_t A = (size_t)kChunk * NP * sizeof(C);
    static constexpr size_t bytes = B + 2 * A;
};

// ---------------------------------------------------------------------------
// Blocked Gauss-Jordan inverse in LDS.  The matrix lives as S[col][row]
// (leading dimension NP + 1); columns are eliminated in panels of kPanel with
// partial pivoting on |re|+|im| (the zgetrf rule; ties go to the lowest row).
// Rows are never swapped: step k's pivot is row cm.pivrow[k], and at the end
// X^-1[i][j] = S[cm.pivstep[j]][cm.pivrow[i]].

// Panel elimination by one wave: columns c0 .. c0+kPanel-1 of S, rows
// lane + 64 s (s < NSET, the row sets), held in registers for the whole
// panel (no barrier per step; the pivot search is a DPP wave maximum plus a
// ballot).  Records the pivots in cm.pivrow / cm.pivstep and writes the panel
// back.  Returns true (every lane) on an exactly zero pivot column.
//
// A row that becomes the pivot at step j is kept unscaled for the rest of the
// panel: it holds u with u[j] = 1 and stands for r_j u (r_j = 1 / pivot).
// Every later step acts on it linearly (its multiplier u[j'] r' is r_j^-1
// times the scaled row's), so the panel runs the same update on every row
// and scales each of its pivot rows by r_j once, at the write-back.
template <int Q, typename R>
__device__ __forceinline__ bool gj_panel(typename Prec<R>::C (*S)[16 * Q + 1], Common<Q> &cm,
                                         int c0, int n, int lane) {
    using P = Prec<R>;
    using C = typename P::C;
    constexpr int NP = 16 * Q;
    constexpr int NSET = (NP + 63) / 64;
    C a[NSET][kPanel];
    bool has[NSET], fr[NSET];
    int live[NSET];  // row set s holds rows of the matrix at all (uniform)
#pragma unroll
    for (int s = 0; s < NSET; ++s) {
        const int r = lane + 64 * s;
        live[s] = s == 0 ? 1 : uniform(64 * s < n ? 1 : 0);
        has[s] = r < n;
#pragma unroll
        for (int j = 0; j < kPanel; ++j) {
            a[s][j].x = a[s][j].y = 0;
            if (has[s]) a[s][j] = S[c0 + j][r];
        }
        fr[s] = has[s] && cm.pivstep[has[s] ? r : 0] < 0;
    }
    bool sing = false;
#pragma unroll
    for (int j = 0; j < kPanel; ++j) {
        const int c = c0 + j;
        if (c >= n) break;
        double v[NSET];
        double vmax = -1.0;
#pragma unroll
        for (int s = 0; s < NSET; ++s) {
            v[s] = fr[s] ? (double)(fabs(a[s][j].x) + fabs(a[s][j].y)) : -1.0;
            vmax = s == 0 ? v[0] : fmax_nocanon(vmax, v[s]);
        }
        const double best = wave_max_f64(vmax);
        if (!(best > 0.0)) {  // zero (or NaN) pivot column: singular
            sing = true;
            break;
        }
        // lowest row attaining the maximum: set 0 before set 1 before ...
        int slot = NSET, pl = 0;
#pragma unroll
        for (int s = NSET - 1; s >= 0; --s) {
            const unsigned long long m = __ballot(v[s] == best);
            if (m) {
                slot = s;
                pl = __ffsll((long long)m) - 1;
            }
        }
        slot = uniform(slot);
        pl = uniform(pl);
        const int p = pl + 64 * slot;
        // pivot row from lane pl of row set `slot`
        C row[kPanel];
#pragma unroll
        for (int s = 0; s < NSET; ++s)
            if (slot == s) {
#pragma unroll
                for (int jj = 0; jj < kPanel; ++jj) {
                    row[jj].x = P::readlane(a[s][jj].x, pl);
                    row[jj].y = P::readlane(a[s][jj].y, pl);
                }
            }
        const C r = crecip_fast(row[j]);
        // eliminate column c from every other row with the multiplier
        // m = f r (f = a[j]):  a[jj] -= m row[jj] for jj != j, a[j] = -m.
        // The pivot row takes m = 0 and a[j] = 1.
#pragma unroll
        for (int s = 0; s < NSET; ++s) {
            if (!live[s]) continue;
            const bool isp = slot == s && lane == pl;
            C m = cmul(a[s][j], r);
            if (isp) m.x = m.y = 0;
#pragma unroll
            for (int jj = 0; jj < kPanel; ++jj) {
                if (jj == j) {
                    a[s][jj].x = isp ? (R)1 : -m.x;
                    a[s][jj].y = -m.y;
                } else {
                    a[s][jj].x = fma(-m.x, row[jj].x, fma(m.y, row[jj].y, a[s][jj].x));
                    a[s][jj].y = fma(-m.x, row[jj].y, fma(-m.y, row[jj].x, a[s][jj].y));
                }
            }
            fr[s] = fr[s] && !isp;
        }
        if (lane == 0) {
            cm.pivrow[c] = p;
            cm.pivstep[p] = c;
            cm.rpiv[c] = make_double2(r.x, r.y);
        }
    }
#pragma unroll
    for (int s = 0; s < NSET; ++s)
        if (has[s]) {
            const int r = lane + 64 * s;
            const int ps = cm.pivstep[r];
            if (ps >= c0 && ps < c0 + kPanel) {  // pivot row of this panel: scale by r_j
                const double2 rp = cm.rpiv[ps];
                C rr;
                rr.x = (R)rp.x;
                rr.y = (R)rp.y;
#pragma unroll
                for (int j = 0; j < kPanel; ++j) a[s][j] = cmul(a[s][j], rr);
            }
#pragma unroll
            for (int j = 0; j < kPanel; ++j) S[c0 + j][r] = a[s][j];
        }
    return sing;
}

// T[j][col] = row pivrow[c0 + j] of S outside the panel columns (zero in the
// panel columns and for steps past the last column), by NT threads.
template <int Q, typename R, int NT>
__device__ __forceinline__ void gj_gather_t(typename Prec<R>::C (*S)[16 * Q + 1],
                                            typename Prec<R>::C (*T)[16 * Q], Common<Q> &cm,
                                            int c0, int n, int tid) {
    using C = typename Prec<R>::C;
    constexpr int NP = 16 * Q;
    for (int e = tid; e < kPanel * NP; e += NT) {
        const int j = e / NP, col = e % NP;
        C tv;
        tv.x = 0;
        tv.y = 0;
        if (c0 + j < n && (col < c0 || col >= c0 + kPanel)) tv = S[col][cm.pivrow[c0 + j]];
        T[j][col] = tv;
    }
}

// Rank-kPanel MFMA update of tile (ti, tj) of S for panel c0, outside the
// panel columns:  S[:, ~C] = S0[:, ~C] + S[:, C] T, where rows pivoted in
// this panel start from zero (S0 = 0) since their old content is now in T.
template <int Q, typename R>
__device__ __forceinline__ void gj_update_tile(typename Prec<R>::C (*S)[16 * Q + 1],
                                               typename Prec<R>::C (*T)[16 * Q],
                                               const Common<Q> &cm, int ti, int tj, int c0,
                                               int lr, int lq) {
    using P = Prec<R>;
    using C = typename P::C;
    typename P::V4 accR = {0, 0, 0, 0}, accI = {0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < kPanel / 4; ++ks) {
        const C a = S[c0 + 4 * ks + lq][16 * ti + lr];
        const C b = T[4 * ks + lq][16 * tj + lr];
        accR = P::mfma(a.x, b.x, accR);
        accR = P::mfma(-a.y, b.y, accR);
        accI = P::mfma(a.x, b.y, accI);
        accI = P::mfma(a.y, b.x, accI);
    }
    const int col = 16 * tj + lr;
    if (col < c0 || col >= c0 + kPanel) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int row = 16 * ti + P::out_row(lq, v);
            const int ps = cm.pivstep[row];
            const bool pivot_here = ps >= c0 && ps < c0 + kPanel;
            C o = S[col][row];
            if (pivot_here) o.x = o.y = 0;
            o.x += accR[v];
            o.y += accI[v];
            S[col][row] = o;
        }
    }
}

// Rank-2kPanel MFMA update of tile (ti, tj) of S for the panel pair p (columns
// c0 .. c0+kPanel-1) and q (the next kPanel), applied at once (orders beyond
// 80, whose S lives in global memory: one read-modify-write of the matrix
// per pair instead of per panel).  T holds p's pivot rows in rows 0..kPanel-1
// and q's, taken after p's update, in rows kPanel..2kPanel-1; Mp holds p's
// columns of S as they were before q's update.  Per element, in the order the
// two single-panel updates would give it:
//   rows pivoted in q:  M_q T_q (their old content is in T_q, p's term drops),
//   rows pivoted in p:  M_p T_p + M_q T_q, except that in p's own columns they
//                       keep their content (the p term is zero there),
//   other rows:         S + M_p T_p + M_q T_q;
// q's columns are left as q's elimination left them.
// A tile's global-memory operands for gj_tile2_finish: q's columns of S in the
// tile's rows (the MFMA A operand) and the tile's old values.
template <typename C>
struct Tile2Ops {
    C aq[kPanel / 4];
    C old[4];
};

template <int Q, typename R>
__device__ __forceinline__ void gj_tile2_load(typename Prec<R>::C (*S)[16 * Q + 1], int ti, int tj,
                                              int c1, int lr, int lq,
                                              Tile2Ops<typename Prec<R>::C> &o) {
#pragma unroll
    for (int ks = 0; ks < kPanel / 4; ++ks) o.aq[ks] = S[c1 + 4 * ks + lq][16 * ti + lr];
    const int col = 16 * tj + lr;
#pragma unroll
    for (int v = 0; v < 4; ++v) o.old[v] = S[col][16 * ti + Prec<R>::out_row(lq, v)];
}

template <int Q, typename R>
__device__ __forceinline__ void gj_tile2_finish(typename Prec<R>::C (*S)[16 * Q + 1],
                                                typename Prec<R>::C (*T)[16 * Q],
                                                typename Prec<R>::C (*Mp)[16 * Q],
                                                const Common<Q> &cm, int ti, int tj, int c0,
                                                int lr, int lq,
                                                const Tile2Ops<typename Prec<R>::C> &o) {
    using P = Prec<R>;
    using C = typename P::C;
    const int c1 = c0 + kPanel;
    typename P::V4 accR = {0, 0, 0, 0}, accI = {0, 0, 0, 0};
    const int arow = 16 * ti + lr;
    const int aps = cm.pivstep[arow];
    const bool drop_p = aps >= c1 && aps < c1 + kPanel;  // pivoted in q
#pragma unroll
    for (int ks = 0; ks < kPanel / 4; ++ks) {
        C a = Mp[4 * ks + lq][arow];
        if (drop_p) a.x = a.y = 0;
        const C b = T[4 * ks + lq][16 * tj + lr];
        accR = P::mfma(a.x, b.x, accR);
        accR = P::mfma(-a.y, b.y, accR);
        accI = P::mfma(a.x, b.y, accI);
        accI = P::mfma(a.y, b.x, accI);
    }
#pragma unroll
    for (int ks = 0; ks < kPanel / 4; ++ks) {
        const C a = o.aq[ks];
        const C b = T[kPanel + 4 * ks + lq][16 * tj + lr];
        accR = P::mfma(a.x, b.x, accR);
        accR = P::mfma(-a.y, b.y, accR);
        accI = P::mfma(a.x, b.y, accI);
        accI = P::mfma(a.y, b.x, accI);
    }
    const int col = 16 * tj + lr;
    if (col < c1 || col >= c1 + kPanel) {
        const bool pcol = col >= c0 && col < c1;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int row = 16 * ti + P::out_row(lq, v);
            const int ps = cm.pivstep[row];
            const bool zero = (ps >= c1 && ps < c1 + kPanel) || (!pcol && ps >= c0 && ps < c1);
            C x = o.old[v];
            if (zero) x.x = x.y = 0;
            x.x += accR[v];
            x.y += accI[v];
            S[col][row] = x;
        }
    }
}

// Rank-2kPanel MFMA update for the panel pair p (columns c0 .. c0+kPanel-1)
// and q (the next kPanel), applied at once to the tiles t = first, first +
// stride, ... < Q*Q (t = tj Q + ti) other than those in tile column skip_tj
// (orders beyond 80, whose S lives in global memory: one read-modify-write of
// the matrix per pair instead of per panel).  T holds p's pivot rows in rows
// 0..kPanel-1 and q's, taken after p's update, in rows kPanel..2kPanel-1; Mp
// holds p's columns of S as they were before q's update.  Per element, in the
// order the two single-panel updates would give it:
//   rows pivoted in q:  M_q T_q (their old content is in T_q, p's term drops),
//   rows pivoted in p:  M_p T_p + M_q T_q, except that in p's own columns they
//                       keep their content (the p term is zero there),
//   other rows:         S + M_p T_p + M_q T_q;
// q's columns are left as q's elimination left them.  Each tile's global
// loads are issued before the previous tile is finished, so the memory
// latency of a wave's tiles overlaps the MFMAs and stores of the tile before.
template <int Q, typename R>
__device__ __forceinline__ void gj_update_tiles2(typename Prec<R>::C (*S)[16 * Q + 1],
                                                 typename Prec<R>::C (*T)[16 * Q],
                                                 typename Prec<R>::C (*Mp)[16 * Q],
                                                 const Common<Q> &cm, int first, int stride,
                                                 int skip_tj, int c0, int lr, int lq) {
    using C = typename Prec<R>::C;
    auto next = [&](int t) {
        while (t < Q * Q && t / Q == skip_tj) t += stride;
        return t;
    };
    int t = next(first);
    if (t >= Q * Q) return;
    Tile2Ops<C> cur, nxt;
    gj_tile2_load<Q, R>(S, t % Q, t / Q, c0 + kPanel, lr, lq, cur);
    for (;;) {
        const int tn = next(t + stride);
        if (tn < Q * Q) gj_tile2_load<Q, R>(S, tn % Q, tn / Q, c0 + kPanel, lr, lq, nxt);
        gj_tile2_finish<Q, R>(S, T, Mp, cm, t % Q, t / Q, c0, lr, lq, cur);
        if (tn >= Q * Q) break;
        cur = nxt;
        t = tn;
    }
}

// Panel quads (orders 16 * kQuadMinQ to 16 * kQuadMaxQ, S in global memory): the block
// of four panels p0..p3 (32 columns, two tile columns, starting on a multiple
// of 32) is eliminated panel by panel on its own columns, and the rest of the
// matrix then takes one rank-32 update, one read-modify-write of S per 32
// columns instead of per 16.  For a column j outside the block and a row r,
// the four single-panel updates compose to
//   S'[r][j] = [r not pivoted in the block] S[r][j]
//              + sum_k [r not pivoted in p(k+1)..p3] M_k[r] T_k[j],
// M_k the columns of p_k right after its elimination (copied to global memory,
// since later panels change them in place) and T_k the pivot rows of p_k with
// the updates of p0..p(k-1) applied:
//   T_k[j] = S[pivrow_k][j] + sum_{l<k} M_l[pivrow_k] T_l[j].
// Inside the block every panel's update is applied at once to the block's
// other columns (two tile columns, all rows), as the single-panel steps do.
constexpr int kQuadMaxQ = 18;  // T of a quad (32 rows of 16 Q) fits in LDS up to here
// Below order 192 the pairs are as fast or faster (measured: -3% at 108, -9% at
// 144, -2% at 160; +4% at 192, +5% at 216, +7% at 240, +12% at 288): the
// quad's three panels eliminated inside the block add more chain than its
// smaller traffic saves.
constexpr int kQuadMinQ = 12;
template <int Q>
constexpr bool use_quads() { return Q >= kQuadMinQ && Q <= kQuadMaxQ; }

// The global-memory operands of one outside tile for gj_quad_finish: the
// block's M columns in the tile's rows (MFMA A operand, rank 32) and the
// tile's old values.
template <typename C>
struct QuadOps {
    C a[4 * kPanel / 4];
    C old[4];
};

template <int Q, typename R>
__device__ __forceinline__ void gj_quad_load(typename Prec<R>::C (*S)[16 * Q + 1],
                                             const typename Prec<R>::C *__restrict__ Mg,
                                             const Common<Q> &cm, int ti, int tj, int c0,
                                             int nin, int lr, int lq,
                                             QuadOps<typename Prec<R>::C> &o) {
    constexpr int NP = 16 * Q;
    const int arow = 16 * ti + lr;
    const int aps = cm.pivstep[arow];
    // panel of the block in which row arow was the pivot (-1: none)
    const int kr = (aps >= c0 && aps < c0 + nin * kPanel) ? (aps - c0) / kPanel : -1;
#pragma unroll
    for (int q = 0; q < kPanel; ++q) {  // k index 4 q + lq of the rank-32 product
        const int l = q / 2;             // panel of that k index
        typename Prec<R>::C a;
        a.x = 0;
        a.y = 0;
        if (l < nin && kr <= l) a = Mg[(size_t)(4 * q + lq) * NP + arow];
        o.a[q] = a;
    }
    const int col = 16 * tj + lr;
#pragma unroll
    for (int v = 0; v < 4; ++v) o.old[v] = S[col][16 * ti + Prec<R>::out_row(lq, v)];
}

template <int Q, typename R>
__device__ __forceinline__ void gj_quad_finish(typename Prec<R>::C (*S)[16 * Q + 1],
                                               typename Prec<R>::C (*T)[16 * Q],
                                               const Common<Q> &cm, int ti, int tj, int c0,
                                               int nin, int lr, int lq,
                                               const QuadOps<typename Prec<R>::C> &o) {
    using P = Prec<R>;
    using C = typename P::C;
    typename P::V4 accR = {0, 0, 0, 0}, accI = {0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < kPanel; ++q) {
        if (q / 2 >= nin) break;
        const C a = o.a[q];
        const C b = T[4 * q + lq][16 * tj + lr];
        accR = P::mfma(a.x, b.x, accR);
        accR = P::mfma(-a.y, b.y, accR);
        accI = P::mfma(a.x, b.y, accI);
        accI = P::mfma(a.y, b.x, accI);
    }
    const int col = 16 * tj + lr;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int row = 16 * ti + P::out_row(lq, v);
        const int ps = cm.pivstep[row];
        C x = o.old[v];
        if (ps >= c0 && ps < c0 + nin * kPanel) x.x = x.y = 0;
        x.x += accR[v];
        x.y += accI[v];
        S[col][row] = x;
    }
}

// The rank-32 update of everything outside the block's tile columns [tb, tb
// + ntb) and tile column skip_tj, by tile-row halves: item = 2 ti + h, items
// first, first + stride, ...  The A operand of a tile row (the block's M
// columns in its 16 rows) is loaded once per item and serves all its tiles;
// each tile's old values are loaded before the previous tile is finished.
template <int Q, typename R>
__device__ __forceinline__ void gj_quad_rows(typename Prec<R>::C (*S)[16 * Q + 1],
                                             typename Prec<R>::C (*T)[16 * Q],
                                             const typename Prec<R>::C *__restrict__ Mg,
                                             const Common<Q> &cm, int first, int stride,
                                             int tb, int ntb, int skip_tj, int c0, int nin,
                                             int lr, int lq) {
    using C = typename Prec<R>::C;
    constexpr int HALF = (Q + 1) / 2;
    auto outside = [&](int tj) { return !(tj >= tb && tj < tb + ntb) && tj != skip_tj; };
#pragma unroll 1
    for (int item = first; item < 2 * Q; item += stride) {
        const int ti = item >> 1, h = item & 1;
        const int tj1 = h ? Q : HALF;
        int tj = h ? HALF : 0;
        while (tj < tj1 && !outside(tj)) ++tj;
        if (tj >= tj1) continue;
        QuadOps<C> cur, nxt;
        gj_quad_load<Q, R>(S, Mg, cm, ti, tj, c0, nin, lr, lq, cur);
        for (;;) {
            int tn = tj + 1;
            while (tn < tj1 && !outside(tn)) ++tn;
            if (tn < tj1) {
                // the same tile row: only the old values are new
                const int col = 16 * tn + lr;
#pragma unroll
                for (int v = 0; v < 4; ++v) nxt.old[v] = S[col][16 * ti + Prec<R>::out_row(lq, v)];
            }
            gj_quad_finish<Q, R>(S, T, cm, ti, tj, c0, nin, lr, lq, cur);
            if (tn >= tj1) break;
#pragma unroll
            for (int v = 0; v < 4; ++v) cur.old[v] = nxt.old[v];
            tj = tn;
        }
    }
}

// The elimination of panels 1..npanel-1 by quads (panel 0 already
// eliminated), NT threads; T is 4 kPanel rows of NP in LDS, Mg 4 kPanel
// columns of NP in global memory.
template <int Q, typename R, int NT>
__device__ __forceinline__ void gj_quads(typename Prec<R>::C (*S)[16 * Q + 1],
                                         typename Prec<R>::C (*T)[16 * Q],
                                         typename Prec<R>::C *__restrict__ Mg, Common<Q> &cm,
                                         int n, int npanel, int wave, int lane) {
    using C = typename Prec<R>::C;
    constexpr int NP = 16 * Q;
    constexpr int NWAVES = NT / kWave;
    const int tid = threadIdx.x;
    const int lr = lane & 15, lq = lane >> 4;
    for (int qb = 0; qb < npanel; qb += 4) {
        const int c0 = qb * kPanel;  // a multiple of 32
        const int nin = uniform(npanel - qb < 4 ? npanel - qb : 4);
        const int tb = c0 / 16, ntb = uniform(Q - tb < 2 ? Q - tb : 2);
        bool sing = false;
        for (int k = 0; k < nin; ++k) {
            const int ck = c0 + k * kPanel;
            // panel k is eliminated: panel 0 before the block, panel k > 0
            // under the block update of panel k - 1
            if (uniform(cm.sing)) {
                sing = true;
                break;
            }
            // M_k, and T_k: p_k's pivot rows outside its columns, with the
            // block's earlier panels applied outside the block
            for (int e = tid; e < kPanel * NP; e += NT) {
                const int j = e / NP, r = e % NP;
                Mg[(size_t)(kPanel * k + j) * NP + r] = S[ck + j][r];
            }
            for (int e = tid; e < kPanel * NP; e += NT) {
                const int jj = e / NP, col = e % NP;
                C tv;
                tv.x = 0;
                tv.y = 0;
                if (ck + jj < n && (col < ck || col >= ck + kPanel)) {
                    const int r = cm.pivrow[ck + jj];
                    tv = S[col][r];
                    if (col < c0 || col >= c0 + 4 * kPanel)
                        for (int l = 0; l < k; ++l)
#pragma unroll
                            for (int j = 0; j < kPanel; ++j) {
                                const C m = Mg[(size_t)(kPanel * l + j) * NP + r];
                                const C t = T[kPanel * l + j][col];
                                tv.x += m.x * t.x - m.y * t.y;
                                tv.y += m.x * t.y + m.y * t.x;
                            }
                }
                T[kPanel * k + jj][col] = tv;
            }
            __syncthreads();
            // p_k's update on the block's other columns, all rows: first the
            // tile column of panel k + 1, which wave 0 then eliminates while
            // the other waves update the block's other tile column
            if (k + 1 < nin) {
                const int tk = (ck + kPanel) / 16;
#pragma unroll 1
                for (int ti = wave; ti < Q; ti += NWAVES)
                    gj_update_tile<Q, R>(S, T + kPanel * k, cm, ti, tk, ck, lr, lq);
                __syncthreads();
                if (wave == 0) {
                    const bool s1 = gj_panel<Q, R>(S, cm, ck + kPanel, n, lane);
                    if (lane == 0 && s1) cm.sing = 1;
                } else {
#pragma unroll 1
                    for (int t = wave - 1; t < Q * ntb; t += NWAVES - 1)
                        if (tb + t / Q != tk)
                            gj_update_tile<Q, R>(S, T + kPanel * k, cm, t % Q, tb + t / Q, ck, lr, lq);
                }
            } else {
#pragma unroll 1
                for (int t = wave; t < Q * ntb; t += NWAVES)
                    gj_update_tile<Q, R>(S, T + kPanel * k, cm, t % Q, tb + t / Q, ck, lr, lq);
            }
            __syncthreads();
        }
        if (sing) break;
        // the rank-32 update of everything outside the block: first the tile
        // column of the next quad's first panel, which wave 0 then eliminates
        // while the other waves update the rest
        const bool ahead = qb + 4 < npanel;
        const int tn = tb + 2;
        if (ahead) {
            for (int ti = wave; ti < Q; ti += NWAVES) {
                QuadOps<C> ops;
                gj_quad_load<Q, R>(S, Mg, cm, ti, tn, c0, nin, lr, lq, ops);
                gj_quad_finish<Q, R>(S, T, cm, ti, tn, c0, nin, lr, lq, ops);
            }
            __syncthreads();
        }
        if (ahead && wave == 0) {
            const bool s1 = gj_panel<Q, R>(S, cm, c0 + 4 * kPanel, n, lane);
            if (lane == 0 && s1) cm.sing = 1;
        } else {
            const int first = ahead ? 1 : 0, nw = ahead ? NWAVES - 1 : NWAVES;
            gj_quad_rows<Q, R>(S, T, Mg, cm, wave - first, nw, tb, ntb, ahead ? tn : -1, c0, nin,
                               lr, lq);
        }
        __syncthreads();
    }
}

// Inverse of X = z*1 - E (the first n x n block of the padded FP64 matrix E,
// or of E + E2 - H when E2 is given) in precision R, by NT threads.  X is
// held in sbuf (NP x (NP+1), LDS for orders up to 80, the slot's global
// workspace beyond), the panel pivot rows T in tbuf (LDS).
//
// Schedule with one panel of lookahead: after panel p is eliminated and its
// pivot rows gathered into T, all waves apply p's update to the tile column
// that holds panel p+1; then wave 0 eliminates panel p+1 while the other
// waves apply p's update to every other tile column.  Panel p+1's pivot rows
// are gathered into T only after the barrier that ends p's update.
//
// out_mode 1: the diagonal of X^-1 into cm.diag (FP64).
// out_mode 2: the diagonal and the unpadded n x n X^-1 into `full` (FP64).
// out_mode 4: X^-1 padded to NP x NP (pad zero), column-major, precision R,
//             into `gout`.
// Returns true if an exactly zero pivot was met; the result is then the
// identity, as the reference's inv hands back (zgesv skips the solve on a
// zero pivot and inv copies back the identity right-hand side,
// src/inverse.f90:44-55).
template <int Q, typename R, int NT>
__device__ __forceinline__ bool gj_inverse(unsigned char *sbuf, unsigned char *tbuf, Common<Q> &cm,
                                           const double2 *__restrict__ E,
                                           const double2 *__restrict__ E2,
                                           const double2 *__restrict__ H, double2 z, int n,
                                           int out_mode, double2 *__restrict__ full,
                                           typename Prec<R>::C *__restrict__ gout,
                                           typename Prec<R>::C *__restrict__ mg = nullptr) {
    using P = Prec<R>;
    using C = typename P::C;
    constexpr int NP = 16 * Q;
    constexpr int LD = NP + 1;
    constexpr int NWAVES = NT / kWave;
    static_assert(NP <= 384, "the panel wave holds at most six rows per lane");
    static_assert(NWAVES >= 2, "the lookahead needs a panel wave and update waves");
    const int tid = threadIdx.x;
    const int wave = uniform(tid >> 6), lane = tid & 63;
    const int lr = lane & 15, lq = lane >> 4;
    C(*S)[LD] = reinterpret_cast<C(*)[LD]>(sbuf);
    C(*T)[NP] = reinterpret_cast<C(*)[NP]>(tbuf);

    // Load in batches of kLoadBatch elements per thread, every global load of
    // a batch issued before its first LDS store: S is reached through a
    // generic pointer, so the compiler would otherwise keep each load behind
    // the previous store and pay one memory round trip per element.
    constexpr int kIter = (NP * NP + NT - 1) / NT;
    constexpr int kLoadBatch = 5;
    for (int it0 = 0; it0 < kIter; it0 += kLoadBatch) {
        double2 xv[kLoadBatch];
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u) {
            const int e = tid + (it0 + u) * NT;
            const int i = e % NP, j = e / NP;
            xv[u] = make_double2(0.0, 0.0);
            if (it0 + u < kIter && e < NP * NP && i < n && j < n) {
                double2 x = E[i + j * NP];
                if (E2) {
                    const double2 y = E2[i + j * NP], h = H[i + j * NP];
                    x.x = (x.x + y.x) - h.x;
                    x.y = (x.y + y.y) - h.y;
                }
                xv[u] = x;
            }
        }
#pragma unroll
        for (int u = 0; u < kLoadBatch; ++u) {
            const int e = tid + (it0 + u) * NT;
            const int i = e % NP, j = e / NP;
            if (it0 + u < kIter && e < NP * NP) {
                C v;
                v.x = 0;
                v.y = 0;
                if (i < n && j < n) {
                    v.x = (R)((i == j ? z.x : 0.0) - xv[u].x);
                    v.y = (R)((i == j ? z.y : 0.0) - xv[u].y);
                }
                S[j][i] = v;
            }
        }
    }
    for (int i = tid; i < NP; i += NT) cm.pivstep[i] = -1;
    if (tid == 0) cm.sing = 0;
    __syncthreads();

    const int npanel = (n + kPanel - 1) / kPanel;
    if (wave == 0) {
        const bool sing = gj_panel<Q, R>(S, cm, 0, n, lane);
        if (lane == 0 && sing) cm.sing = 1;
    }
    __syncthreads();
    if constexpr (use_quads<Q>()) {
        gj_quads<Q, R, NT>(S, T, mg, cm, n, npanel, wave, lane);
    } else if constexpr (Q > 5) {
        // S in global memory: panels in pairs, one rank-2kPanel update each
        C(*Mp)[NP] = reinterpret_cast<C(*)[NP]>(tbuf + 2 * kPanel * NP * sizeof(C));
        for (int pb = 0; pb < npanel; pb += 2) {
            if (uniform(cm.sing)) break;
            const int c0 = pb * kPanel, c1 = c0 + kPanel;
            gj_gather_t<Q, R, NT>(S, T, cm, c0, n, tid);
            if (pb + 1 >= npanel) {  // a last panel of its own
                __syncthreads();
#pragma unroll 1
                for (int t = wave; t < Q * Q; t += NWAVES)
                    gj_update_tile<Q, R>(S, T, cm, t % Q, t / Q, c0, lr, lq);
                __syncthreads();
                break;
            }
            for (int e = tid; e < kPanel * NP; e += NT) Mp[e / NP][e % NP] = S[c0 + e / NP][e % NP];
            __syncthreads();
            // q's columns (tile column c0 / 16, outside p's) updated with p,
            // then q eliminated
            const int tp = c0 / 16;
#pragma unroll 1
            for (int ti = wave; ti < Q; ti += NWAVES) gj_update_tile<Q, R>(S, T, cm, ti, tp, c0, lr, lq);
            __syncthreads();
            if (wave == 0) {
                const bool sing = gj_panel<Q, R>(S, cm, c1, n, lane);
                if (lane == 0 && sing) cm.sing = 1;
            }
            __syncthreads();
            if (uniform(cm.sing)) break;
            // q's pivot rows after p's update, outside q's columns
            for (int e = tid; e < kPanel * NP; e += NT) {
                const int k = e / NP, col = e % NP;
                C tv;
                tv.x = 0;
                tv.y = 0;
                if (c1 + k < n && (col < c1 || col >= c1 + kPanel)) {
                    const int r = cm.pivrow[c1 + k];
                    tv = S[col][r];
                    if (col < c0 || col >= c1)
#pragma unroll
                        for (int j = 0; j < kPanel; ++j) {
                            const C m = Mp[j][r], t = T[j][col];
                            tv.x += m.x * t.x - m.y * t.y;
                            tv.y += m.x * t.y + m.y * t.x;
                        }
                }
                T[kPanel + k][col] = tv;
            }
            __syncthreads();
            // the pair's update: first the tile column of the next pair, which
            // wave 0 then eliminates while the other waves update the rest
            const bool ahead = pb + 2 < npanel;
            const int tn = tp + 1;
            if (ahead) {
                // tiles ti = wave, wave + NWAVES, ... of tile column tn
                for (int ti = wave; ti < Q; ti += NWAVES) {
                    Tile2Ops<C> ops;
                    gj_tile2_load<Q, R>(S, ti, tn, c1, lr, lq, ops);
                    gj_tile2_finish<Q, R>(S, T, Mp, cm, ti, tn, c0, lr, lq, ops);
                }
                __syncthreads();
            }
            if (ahead && wave == 0) {
                const bool sing = gj_panel<Q, R>(S, cm, c1 + kPanel, n, lane);
                if (lane == 0 && sing) cm.sing = 1;
            } else {
                const int first = ahead ? 1 : 0, nw = ahead ? NWAVES - 1 : NWAVES;
                gj_update_tiles2<Q, R>(S, T, Mp, cm, wave - first, nw, ahead ? tn : -1, c0, lr, lq);
            }
            __syncthreads();
        }
    } else
    for (int pb = 0; pb < npanel; ++pb) {
        if (uniform(cm.sing)) break;
        const int c0 = pb * kPanel;
        gj_gather_t<Q, R, NT>(S, T, cm, c0, n, tid);
        __syncthreads();
        const bool ahead = pb + 1 < npanel;
        const int tn = (c0 + kPanel) / 16;  // tile column of panel pb + 1
        if (ahead) {
            // the Q tiles of column tn first, shared by all waves
#pragma unroll 1
            for (int ti = wave; ti < Q; ti += NWAVES) gj_update_tile<Q, R>(S, T, cm, ti, tn, c0, lr, lq);
            __syncthreads();
        }
        if (ahead && wave == 0) {
            const bool sing = gj_panel<Q, R>(S, cm, c0 + kPanel, n, lane);
            if (lane == 0 && sing) cm.sing = 1;
        } else {
            // tiles t = tj*Q + ti outside column tn (all of them after the last
            // panel), dealt round-robin over the update waves
            const int first = ahead ? 1 : 0, nw = ahead ? NWAVES - 1 : NWAVES;
#pragma unroll 1
            for (int t = wave - first; t < Q * Q; t += nw) {
                const int ti = t % Q, tj = t / Q;
                if (ahead && tj == tn) continue;
                gj_update_tile<Q, R>(S, T, cm, ti, tj, c0, lr, lq);
            }
        }
        __syncthreads();
    }

    const bool singular = uniform(cm.sing) != 0;
    if (out_mode == 4) {
        for (int e = tid; e < NP * NP; e += NT) {
            const int i = e % NP, j = e / NP;
            C v;
            v.x = 0;
            v.y = 0;
            if (i < n && j < n) {
                if (singular)
                    v.x = (i == j) ? 1 : 0;
                else
                    v = S[cm.pivstep[j]][cm.pivrow[i]];
            }
            gout[e] = v;
        }
    } else {
        for (int i = tid; i < n; i += NT) {
            const C v = singular ? C{1, 0} : S[cm.pivstep[i]][cm.pivrow[i]];
            cm.diag[i] = make_double2(v.x, v.y);
        }
        if (out_mode == 2)
            for (int e = tid; e < n * n; e += NT) {
                const int i = e % n, j = e / n;
                C v;
                if (singular) {
                    v.x = (i == j) ? 1 : 0;
                    v.y = 0;
                } else {
                    v = S[cm.pivstep[j]][cm.pivrow[i]];
                }
                full[i + j * n] = make_double2(v.x, v.y);
            }
    }
    __syncthreads();
    return singular;
}

// Element (i, j) of the FP64 inverse that the last gj_inverse left in sbuf
// (valid until the next gj_inverse on that buffer).
template <int Q>
__device__ __forceinline__ double2 gj_inverse_at(const unsigned char *sbuf, const Common<Q> &cm,
                                                 int i, int j) {
    constexpr int LD = 16 * Q + 1;
    if (cm.sing) return make_double2(i == j ? 1.0 : 0.0, 0.0);
    const double2(*S)[LD] = reinterpret_cast<const double2(*)[LD]>(sbuf);
    return S[cm.pivstep[j]][cm.pivrow[i]];
}

// Element access to the FP64 inverse the LDS Gauss-Jordan left in sbuf.
template <int Q>
struct LdsInverse {
    const unsigned char *sbuf;
    const Common<Q> &cm;
    __device__ double2 operator()(int i, int j) const { return gj_inverse_at(sbuf, cm, i, j); }
};



// ---------------------------------------------------------------------------
// One complex 16x16x4 MFMA step on (re, im) fragments:
//   accR += a.x b.x - a.y b.y,   accI += a.x b.y + a.y b.x
// nby = -b.y is passed in so that tiles sharing b negate it once.
template <typename R>
__device__ __forceinline__ void cmfma(typename Prec<R>::V4 &accR, typename Prec<R>::V4 &accI,
                                      typename Prec<R>::C a, typename Prec<R>::C b, R nby) {
    using P = Prec<R>;
    accR = P::mfma(a.x, b.x, accR);
    accR = P::mfma(a.y, nby, accR);
    accI = P::mfma(a.x, b.y, accI);
    accI = P::mfma(a.y, b.x, accI);
}

// Write-back of one output tile (lane layout of the MFMA accumulator) to O,
// adding sum |P_ij| (FP64) to asum when SUM.
template <int Q, typename R, bool SUM>
__device__ __forceinline__ void store_tile(int ti, int tj, int lr, int lq,
                                           const typename Prec<R>::V4 &accR,
                                           const typename Prec<R>::V4 &accI,
                                           typename Prec<R>::C *O, double &asum) {
    using P = Prec<R>;
    using C = typename P::C;
    constexpr int NP = 16 * Q;
    const int col = 16 * tj + lr;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int idx = 16 * ti + P::out_row(lq, v) + col * NP;
        C val;
        val.x = accR[v];
        val.y = accI[v];
        O[idx] = val;
        if (SUM) asum += hypot((double)val.x, (double)val.y);
    }
}

// One FP64 accumulator tile, read ahead of its update.
struct ETile {
    double2 e[4];
};

template <int Q, typename R>
__device__ __forceinline__ void load_etile(ETile &t, int ti, int tj, int lr, int lq,
                                           const double2 *__restrict__ E) {
    constexpr int NP = 16 * Q;
    const int col = 16 * tj + lr;
#pragma unroll
    for (int v = 0; v < 4; ++v) t.e[v] = E[16 * ti + Prec<R>::out_row(lq, v) + col * NP];
}

template <int Q, typename R>
__device__ __forceinline__ void add_etile(const ETile &t, int ti, int tj, int lr, int lq,
                                          const typename Prec<R>::V4 &accR,
                                          const typename Prec<R>::V4 &accI,
                                          double2 *__restrict__ E) {
    constexpr int NP = 16 * Q;
    const int col = 16 * tj + lr;
#pragma unroll
    for (int v = 0; v < 4; ++v)
        E[16 * ti + Prec<R>::out_row(lq, v) + col * NP] =
            cadd(t.e[v], make_double2(accR[v], accI[v]));
}

// E += P over this wave's product-0 tiles (pairs s < PPW, then the single
// tile when it is product 0).  The pair tiles' reads are all issued before
// the first update, so the wave waits for one memory round trip for them,
// not one per tile.
template <int Q, typename R, int PPW>
__device__ __forceinline__ void accumulate_p0(const typename Prec<R>::V4 (*pR)[2],
                                              const typename Prec<R>::V4 (*pI)[2],
                                              const typename Prec<R>::V4 &qR,
                                              const typename Prec<R>::V4 &qI, int wave,
                                              bool single0, int su, int lr, int lq,
                                              double2 *__restrict__ E) {
    ETile t[PPW > 0 ? PPW : 1];
#pragma unroll
    for (int s = 0; s < PPW; ++s) {
        const int u = wave + kWaves * s;
        load_etile<Q, R>(t[s], u % Q, u / Q, lr, lq, E);
    }
#pragma unroll
    for (int s = 0; s < PPW; ++s) {
        const int u = wave + kWaves * s;
        add_etile<Q, R>(t[s], u % Q, u / Q, lr, lq, pR[s][0], pI[s][0], E);
    }
    if (single0) {
        ETile t1;
        load_etile<Q, R>(t1, su % Q, su / Q, lr, lq, E);
        add_etile<Q, R>(t1, su % Q, su / Q, lr, lq, qR, qI, E);
    }
}

// Dual GEMM sharing the right operand:  P0 = A0 * B,  P1 = A1 * B  (padded
// NP x NP in precision R, K = kdim rounded up to the chunk), by 8 waves.  The
// A column panels and the B rows are staged through LDS in chunks of kChunk,
// the next chunk's global loads in flight while the current one is
// multiplied.  O1 may be the same array as B: every read of B is done before
// the write-back.
//
// Work split: tile (ti, tj) of P0 and the same tile of P1 form a pair that
// reads one B fragment per step.  Pair u = wave + 8 s (s < PPW) belongs
// whole to `wave`; the PAIRS % 8 leftover pairs are split into single tiles,
// one per wave (wave w < 2 REM: pair 8 PPW + w/2, product w % 2).  The pair
// loop is free of branches so the LDS reads of a chunk can be issued ahead
// of its MFMAs.  Accumulators stay in registers for the whole K loop.
//
//   MODE 0: O0 = P0, O1 = P1
//   MODE 1: E += P0 (FP64), O1 = P1
//   MODE 2: as MODE 1, and returns sum_ij |P1_ij| (FP64) to every thread
template <int Q, typename R, int MODE>
__device__ __forceinline__ double dual_gemm(unsigned char *lds, double *red,
                                            const typename Prec<R>::C *__restrict__ A0,
                                            const typename Prec<R>::C *__restrict__ A1,
                                            const typename Prec<R>::C *B, int kdim,
                                            typename Prec<R>::C *O0, typename Prec<R>::C *O1,
                                            double2 *__restrict__ E) {
    using P = Prec<R>;
    using C = typename P::C;
    using V4 = typename P::V4;
    constexpr int NP = 16 * Q;
    constexpr int PAIRS = Q * Q;
    constexpr int PPW = PAIRS / kWaves;
    constexpr int REM = PAIRS - PPW * kWaves;
    static_assert(2 * REM <= kWaves, "leftover tiles must fit one per wave");
    const int tid = opaque_tid();
    const int wave = uniform(tid >> 6), lane = tid & 63;
    const int lr = lane & 15, lq = lane >> 4;
    const bool single = wave < 2 * REM;
    const int su = kWaves * PPW + (wave >> 1), sw = wave & 1;
    C(*bs)[NP + 1] = reinterpret_cast<C(*)[NP + 1]>(lds);
    C(*as0)[NP] = reinterpret_cast<C(*)[NP]>(lds + GemmLay<Q, R>::B);
    C(*as1)[NP] = reinterpret_cast<C(*)[NP]>(lds + GemmLay<Q, R>::B + GemmLay<Q, R>::A);

    V4 pR[PPW > 0 ? PPW : 1][2], pI[PPW > 0 ? PPW : 1][2];
    V4 qR = {0, 0, 0, 0}, qI = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < PPW; ++s)
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            pR[s][w] = V4{0, 0, 0, 0};
            pI[s][w] = V4{0, 0, 0, 0};
        }

    const int nchunks = (kdim + kChunk - 1) / kChunk;
    // Staging: element e = tid (+ kBlock) of the B rows and the A0/A1 column
    // panels of a chunk, loaded one chunk ahead into registers.
    constexpr int PER = kChunk * NP;
    static_assert(PER <= 2 * kBlock, "chunk larger than the register stage");
    const int e0 = tid, e1 = tid + kBlock;
    const bool has0 = e0 < PER, has1 = e1 < PER;
    const int bo0 = e0 % kChunk + (e0 / kChunk) * NP, ao0 = e0 % NP + (e0 / NP) * NP;
    const int bo1 = e1 % kChunk + (e1 / kChunk) * NP, ao1 = e1 % NP + (e1 / NP) * NP;
    C b0, x0, y0, b1, x1, y1;
    auto load = [&](int c) {
        const int k0 = c * kChunk;
        if (has0) {
            b0 = B[bo0 + k0];
            x0 = A0[ao0 + k0 * NP];
            y0 = A1[ao0 + k0 * NP];
        }
        if (has1) {
            b1 = B[bo1 + k0];
            x1 = A0[ao1 + k0 * NP];
            y1 = A1[ao1 + k0 * NP];
        }
    };
    auto stash = [&]() {
        if (has0) {
            bs[e0 % kChunk][e0 / kChunk] = b0;
            as0[e0 / NP][e0 % NP] = x0;
            as1[e0 / NP][e0 % NP] = y0;
        }
        if (has1) {
            bs[e1 % kChunk][e1 / kChunk] = b1;
            as0[e1 / NP][e1 % NP] = x1;
            as1[e1 / NP][e1 % NP] = y1;
        }
    };

    load(0);
    for (int c = 0; c < nchunks; ++c) {
        stash();
        __syncthreads();
        if (c + 1 < nchunks) load(c + 1);
#pragma unroll
        for (int ks = 0; ks < kChunk / 4; ++ks) {
            const int kk = 4 * ks + lq;
#pragma unroll
            for (int s = 0; s < PPW; ++s) {
                const int u = wave + kWaves * s;
                const int ti = u % Q, tj = u / Q;
                const C b = bs[kk][16 * tj + lr];
                const C x = as0[kk][16 * ti + lr];
                const C y = as1[kk][16 * ti + lr];
                const R nby = -b.y;
                cmfma<R>(pR[s][0], pI[s][0], x, b, nby);
                cmfma<R>(pR[s][1], pI[s][1], y, b, nby);
            }
        }
        if (REM > 0 && single) {
            const int ti = su % Q, tj = su / Q;
            const C(*as)[NP] = sw ? as1 : as0;
#pragma unroll
            for (int ks = 0; ks < kChunk / 4; ++ks) {
                const int kk = 4 * ks + lq;
                const C b = bs[kk][16 * tj + lr];
                const C x = as[kk][16 * ti + lr];
                cmfma<R>(qR, qI, x, b, -b.y);
            }
        }
        __syncthreads();
    }

    // Write-back.  For MODE 1/2 the product-0 tiles read-modify-write the
    // FP64 accumulator E.
    double asum = 0.0;
    const bool single0 = REM > 0 && single && sw == 0;
    if (MODE == 0) {
#pragma unroll
        for (int s = 0; s < PPW; ++s) {
            const int u = wave + kWaves * s;
            store_tile<Q, R, false>(u % Q, u / Q, lr, lq, pR[s][0], pI[s][0], O0, asum);
        }
        if (single0) store_tile<Q, R, false>(su % Q, su / Q, lr, lq, qR, qI, O0, asum);
    } else {
        accumulate_p0<Q, R, PPW>(pR, pI, qR, qI, wave, single0, su, lr, lq, E);
    }
#pragma unroll
    for (int s = 0; s < PPW; ++s) {
        const int u = wave + kWaves * s;
        store_tile<Q, R, MODE == 2>(u % Q, u / Q, lr, lq, pR[s][1], pI[s][1], O1, asum);
    }
    if (REM > 0 && single && sw == 1)
        store_tile<Q, R, MODE == 2>(su % Q, su / Q, lr, lq, qR, qI, O1, asum);
    if (MODE == 2) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) asum += __shfl_xor(asum, off, 64);
        if (lane == 0) red[wave] = asum;
        __syncthreads();
        double tot = 0.0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) tot += red[w];
        return tot;
    }
    return 0.0;
}

// One stacked tile of dual_gemm_half: rows 0..7 of the MFMA tile are rows
// 16 (Q-1) .. 16 (Q-1) + 7 of P0, rows 8..15 the same rows of P1, in tile
// column tj.  P0's part goes to O0 (MODE 0) or is added to E (MODE 1, 2);
// P1's part goes to O1 (and into asum in MODE 2).
template <int Q, typename R, int MODE>
__device__ __forceinline__ void store_stacked(int tj, int lr, int lq,
                                              const typename Prec<R>::V4 &accR,
                                              const typename Prec<R>::V4 &accI,
                                              typename Prec<R>::C *O0, typename Prec<R>::C *O1,
                                              double2 *__restrict__ E, double &asum) {
    using P = Prec<R>;
    using C = typename P::C;
    constexpr int NP = 16 * Q;
    const int col = 16 * tj + lr;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int r = P::out_row(lq, v);
        const int idx = 16 * (Q - 1) + (r & 7) + col * NP;
        C val;
        val.x = accR[v];
        val.y = accI[v];
        if (r < 8) {
            if (MODE == 0)
                O0[idx] = val;
            else
                E[idx] = cadd(E[idx], make_double2(accR[v], accI[v]));
        } else {
            O1[idx] = val;
            if (MODE == 2) asum += hypot((double)val.x, (double)val.y);
        }
    }
}

// The dual GEMM of dual_gemm (same products, operands, MODEs and LDS) for
// orders kdim <= 16 Q - 8, whose last tile row holds at most 8 real rows.
// The last tile row of P0 and that of P1 then share one MFMA tile: its A
// operand takes rows 16 (Q-1) .. 16 (Q-1) + 7 of A0 in its rows 0..7 and the
// same rows of A1 in rows 8..15, against the one B.  The products take
// (Q-1) Q tile pairs and Q stacked tiles: 2 Q^2 - Q tiles where dual_gemm
// takes 2 Q^2 (45 for 50 at Q = 5).  Rows 16 Q - 8 .. NP - 1 of O0, O1 and E
// are not written; no caller reads them (an A operand's rows at or beyond
// kdim never enter a product, and B's rows there lie beyond K).
//
// Work split: pair u = wave + 8 s (s < PPW) is tile (u % (Q-1), u / (Q-1))
// of both products; the REM leftover pairs go one to each wave w < REM; the
// stacked tiles two to a wave from wave REM on, the last one alone when Q is
// odd.  At Q = 5: waves 0-3 take three pairs, waves 4 and 5 two pairs and
// two stacked tiles, wave 6 two pairs and one stacked tile, wave 7 two
// pairs; 12 tiles on each of two SIMDs where dual_gemm puts 13.
template <int Q, typename R, int MODE>
__device__ __forceinline__ double dual_gemm_half(unsigned char *lds, double *red,
                                                 const typename Prec<R>::C *__restrict__ A0,
                                                 const typename Prec<R>::C *__restrict__ A1,
                                                 const typename Prec<R>::C *B, int kdim,
                                                 typename Prec<R>::C *O0, typename Prec<R>::C *O1,
                                                 double2 *__restrict__ E) {
    using P = Prec<R>;
    using C = typename P::C;
    using V4 = typename P::V4;
    constexpr int NP = 16 * Q;
    constexpr int QR = Q - 1;  // full tile rows
    constexpr int PAIRS = QR * Q;
    constexpr int PPW = PAIRS / kWaves;
    constexpr int REM = PAIRS - PPW * kWaves;
    constexpr int SW = (Q + 1) / 2;  // waves holding stacked tiles
    static_assert(Q >= 2 && REM + SW <= kWaves, "stacked tiles must fit the waves after the pairs");
    const int tid = opaque_tid();
    const int wave = uniform(tid >> 6), lane = tid & 63;
    const int lr = lane & 15, lq = lane >> 4;
    // this wave's work beyond its PPW pairs: 1 = a leftover pair, 2 = two
    // stacked tiles (columns stj, stj + 1), 3 = one stacked tile (column
    // stj), 0 = none
    const int sk = wave - REM;
    const int kind = wave < REM ? 1 : sk < SW ? (2 * sk + 1 < Q ? 2 : 3) : 0;
    const int xu = kWaves * PPW + wave;
    const int xti = xu % QR, xtj = xu / QR;
    const int stj = kind >= 2 ? 2 * sk : 0;
    C(*bs)[NP + 1] = reinterpret_cast<C(*)[NP + 1]>(lds);
    C(*as0)[NP] = reinterpret_cast<C(*)[NP]>(lds + GemmLay<Q, R>::B);
    C(*as1)[NP] = reinterpret_cast<C(*)[NP]>(lds + GemmLay<Q, R>::B + GemmLay<Q, R>::A);
    // LDS element offsets of the extra tiles' operands: A from sa (as0, then
    // as1 at offset kChunk NP), B from sb; the stacked A operand takes lane
    // row lr < 8 from A0 and lr >= 8 from A1
    const C *sa = &as0[0][0];
    const C *sb = &bs[0][0];
    const int srow = 16 * QR + (lr & 7) + (lr < 8 ? 0 : kChunk * NP);
    const int xa = kind == 1 ? 16 * xti + lr : srow;
    const int ya = kind == 1 ? kChunk * NP + 16 * xti + lr : srow;
    const int xb = (kind == 1 ? 16 * xtj : 16 * stj) + lr;
    const int yb = kind == 1 ? xb : kind == 2 ? xb + 16 : xb;

    V4 pR[PPW > 0 ? PPW : 1][2], pI[PPW > 0 ? PPW : 1][2], xR[2], xI[2];
#pragma unroll
    for (int w = 0; w < 2; ++w) {
#pragma unroll
        for (int s = 0; s < PPW; ++s) {
            pR[s][w] = V4{0, 0, 0, 0};
            pI[s][w] = V4{0, 0, 0, 0};
        }
        xR[w] = V4{0, 0, 0, 0};
        xI[w] = V4{0, 0, 0, 0};
    }

    const int nchunks = (kdim + kChunk - 1) / kChunk;
    constexpr int PER = kChunk * NP;
    static_assert(PER <= 2 * kBlock, "chunk larger than the register stage");
    const int e0 = tid, e1 = tid + kBlock;
    const bool has0 = e0 < PER, has1 = e1 < PER;
    const int bo0 = e0 % kChunk + (e0 / kChunk) * NP, ao0 = e0 % NP + (e0 / NP) * NP;
    const int bo1 = e1 % kChunk + (e1 / kChunk) * NP, ao1 = e1 % NP + (e1 / NP) * NP;
    C b0, x0, y0, b1, x1, y1;
    auto load = [&](int c) {
        const int k0 = c * kChunk;
        if (has0) {
            b0 = B[bo0 + k0];
            x0 = A0[ao0 + k0 * NP];
            y0 = A1[ao0 + k0 * NP];
        }
        if (has1) {
            b1 = B[bo1 + k0];
            x1 = A0[ao1 + k0 * NP];
            y1 = A1[ao1 + k0 * NP];
        }
    };
    auto stash = [&]() {
        if (has0) {
            bs[e0 % kChunk][e0 / kChunk] = b0;
            as0[e0 / NP][e0 % NP] = x0;
            as1[e0 / NP][e0 % NP] = y0;
        }
        if (has1) {
            bs[e1 % kChunk][e1 / kChunk] = b1;
            as0[e1 / NP][e1 % NP] = x1;
            as1[e1 / NP][e1 % NP] = y1;
        }
    };

    load(0);
    for (int c = 0; c < nchunks; ++c) {
        stash();
        __syncthreads();
        if (c + 1 < nchunks) load(c + 1);
#pragma unroll
        for (int ks = 0; ks < kChunk / 4; ++ks) {
            const int kk = 4 * ks + lq;
#pragma unroll
            for (int s = 0; s < PPW; ++s) {
                const int u = wave + kWaves * s;
                const int ti = u % QR, tj = u / QR;
                const C b = bs[kk][16 * tj + lr];
                const C x = as0[kk][16 * ti + lr];
                const C y = as1[kk][16 * ti + lr];
                const R nby = -b.y;
                cmfma<R>(pR[s][0], pI[s][0], x, b, nby);
                cmfma<R>(pR[s][1], pI[s][1], y, b, nby);
            }
        }
        if (kind != 0) {
            // the extra tiles: acc 0 = A[xa] B[xb], acc 1 = A[ya] B[yb] (none
            // for a lone stacked tile)
#pragma unroll
            for (int ks = 0; ks < kChunk / 4; ++ks) {
                const int kk = 4 * ks + lq;
                const C x = sa[xa + kk * NP];
                const C y = sa[ya + kk * NP];
                const C b = sb[xb + kk * (NP + 1)];
                const C bb = sb[yb + kk * (NP + 1)];
                cmfma<R>(xR[0], xI[0], x, b, -b.y);
                if (kind != 3) cmfma<R>(xR[1], xI[1], y, bb, -bb.y);
            }
        }
        __syncthreads();
    }

    // Write-back.  For MODE 1/2 the product-0 tiles read-modify-write the
    // FP64 accumulator E; their reads are issued before the first update.
    double asum = 0.0;
    if (MODE == 0) {
#pragma unroll
        for (int s = 0; s < PPW; ++s) {
            const int u = wave + kWaves * s;
            store_tile<Q, R, false>(u % QR, u / QR, lr, lq, pR[s][0], pI[s][0], O0, asum);
        }
        if (REM > 0 && kind == 1) store_tile<Q, R, false>(xti, xtj, lr, lq, xR[0], xI[0], O0, asum);
    } else {
        ETile t[PPW > 0 ? PPW : 1], tx;
#pragma unroll
        for (int s = 0; s < PPW; ++s) {
            const int u = wave + kWaves * s;
            load_etile<Q, R>(t[s], u % QR, u / QR, lr, lq, E);
        }
        if (REM > 0 && kind == 1) load_etile<Q, R>(tx, xti, xtj, lr, lq, E);
#pragma unroll
        for (int s = 0; s < PPW; ++s) {
            const int u = wave + kWaves * s;
            add_etile<Q, R>(t[s], u % QR, u / QR, lr, lq, pR[s][0], pI[s][0], E);
        }
        if (REM > 0 && kind == 1) add_etile<Q, R>(tx, xti, xtj, lr, lq, xR[0], xI[0], E);
    }
#pragma unroll
    for (int s = 0; s < PPW; ++s) {
        const int u = wave + kWaves * s;
        store_tile<Q, R, MODE == 2>(u % QR, u / QR, lr, lq, pR[s][1], pI[s][1], O1, asum);
    }
    if (REM > 0 && kind == 1) store_tile<Q, R, MODE == 2>(xti, xtj, lr, lq, xR[1], xI[1], O1, asum);
    if (kind >= 2) store_stacked<Q, R, MODE>(stj, lr, lq, xR[0], xI[0], O0, O1, E, asum);
    if (kind == 2) store_stacked<Q, R, MODE>(stj + 1, lr, lq, xR[1], xI[1], O0, O1, E, asum);
    if (MODE == 2) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) asum += __shfl_xor(asum, off, 64);
        if (lane == 0) red[wave] = asum;
        __syncthreads();
        double tot = 0.0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) tot += red[w];
        return tot;
    }
    return 0.0;
}

// dual_gemm, or dual_gemm_half when HALF (orders kdim <= 16 Q - 8).
template <int Q, typename R, int MODE, bool HALF>
__device__ __forceinline__ double dual_gemm_any(unsigned char *lds, double *red,
                                                const typename Prec<R>::C *__restrict__ A0,
                                                const typename Prec<R>::C *__restrict__ A1,
                                                const typename Prec<R>::C *B, int kdim,
                                                typename Prec<R>::C *O0, typename Prec<R>::C *O1,
                                                double2 *__restrict__ E) {
    if constexpr (HALF)
        return dual_gemm_half<Q, R, MODE>(lds, red, A0, A1, B, kdim, O0, O1, E);
    else
        return dual_gemm<Q, R, MODE>(lds, red, A0, A1, B, kdim, O0, O1, E);
}

// LDS of the blocked GEMM (orders beyond 80): one K-chunk of the A0 and A1
// row blocks (16 BI rows) and of the B column block (16 BJ columns, padded).
constexpr int kBI = 4, kBJ = 6;  // output block of the blocked GEMM, in tiles
// K-chunk of the blocked GEMM: twice the small-order one, since its workgroup
// does not share the CU with an inverse workgroup (the two kernels' registers
// do not fit one CU together at these orders) and so has the LDS to spare;
// a deeper chunk halves the barriers per K and gives each chunk's loads more
// MFMA work to hide behind.
constexpr int kChunkL = 16;
template <int Q, typename R>
struct GemmLayL {
    using C = typename Prec<R>::C;
    static constexpr size_t A = (size_t)kChunkL * 16 * kBI * sizeof(C);
    static constexpr size_t B = (size_t)kChunkL * (16 * kBJ + 1) * sizeof(C);
    static constexpr size_t bytes = 2 * A + B;
};

// The dual GEMM of dual_gemm (same products and MODEs) for orders whose
// Q x Q tile pairs do not fit the waves' registers: the output is covered in
// blocks of kBI x kBJ tile pairs, one pass over K per block, the block's A0 /
// A1 rows and B columns staged through LDS by K-chunks.  kBI kBJ = 24 pairs
// per block, three per wave.  B is read in every pass, so O1 must not be B.
// Only NIB row blocks of kBI tiles from ib0 on are formed (and summed); they
// depend on no other rows of A0 and A1.  In MODE 2 the sum of |O1| is formed row
// block by row block, so that it does not depend on which workgroup forms
// which; red: NIB kWaves.
template <int Q, typename R, int MODE, int NIB>
__device__ __forceinline__ double dual_gemm_blocked(unsigned char *lds, double *red,
                                                    const typename Prec<R>::C *__restrict__ A0,
                                                    const typename Prec<R>::C *__restrict__ A1,
                                                    const typename Prec<R>::C *__restrict__ B,
                                                    int kdim, typename Prec<R>::C *__restrict__ O0,
                                                    typename Prec<R>::C *__restrict__ O1,
                                                    double2 *__restrict__ E, int ib0) {
    using P = Prec<R>;
    using C = typename P::C;
    using V4 = typename P::V4;
    constexpr int NP = 16 * Q;
    constexpr int RI = 16 * kBI, CJ = 16 * kBJ;
    constexpr int NBJ = (Q + kBJ - 1) / kBJ;
    constexpr int PPW = kBI * kBJ / kWaves;
    static_assert(PPW * kWaves == kBI * kBJ, "block pairs must split evenly over the waves");
    constexpr int NA = kChunkL * RI / kBlock, NB = kChunkL * CJ / kBlock;
    static_assert(NA * kBlock == kChunkL * RI, "whole A elements per thread and chunk");
    static_assert(NB * kBlock == kChunkL * CJ, "whole B elements per thread and chunk");
    const int tid = threadIdx.x;
    const int wave = uniform(tid >> 6), lane = tid & 63;
    const int lr = lane & 15, lq = lane >> 4;
    C(*as0)[RI] = reinterpret_cast<C(*)[RI]>(lds);
    C(*as1)[RI] = reinterpret_cast<C(*)[RI]>(lds + GemmLayL<Q, R>::A);
    C(*bs)[CJ + 1] = reinterpret_cast<C(*)[CJ + 1]>(lds + 2 * GemmLayL<Q, R>::A);
    const int nchunks = (kdim + kChunkL - 1) / kChunkL;
    // staging: A elements e = tid + u kBlock of a chunk (kk = e / RI, row e % RI),
    // B elements e = tid + u kBlock (kk = e % kChunkL, column e / kChunkL)

    double rsum[NIB];
#pragma unroll
    for (int i = 0; i < NIB; ++i) rsum[i] = 0.0;
    for (int blk = 0; blk < NIB * NBJ; ++blk) {
        double asum = 0.0;
        const int i0 = kBI * (ib0 + blk % NIB), j0 = kBJ * (blk / NIB);
        const int ni = Q - i0 < kBI ? Q - i0 : kBI, nj = Q - j0 < kBJ ? Q - j0 : kBJ;
        int ti[PPW], tj[PPW];
        bool act[PPW];
        V4 pR[PPW][2], pI[PPW][2];
#pragma unroll
        for (int s = 0; s < PPW; ++s) {
            const int pp = wave + kWaves * s;
            act[s] = pp < ni * nj;
            ti[s] = act[s] ? pp % ni : 0;
            tj[s] = act[s] ? pp / ni : 0;
#pragma unroll
            for (int w = 0; w < 2; ++w) {
                pR[s][w] = V4{0, 0, 0, 0};
                pI[s][w] = V4{0, 0, 0, 0};
            }
        }
        C xa[NA], ya[NA], bb[NB];
        auto load = [&](int c) {
            const int k0 = c * kChunkL;
#pragma unroll
            for (int u = 0; u < NA; ++u) {
                const int e = tid + u * kBlock, ka = e / RI, ra = e % RI;
                xa[u].x = xa[u].y = ya[u].x = ya[u].y = 0;
                if (16 * i0 + ra < NP) {
                    xa[u] = A0[16 * i0 + ra + (k0 + ka) * NP];
                    ya[u] = A1[16 * i0 + ra + (k0 + ka) * NP];
                }
            }
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const int e = tid + u * kBlock, kb = e % kChunkL, cb = e / kChunkL;
                bb[u].x = bb[u].y = 0;
                if (16 * j0 + cb < NP) bb[u] = B[k0 + kb + (16 * j0 + cb) * NP];
            }
        };
        auto stash = [&]() {
#pragma unroll
            for (int u = 0; u < NA; ++u) {
                const int e = tid + u * kBlock;
                as0[e / RI][e % RI] = xa[u];
                as1[e / RI][e % RI] = ya[u];
            }
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const int e = tid + u * kBlock;
                bs[e % kChunkL][e / kChunkL] = bb[u];
            }
        };
        load(0);
        for (int c = 0; c < nchunks; ++c) {
            stash();
            __syncthreads();
            if (c + 1 < nchunks) load(c + 1);
#pragma unroll
            for (int ks = 0; ks < kChunkL / 4; ++ks) {
                const int kk = 4 * ks + lq;
#pragma unroll
                for (int s = 0; s < PPW; ++s) {
                    if (!act[s]) continue;
                    const C b = bs[kk][16 * tj[s] + lr];
                    const C x = as0[kk][16 * ti[s] + lr];
                    const C y = as1[kk][16 * ti[s] + lr];
                    const R nby = -b.y;
                    cmfma<R>(pR[s][0], pI[s][0], x, b, nby);
                    cmfma<R>(pR[s][1], pI[s][1], y, b, nby);
                }
            }
            __syncthreads();
        }
        if (MODE == 0) {
#pragma unroll
            for (int s = 0; s < PPW; ++s)
                if (act[s]) store_tile<Q, R, false>(i0 + ti[s], j0 + tj[s], lr, lq, pR[s][0], pI[s][0], O0, asum);
        } else {
            ETile t[PPW];
#pragma unroll
            for (int s = 0; s < PPW; ++s)
                if (act[s]) load_etile<Q, R>(t[s], i0 + ti[s], j0 + tj[s], lr, lq, E);
#pragma unroll
            for (int s = 0; s < PPW; ++s)
                if (act[s]) add_etile<Q, R>(t[s], i0 + ti[s], j0 + tj[s], lr, lq, pR[s][0], pI[s][0], E);
        }
#pragma unroll
        for (int s = 0; s < PPW; ++s)
            if (act[s])
                store_tile<Q, R, MODE == 2>(i0 + ti[s], j0 + tj[s], lr, lq, pR[s][1], pI[s][1], O1, asum);
        if (MODE == 2) {
#pragma unroll
            for (int i = 0; i < NIB; ++i) rsum[i] += blk % NIB == i ? asum : 0.0;
        }
    }
    if (MODE == 2) {
#pragma unroll
        for (int i = 0; i < NIB; ++i) {
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) rsum[i] += __shfl_xor(rsum[i], off, 64);
            if (lane == 0) red[i * kWaves + wave] = rsum[i];
        }
        __syncthreads();
        double tot = 0.0;
        for (int i = 0; i < NIB; ++i) {
            double part = 0.0;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) part += red[i * kWaves + w];
            tot += part;
        }
        return tot;
    }
    return 0.0;
}

// Per-slot workspace: alpha, beta, m1, m2, g in precision R, then eps_s and
// eps_t in FP64, each NP x NP column-major.
template <int Q, typename R>
struct SlotWork {
    using C = typename Prec<R>::C;
    static constexpr size_t NN = (size_t)(16 * Q) * (16 * Q);
    static constexpr size_t bytes = 5 * NN * sizeof(C) + 2 * NN * sizeof(double2);
    static_assert(!std::is_same_v<R, double> || bytes == slot_bytes_lds_fp64(Q),
                  "slot layout and its host-side size disagree");
    C *al, *be, *m1, *m2, *g;
    double2 *es, *et;
    // alpha / beta of the current iteration and where the next ones go: the
    // single-pass GEMMs overwrite them in place
    __device__ C *alpha(int) const { return al; }
    __device__ C *beta(int) const { return be; }
    __device__ C *alpha_next(int) const { return al; }
    __device__ C *beta_next(int) const { return be; }
    __device__ SlotWork(void *work, int slot) {
        unsigned char *base = reinterpret_cast<unsigned char *>(work) + (size_t)slot * bytes;
        C *c = reinterpret_cast<C *>(base);
        al = c;
        be = c + NN;
        m1 = c + 2 * NN;
        m2 = c + 3 * NN;
        g = c + 4 * NN;
        double2 *d = reinterpret_cast<double2 *>(base + 5 * NN * sizeof(C));
        es = d;
        et = d + NN;
    }
};

// Per-slot workspace beyond order 80: alpha and beta twice (current and next,
// swapped every iteration: the blocked GEMM reads B over several passes, so it
// cannot overwrite it), m1, m2, g in precision R, eps_s and eps_t in FP64, and
// the Gauss-Jordan matrix (NP x (NP+1), FP64-sized), all in global memory.
template <int Q, typename R>
struct SlotWorkL {
    using C = typename Prec<R>::C;
    static constexpr size_t NN = (size_t)(16 * Q) * (16 * Q);
    static constexpr size_t SB = (size_t)(16 * Q) * (16 * Q + 1) * sizeof(double2);
    // the block columns of a panel quad (4 kPanel columns of 16 Q, FP64-sized)
    static constexpr size_t MB = (size_t)4 * kPanel * (16 * Q) * sizeof(double2);
    static constexpr size_t bytes = 7 * NN * sizeof(C) + 2 * NN * sizeof(double2) + SB + MB;
    C *ab, *m1, *m2, *g;  // ab: alpha[0], alpha[1], beta[0], beta[1]
    double2 *es, *et;
    unsigned char *S, *Mq;
    __device__ C *alpha(int par) const { return ab + par * NN; }
    __device__ C *beta(int par) const { return ab + (2 + par) * NN; }
    __device__ C *alpha_next(int par) const { return ab + (par ^ 1) * NN; }
    __device__ C *beta_next(int par) const { return ab + (2 + (par ^ 1)) * NN; }
    __device__ SlotWorkL(void *work, int slot) {
        unsigned char *base = reinterpret_cast<unsigned char *>(work) + (size_t)slot * bytes;
        C *c = reinterpret_cast<C *>(base);
        ab = c;
        m1 = c + 4 * NN;
        m2 = c + 5 * NN;
        g = c + 6 * NN;
        double2 *d = reinterpret_cast<double2 *>(base + 7 * NN * sizeof(C));
        es = d;
        et = d + NN;
        S = reinterpret_cast<unsigned char *>(d + 2 * NN);
        Mq = S + SB;
    }
};

// One Gauss-Jordan per slot: a slot without an instance takes the next one
// (eps_s = eps_t = H00, alpha = H01, beta = H01^dagger) and starts its first
// iteration; kLoop computes g = (z - eps_i)^-1 for the GEMM round; kFinal0..2
// compute the diagonals of GLL = (z - eps_s)^-1, GRR = (z - eps_t)^-1,
// GB = (z - eps_i)^-1 in FP64 and their traces, and the last of them writes
// the instance's outputs.  sR / tR hold the matrix and the panel pivot rows
// for the precision-R inverse, s64 / t64 for the FP64 final ones.
// New-instance set-up of a slot in kEmpty, by NT threads: claim the next
// instance from the queue (kDone past the last one) and start eps_s = eps_t =
// H00, alpha = H01, beta = H01^dagger (src/surfgreen.f90:74-78), iteration 1.
// st is the slot's state in shared memory; returns its new phase.
template <int Q, typename R, int NT, typename W>
__device__ __forceinline__ int setup_instance(const DecimateArgs &a, const W &w, SlotState &st) {
    using C = typename Prec<R>::C;
    constexpr int NP = 16 * Q;
    constexpr int NN = NP * NP;
    const int tid = threadIdx.x;
    if (tid == 0) st.t = (int)atomicAdd(a.queue, 1u);
    __syncthreads();
    const int t = uniform(st.t);
    if (queue_empty((unsigned)t, a.ninst)) {
        if (tid == 0) st.phase = kDone;
        __syncthreads();
        return kDone;
    }
    int ik;
    double2 z;
    instance_of(a, t, ik, z);
    const double2 *H00 = a.hk + (size_t)ik * 2 * NN;
    const double2 *H01 = H00 + NN;
    C *al = w.alpha(0), *be = w.beta(0);
    // batches whose loads are all issued before their stores (the stores
    // may alias the loads as far as the compiler knows)
    constexpr int kIter = (NN + NT - 1) / NT, kBatch = 4;
    for (int it0 = 0; it0 < kIter; it0 += kBatch) {
        double2 h[kBatch], h1[kBatch], ht[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) h[u] = h1[u] = ht[u] = make_double2(0.0, 0.0);
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int e = tid + (it0 + u) * NT;
            if (it0 + u < kIter && e < NN) {
                const int i = e % NP, j = e / NP;
                h[u] = H00[e];
                h1[u] = H01[e];
                ht[u] = H01[j + i * NP];
            }
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int e = tid + (it0 + u) * NT;
            if (it0 + u < kIter && e < NN) {
                w.es[e] = h[u];
                w.et[e] = h[u];
                C av;
                av.x = (R)h1[u].x;
                av.y = (R)h1[u].y;
                al[e] = av;
                C bv;
                bv.x = (R)ht[u].x;
                bv.y = (R)(-ht[u].y);
                be[e] = bv;
            }
        }
    }
    if (tid == 0) {
        st.it = 1;
        st.status = 0;
        st.dl = 0.0;
        st.dr = 0.0;
        st.phase = kLoop;
    }
    __syncthreads();
    return kLoop;
}

template <int Q, typename R, int NT, typename W>
__device__ __forceinline__ void gj_round(const DecimateArgs &a, int slot, const W &w,
                                         Common<Q> &cm, unsigned char *sR, unsigned char *tR,
                                         unsigned char *s64, unsigned char *t64) {
    using C = typename Prec<R>::C;
    constexpr int NP = 16 * Q;
    constexpr int NN = NP * NP;
    const int tid = threadIdx.x;
    SlotState *st = a.state + slot;
    const int n = a.n;

    if (tid == 0) cm.s = *st;
    __syncthreads();
    int phase = uniform(cm.s.phase);
    if (phase == kGemm || phase == kDone) return;
    if (phase == kEmpty) {
        // only on a slot's first round: afterwards the GEMM round that follows
        // an instance's last inverse starts the next one
        phase = setup_instance<Q, R, NT>(a, w, cm.s);
        if (phase == kDone) {
            if (tid == 0) *st = cm.s;
            return;
        }
    }
    int ik;
    double2 z;
    instance_of(a, uniform(cm.s.t), ik, z);
    const double2 *H00 = a.hk + (size_t)ik * 2 * NN;
    // the block columns of the panel quads (orders beyond 80)
    C *mgR = nullptr;
    double2 *mg64 = nullptr;
    if constexpr (Q > 5) {
        mgR = reinterpret_cast<C *>(w.Mq);
        mg64 = reinterpret_cast<double2 *>(w.Mq);
    }
    if (phase == kLoop) {
        const bool sing = gj_inverse<Q, R, NT>(sR, tR, cm, w.es, w.et, H00, z, n, 4, nullptr, w.g,
                                               mgR);
        if (tid == 0) {
            if (sing) cm.s.status |= 1;
            cm.s.phase = kGemm;
        }
    } else {
        const int q = phase - kFinal0;
        double2 *full = a.gfull ? a.gfull + ((size_t)cm.s.t * 3 + q) * n * n : nullptr;
        // eps_s, eps_t, eps_i = eps_s + eps_t - H00
        const double2 *eps = q == 1 ? w.et : w.es;
        const double2 *eps2 = q == 2 ? w.et : nullptr;
        const bool sing = gj_inverse<Q, double, NT>(s64, t64, cm, eps, eps2, H00, z, n,
                                                    full ? 2 : 1, full, nullptr, mg64);
        if (tid == 0) {
            if (sing) cm.s.status |= 1;
            final_traces<Q>(a, cm, LdsInverse<Q>{s64, cm}, q, ik);
            cm.s.phase = q == 0 ? kFinal1 : q == 1 ? kFinal2 : kEmpty;
        }
    }
    if (tid == 0) *st = cm.s;
}

// Orders up to 80: the matrix in LDS, 4 waves (one per SIMD).
template <int Q, typename R>
__global__ void __launch_bounds__(kGjBlock) gj_round_kernel(DecimateArgs a, int slot0) {
    // The matrix region is dynamic shared memory (GjLay<Q, R>::bytes at
    // launch): with its size unknown here, the compiler does not take the
    // one-workgroup-per-CU occupancy it implies as licence to claim every
    // register, and the kernel's register count stays what it uses, small
    // enough to leave room for a GEMM workgroup beside it.
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ Common<Q> cm;
    const int slot = slot0 + blockIdx.x;
    const SlotWork<Q, R> w(a.work, slot);
    gj_round<Q, R, kGjBlock>(a, slot, w, cm, lds, lds + GjLay<Q, R>::S, lds,
                             lds + GjLay<Q, double>::S);
}

// Orders beyond 80: the matrix in the slot's global workspace (it no longer
// fits in LDS), the panel pivot rows in LDS, 8 waves.
// Its LDS (dynamic, GjLayL<Q>::bytes): the pivot rows of a panel quad (4
// kPanel rows of 16 Q) where the quads run, else those of a panel pair and
// the first panel's columns (3 kPanel rows), FP64 at most.
template <int Q>
struct GjLayL {
    static constexpr size_t bytes = (size_t)(use_quads<Q>() ? 4 : 3) * kPanel * 16 * Q * sizeof(double2);
};

template <int Q, typename R>
__global__ void __launch_bounds__(kBlock) gj_large_round_kernel(DecimateArgs a, int slot0) {
    extern __shared__ __align__(16) unsigned char tlds[];
    __shared__ Common<Q> cm;
    const int slot = slot0 + blockIdx.x;
    const SlotWorkL<Q, R> w(a.work, slot);
    gj_round<Q, R, kBlock>(a, slot, w, cm, w.S, tlds, w.S, tlds);
}

// The three dual GEMMs of one iteration for every slot in kGemm, then the
// stop rule: kFinal0 when sum |alpha'| <= accuracy or at itermax (status bit
// 1, iterations = itermax), else the next iteration's kLoop.  beta' and
// alpha' overwrite beta and alpha in place.  A slot in kEmpty (its instance
// finished in the inverse round before) is set up for its next instance
// here, where the round has no GEMMs for it, instead of in the inverse round,
// whose workgroups set the pace of the rounds.
// HALF: the order is at most 16 Q - 8 (dual_gemm_half).
template <int Q, typename R, bool HALF>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_num_vgpr(kGemmVgprHalf)))
gemm_round_kernel(DecimateArgs a, int slot0) {
    __shared__ __align__(16) unsigned char lds[GemmLay<Q, R>::bytes];
    __shared__ double red[kWaves];
    __shared__ SlotState sst;
    const int slot = slot0 + blockIdx.x;
    SlotState *st = a.state + slot;
    if (threadIdx.x == 0) sst = *st;
    __syncthreads();
    const int phase = uniform(sst.phase);
    const SlotWork<Q, R> w(a.work, slot);
    if (phase == kEmpty) {
        setup_instance<Q, R, kBlock>(a, w, sst);
        if (threadIdx.x == 0) *st = sst;
        return;
    }
    if (phase != kGemm) return;
    const int n = a.n;
    dual_gemm_any<Q, R, 0, HALF>(lds, red, w.al, w.be, w.g, n, w.m1, w.m2, nullptr);
    __syncthreads();
    dual_gemm_any<Q, R, 1, HALF>(lds, red, w.m1, w.m2, w.be, n, nullptr, w.be, w.es);
    __syncthreads();
    const double s =
        dual_gemm_any<Q, R, 2, HALF>(lds, red, w.m2, w.m1, w.al, n, nullptr, w.al, w.et);
    if (threadIdx.x == 0) {
        SlotState v = sst;
        if (s <= a.accuracy) {
            v.phase = kFinal0;
        } else if (v.it >= a.itermax) {
            v.status |= 2;
            v.phase = kFinal0;
        } else {
            v.it += 1;
            v.phase = kLoop;
        }
        *st = v;
    }
}

// The same for orders beyond 112, with the blocked GEMM; alpha' and beta' go to
// the other half of the slot's alpha / beta pair (iteration parity).  A slot's
// row blocks go to one workgroup, or (SPREAD) to one each (on one XCD, whose L2
// then serves g, alpha and beta to all of them): the rows of all three
// products depend on the same rows of alpha and beta only.  The last of them to
// finish adds their parts of sum |alpha'| in order and applies the stop rule;
// one workgroup alone adds the same parts in the same order.
// (With the share a run-time number the unspread rounds took 1% longer.)
template <int Q, typename R, bool SPREAD>
__global__ void __launch_bounds__(kBlock) gemm_large_round_kernel(DecimateArgs a, int slot0,
                                                                  int slots) {
    __shared__ __align__(16) unsigned char lds[GemmLayL<Q, R>::bytes];
    __shared__ double red[kMaxSplit * kWaves];
    __shared__ SlotState sst;
    constexpr int NBI = (Q + kBI - 1) / kBI;
    static_assert(NBI <= kMaxSplit, "a part for every row block");
    constexpr int split = SPREAD ? NBI : 1, NIB = SPREAD ? 1 : NBI;
    const int qd = blockIdx.x >> 3;
    const int local = SPREAD ? (qd / split) * 8 + (blockIdx.x & 7) : blockIdx.x;
    const int share = SPREAD ? qd % split : 0;
    if (SPREAD && local >= slots) return;
    const int slot = slot0 + local;
    SlotState *st = a.state + slot;
    if (threadIdx.x == 0) sst = *st;
    __syncthreads();
    const int phase = uniform(sst.phase);
    const SlotWorkL<Q, R> w(a.work, slot);
    if (phase == kEmpty) {
        if (share != 0) return;
        setup_instance<Q, R, kBlock>(a, w, sst);
        if (threadIdx.x == 0) *st = sst;
        return;
    }
    if (phase != kGemm) return;
    const int par = uniform((sst.it - 1) & 1);
    const int n = a.n;
    dual_gemm_blocked<Q, R, 0, NIB>(lds, red, w.alpha(par), w.beta(par), w.g, n, w.m1, w.m2, nullptr,
                                    share);
    __syncthreads();
    dual_gemm_blocked<Q, R, 1, NIB>(lds, red, w.m1, w.m2, w.beta(par), n, nullptr, w.beta_next(par),
                                    w.es, share);
    __syncthreads();
    double s = dual_gemm_blocked<Q, R, 2, NIB>(lds, red, w.m2, w.m1, w.alpha(par), n, nullptr,
                                               w.alpha_next(par), w.et, share);
    if (threadIdx.x == 0) {
        if constexpr (SPREAD) {
            __hip_atomic_store(&st->part[share], s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __threadfence();
            if (atomicAdd(&st->arrived, 1u) + 1 < (unsigned)split) return;
            __threadfence();
            s = 0.0;
            for (int k = 0; k < split; ++k)
                s += __hip_atomic_load(&st->part[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        SlotState v = sst;
        v.arrived = 0;
        if (s <= a.accuracy) {
            v.phase = kFinal0;
        } else if (v.it >= a.itermax) {
            v.status |= 2;
            v.phase = kFinal0;
        } else {
            v.it += 1;
            v.phase = kLoop;
        }
        *st = v;
    }
}

// ---------------------------------------------------------------------------
// Persistent schedule (orders up to 80).  One workgroup per CU owns one
// instance at a time and runs its whole decimation without leaving the
// kernel -- per iteration the inverse, the three dual GEMMs and the stop
// rule, then the three final inverses and the traces -- and then claims the
// next instance from the queue.  An instance's matrices stay in its
// workgroup's slot of global memory and never pass to another workgroup or
// kernel, so the only word the workgroups share is the queue counter, and
// instances of uneven iteration counts need no common pace.
template <int Q, typename R>
struct PersistLay {
    static constexpr size_t bytes = cmax(GjLay<Q, R>::bytes, GemmLay<Q, R>::bytes);
};

// HALF: the order is at most 16 Q - 8 (dual_gemm_half).
template <int Q, typename R, bool HALF>
__global__ void __launch_bounds__(kBlock) persist_kernel(DecimateArgs a) {
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ Common<Q> cm;
    __shared__ double red[kWaves];
    constexpr int NN = 16 * Q * 16 * Q;
    const int tid = threadIdx.x;
    const int n = a.n;
    const SlotWork<Q, R> w(a.work, blockIdx.x);
    for (;;) {
        if (setup_instance<Q, R, kBlock>(a, w, cm.s) == kDone) break;
        int ik;
        double2 z;
        instance_of(a, uniform(cm.s.t), ik, z);
        const double2 *H00 = a.hk + (size_t)ik * 2 * NN;
        for (;;) {
            const bool sing = gj_inverse<Q, R, kBlock>(lds, lds + GjLay<Q, R>::S, cm, w.es, w.et,
                                                       H00, z, n, 4, nullptr, w.g);
            if (tid == 0 && sing) cm.s.status |= 1;
            dual_gemm_any<Q, R, 0, HALF>(lds, red, w.al, w.be, w.g, n, w.m1, w.m2, nullptr);
            __syncthreads();
            dual_gemm_any<Q, R, 1, HALF>(lds, red, w.m1, w.m2, w.be, n, nullptr, w.be, w.es);
            __syncthreads();
            const double asum = dual_gemm_any<Q, R, 2, HALF>(lds, red, w.m2, w.m1, w.al, n, nullptr, w.al,
                                                   w.et);
            const int it = uniform(cm.s.it);
            const int converged = uniform(asum <= a.accuracy ? 1 : 0);
            __syncthreads();
            if (converged) break;
            if (it >= a.itermax) {
                if (tid == 0) cm.s.status |= 2;
                break;
            }
            if (tid == 0) cm.s.it = it + 1;
        }
        // G_LL = (z - eps_s)^-1, G_RR = (z - eps_t)^-1, G_B = (z - eps_i)^-1 in FP64
        for (int q = 0; q < 3; ++q) {
            double2 *full = a.gfull ? a.gfull + ((size_t)cm.s.t * 3 + q) * n * n : nullptr;
            const double2 *eps = q == 1 ? w.et : w.es;
            const double2 *eps2 = q == 2 ? w.et : nullptr;
            const bool sing = gj_inverse<Q, double, kBlock>(lds, lds + GjLay<Q, double>::S, cm,
                                                            eps, eps2, H00, z, n, full ? 2 : 1,
                                                            full, nullptr);
            if (tid == 0) {
                if (sing) cm.s.status |= 1;
                final_traces<Q>(a, cm, LdsInverse<Q>{lds, cm}, q, ik);
            }
            __syncthreads();
        }
    }
}

constexpr int kMaxQ = 24;
constexpr int kRoundsPerBatch = 8;

// Orders are padded to 16 Q (the pad rows and columns are exact zeros);
// kernels exist for Q = 1..5 (matrix in LDS) and Q = 6..24 (matrix in the
// slot's global workspace).  Q = 24 is the limit: the panel wave then holds
// six rows per lane (256 VGPRs), and the Gauss-Jordan kernel's LDS comes to
// 162,864 of the CU's 163,840 bytes.
int padded_q(int n) { return (n + 15) / 16; }
int decimate_max_q() { return kMaxQ; }

template <int Q, typename R>
static int launch_round(const DecimateArgs &a, int per_set, int set, bool gj, bool spread, hipStream_t s) {
    if constexpr (std::is_same_v<R, float> ? Q > 5 : Q <= 7) {
        // no FP32 kernels beyond order 80 (the C ABI refuses that case); FP64
        // rounds up to order 112 are mid.hip's
        return -1;
    } else if constexpr (Q <= 5) {
        constexpr size_t gj_lds = GjLay<Q, R>::bytes;
        if (gj)
            hipLaunchKernelGGL((gj_round_kernel<Q, R>), dim3(per_set), dim3(kGjBlock), gj_lds, s, a,
                               set * per_set);
        else if (Q >= 2 && a.n <= 16 * Q - 8)
            hipLaunchKernelGGL((gemm_round_kernel<Q, R, (Q >= 2)>), dim3(per_set), dim3(kBlock), 0,
                               s, a, set * per_set);
        else
            hipLaunchKernelGGL((gemm_round_kernel<Q, R, false>), dim3(per_set), dim3(kBlock), 0, s,
                               a, set * per_set);
    } else {
        constexpr size_t gj_lds = GjLayL<Q>::bytes;
        if (gj)
            hipLaunchKernelGGL((gj_large_round_kernel<Q, R>), dim3(per_set), dim3(kBlock), gj_lds, s,
                               a, set * per_set);
        else {
            constexpr int NBI = (Q + kBI - 1) / kBI;
            if (spread)
                hipLaunchKernelGGL((gemm_large_round_kernel<Q, R, true>),
                                   dim3((per_set + 7) / 8 * 8 * NBI), dim3(kBlock), 0, s, a,
                                   set * per_set, per_set);
            else
                hipLaunchKernelGGL((gemm_large_round_kernel<Q, R, false>), dim3(per_set), dim3(kBlock),
                                   0, s, a, set * per_set, per_set);
        }
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

#define WTSURF_FOR_EACH_Q(X) \
    X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15) X(16) X(17) X(18) X(19) X(20) \
        X(21) X(22) X(23) X(24)

template <typename R>
static int dispatch_round(const DecimateArgs &a, int q, int per_set, int set, bool gj, bool spread,
                          hipStream_t s) {
    switch (q) {
#define WTSURF_CASE(Q) \
    case Q: return launch_round<Q, R>(a, per_set, set, gj, spread, s);
        WTSURF_FOR_EACH_Q(WTSURF_CASE)
#undef WTSURF_CASE
        default: return -1;
    }
}

template <typename R>
static size_t dispatch_slot_bytes(int q) {
    switch (q) {
#define WTSURF_CASE(Q) \
    case Q: return Q <= 5 ? SlotWork<Q, R>::bytes : SlotWorkL<Q, R>::bytes;
        WTSURF_FOR_EACH_Q(WTSURF_CASE)
#undef WTSURF_CASE
        default: return 0;
    }
}

// Raise the dynamic-LDS limit of the Gauss-Jordan kernel to what it uses.  A
// runtime that does not need the call may refuse it; the launch itself then
// reports whether the size is accepted.
template <int Q, typename R>
static void allow_lds() {
    hipError_t e;
    if constexpr (Q <= 5 && std::is_same_v<R, float>)
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gj_round_kernel<Q, R>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)GjLay<Q, R>::bytes);
    else if constexpr (Q > 7 && std::is_same_v<R, double>)
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gj_large_round_kernel<Q, R>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)GjLayL<Q>::bytes);
    else
        return;
    if (e != hipSuccess) (void)hipGetLastError();
}

template <typename R>
static void dispatch_allow_lds(int q) {
    switch (q) {
#define WTSURF_CASE(Q) \
    case Q: allow_lds<Q, R>(); break;
        WTSURF_FOR_EACH_Q(WTSURF_CASE)
#undef WTSURF_CASE
        default: break;
    }
}

int decimate_slots_per_set(int ninst, int num_cu) {
    const int half = (ninst + 1) / 2;
    return half < num_cu ? (half > 0 ? half : 1) : num_cu;
}

size_t decimate_slot_bytes(int q, int precision) {
    return precision == 0 ? dispatch_slot_bytes<double>(q) : dispatch_slot_bytes<float>(q);
}

static int launch_phase(const DecimateArgs &a, int q, int precision, int per_set, int set, bool gj,
                        bool spread, hipStream_t s) {
    return precision == 0 ? dispatch_round<double>(a, q, per_set, set, gj, spread, s)
                          : dispatch_round<float>(a, q, per_set, set, gj, spread, s);
}

int decimate_run(const DecimateArgs &a, int q, int precision, int per_set, const RoundCtl &ctl) {
    constexpr int NS = kSlotSets;
    const hipStream_t s0 = ctl.s[0], sc = ctl.s[NS];
    const hipEvent_t start = ctl.ev[2 * NS + 2];
    if (precision == 0)
        dispatch_allow_lds<double>(q);
    else
        dispatch_allow_lds<float>(q);
    // An instance takes at most itermax (inverse, GEMMs) rounds plus four
    // inverse rounds (start, three finals); a slot runs ceil(ninst / slots)
    // instances.  Past that bound (with slack) the device has stopped making
    // progress and the run fails instead of launching rounds forever.
    const long slots = (long)NS * per_set;
    // Beyond order 112 a product or inverse workgroup fills its CU.  While one
    // set's inverses hold per_set CUs, the other's products have num_cu -
    // per_set: with fewer than 0.4 num_cu slots a set their row blocks are
    // spread over the CUs left (150 instances of order 288, 75 a set: 146 ->
    // 107 ms; one instance 117 -> 53), with more there is nothing to gain and
    // the operands are read again (300 of order 216 in halves: 96 -> 99 ms).
    const bool spread = 5 * per_set <= 2 * ctl.num_cu;
    const long per_slot = (a.ninst + slots - 1) / slots + 1;
    const long max_batches = per_slot * (a.itermax + 4) / kRoundsPerBatch + 4;
    if (hipMemsetAsync(a.state, 0, (size_t)slots * sizeof(SlotState), s0) != hipSuccess ||
        hipMemsetAsync(a.queue, 0, 2 * sizeof(unsigned), s0) != hipSuccess ||
        hipEventRecord(start, s0) != hipSuccess)
        return -1;
    for (int k = 1; k < NS; ++k)
        if (hipStreamWaitEvent(ctl.s[k], start, 0) != hipSuccess) return -1;
    // Stream k runs set k as (inverse, GEMMs) rounds for even k and (GEMMs,
    // inverse) for odd k: the sets stay half a round apart.  Each stream marks
    // the end of every batch of rounds with an event; the counter stream waits
    // for every set's mark of a batch and copies the finished-instance count
    // to pinned host memory, so the count it reports covers whole batches of
    // all sets whichever stream runs ahead, and the work streams never wait
    // for each other.  The host reads the count of the batch before while
    // this one runs, so the device never waits for the host.
    for (long b = 0;; ++b) {
        if (b > max_batches) return -2;
        for (int r = 0; r < kRoundsPerBatch; ++r)
            for (int k = 0; k < NS; ++k) {
                const bool gj_first = (k & 1) == 0;
                if (launch_phase(a, q, precision, per_set, k, gj_first, spread, ctl.s[k]) ||
                    launch_phase(a, q, precision, per_set, k, !gj_first, spread, ctl.s[k]))
                    return -1;
            }
        const int h = (int)(b & 1);
        for (int k = 0; k < NS; ++k)
            if (hipEventRecord(ctl.ev[2 * k + h], ctl.s[k]) != hipSuccess ||
                hipStreamWaitEvent(sc, ctl.ev[2 * k + h], 0) != hipSuccess)
                return -1;
        if (hipMemcpyAsync(ctl.pinned + h, a.queue + 1, sizeof(unsigned), hipMemcpyDeviceToHost, sc) !=
                hipSuccess ||
            hipEventRecord(ctl.ev[2 * NS + h], sc) != hipSuccess)
            return -1;
        if (b > 0) {
            if (hipEventSynchronize(ctl.ev[2 * NS + (h ^ 1)]) != hipSuccess) return -1;
            if (ctl.pinned[h ^ 1] >= (unsigned)a.ninst) break;
        }
    }
    for (int k = 1; k < NS; ++k)
        if (hipEventRecord(ctl.ev[2 * k], ctl.s[k]) != hipSuccess ||
            hipStreamWaitEvent(s0, ctl.ev[2 * k], 0) != hipSuccess)
            return -1;
    return 0;
}

template <int Q, typename R>
static int launch_persist(const DecimateArgs &a, int nblocks, hipStream_t s) {
    if constexpr (Q > 5) {
        return -1;  // orders beyond 80 run as rounds only
    } else {
        constexpr size_t lds = PersistLay<Q, R>::bytes;
        auto go = [&](auto kernel) {
            if (hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)lds) != hipSuccess)
                (void)hipGetLastError();  // the launch reports whether the size is accepted
            hipLaunchKernelGGL(kernel, dim3(nblocks), dim3(kBlock), lds, s, a);
        };
        if (Q >= 2 && a.n <= 16 * Q - 8)
            go(persist_kernel<Q, R, (Q >= 2)>);
        else
            go(persist_kernel<Q, R, false>);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
}

template <typename R>
static int dispatch_persist(const DecimateArgs &a, int q, int nblocks, hipStream_t s) {
    switch (q) {
        case 1: return launch_persist<1, R>(a, nblocks, s);
        case 2: return launch_persist<2, R>(a, nblocks, s);
        case 3: return launch_persist<3, R>(a, nblocks, s);
        case 4: return launch_persist<4, R>(a, nblocks, s);
        case 5: return launch_persist<5, R>(a, nblocks, s);
        default: return -1;
    }
}

int decimate_persistent_max_q() { return 5; }

int decimate_persistent_run(const DecimateArgs &a, int q, int precision, int nblocks,
                            hipStream_t s) {
    if (q < 1 || q > decimate_persistent_max_q() || nblocks < 1) return -1;
    if (hipMemsetAsync(a.queue, 0, 2 * sizeof(unsigned), s) != hipSuccess) return -1;
    return precision == 0 ? dispatch_persist<double>(a, q, nblocks, s)
                          : dispatch_persist<float>(a, q, nblocks, s);
}

}  // namespace wtsurf
