// k_daf.hip -- diagonalized approximate-factorization implicit operator.
//
// rhs_modal_matrices + rhs_diag_solver (src/rhs_modal_matrices.F90,
// src/rhs_diag_solver.F90).  Each direction D is one kernel, k_daf_sweep<D>:
// it loads the rows of its lines, applies the modal transform that precedes
// the sweep (S and Ma^-1 for i, N1^-1 = Mb^-1 Ma for j, N2^-1 = Mc^-1 Mb for k)
// as the rows arrive, solves the four scalar tridiagonal systems of every
// line and writes the solution; the k sweep applies Mc and adds dq to q
// instead (rhs_diag_solver.F90:624-633, solver_daf.F90:409-418).  The
// eigenvector matrices are rebuilt in registers from the metrics and dtau of
// each node instead of being stored (the reference keeps 67 words per node),
// and the line solves keep every row on chip.
//
// Line solve.  Thomas elimination is a pair of first-order recurrences,
//   c'_s = c_s / (b_s - a_s c'_(s-1)),  d'_s = (d_s - a_s d'_(s-1)) / den_s,
// and the back substitution x_s = d'_s - c'_s x_(s+1).  A workgroup owns TI
// lines and cuts each into P segments of at most R consecutive rows; the
// thread of a segment holds its rows in registers.  Each recurrence, seen as
// a map from the value entering a segment to the value leaving it, is a
// Moebius map (c') or an affine map (d', x) that the thread composes over its
// rows; one thread per (line, system) then walks the P segment maps in LDS to
// find the value entering every segment, and every thread runs the exact
// sequential recurrence over its own rows from there.  So each row is
// eliminated with the recurrence LAPACK SGTSV applies when it does not
// interchange rows, and the values at segment starts differ from a one-thread
// sweep only by rounding.  The three systems with distinct matrices are
// eliminated once each: systems 1 and 2 (eigenvalue 0) share theirs.
//
// SGTSV (src/sgtsv.f:89-259) interchanges rows where |den_s| < |a_(s+1)|;
// every sweep counts those rows in F.pivots (systems 1 and 2 each), so a
// caller sees when the pivot-free elimination left SGTSV's row order, and
// records the first row whose pivot den_s is zero or not finite (1-based, in
// line order) in F.zero_pivot, the INFO that SGTSV would return.
#include <algorithm>

#include "desalm_internal.h"

namespace desalm {

namespace {

// ---- modal matrices (rhs_modal_matrices.F90:112-264), applied in registers ----
// dtau-dependent factors of a node: sigma = sqrt(beta alpha) with
// alpha = 1 + e_source 1.5 dtau / delti, and theta = sqrt(beta / alpha) =
// beta / sigma (rhs_modal_matrices.F90:82-84)
//
// The FP64 form takes reciprocals and roots from the hardware estimates
// (rcp64 and its like, correctly rounded as the IEEE operations they stand for
// but for rare operands).  Roots to 1 ulp only moved the solution by rounding,
// and a network trained on such solutions by 1e-8 of its loss.  The sweeps
// spent up to half their time issuing instructions, two fifths of them
// divisions and roots: with these, and with the scaling of maps and the
// divisions of the c' scan moved out of its serial chain, i 124 -> 110 us,
// j 120 -> 109 us, k 150 -> 142 us on 193x129x129 and 15.7 -> 12.4 us for the
// k sweep of 49x33x33, where the chain is all there is.
// The FP32 form keeps the IEEE operations.  Its solves amplify any difference
// of the transformed rows (one ulp of FP64 changes which FP32 value a row
// rounds to), to 1e-9 of the solution within some thirty iterations, and
// although the helpers round as IEEE does, the compiler contracts the
// arithmetic around them otherwise: the FP64 form moved by rounding on
// curvilinear grids when it took them.
template <typename S>
struct Num {  // S = double
    static __device__ __forceinline__ double rcp(double x) { return rcp64(x); }
    static __device__ __forceinline__ double div(double a, double b) { return div64(a, b); }
    // sqrt(x) and 1 / sqrt(x)
    static __device__ __forceinline__ void root(double x, double& s, double& is) {
        root64(x, s, is);
    }
};
template <>
struct Num<float> {
    static __device__ __forceinline__ double rcp(double x) { return 1.0 / x; }
    static __device__ __forceinline__ double div(double a, double b) { return a / b; }
    static __device__ __forceinline__ void root(double x, double& s, double& is) {
        s = sqrt(x);
        is = 1.0 / s;
    }
};

struct NodeDt {
    double dt, alpha, sigma, isigma, theta;
};
template <typename S>
__device__ __forceinline__ NodeDt node_dt(const Consts& C, double dt) {
    NodeDt n;
    n.dt = dt;
    n.alpha = 1.0 + Num<S>::div(C.e_source * 1.5 * dt, C.delti);
    Num<S>::root(C.beta * n.alpha, n.sigma, n.isigma);
    n.theta = C.beta * n.isigma;
    return n;
}

// v <- M v for the Ma-type matrix of metric row (m1, m2, m3):
//   row 0 = (0, 0, sigma, sigma); rows 1-3 = (t1/s, t2/(s sg), m/sg, -m/sg)
//   with sg = |m|, s = sqrt(2 |m|^2 + (m2 - m3)^2)
template <typename S>
__device__ __forceinline__ void mul_m(double m1, double m2, double m3, double sigma, double v[4]) {
    const double g = m1 * m1 + m2 * m2 + m3 * m3;
    double sg, isg, s, is;
    Num<S>::root(g, sg, isg);
    Num<S>::root(2.0 * g + (m2 - m3) * (m2 - m3), s, is);
    const double w0 = v[0] * is, w1 = v[1] * (is * isg), u = (v[2] - v[3]) * isg;
    const double dm = m3 - m2;
    const double o0 = sigma * (v[2] + v[3]);
    const double o1 = -(m2 + m3) * w0 + m1 * dm * w1 + m1 * u;
    const double o2 = m1 * w0 + (g + m2 * dm) * w1 + m2 * u;
    const double o3 = m1 * w0 - (g - m3 * dm) * w1 + m3 * u;
    v[0] = o0; v[1] = o1; v[2] = o2; v[3] = o3;
}

// v <- M^-1 v for the same matrix, given g = |m|^2 and isg = 1 / |m| (the
// inverse in closed form, d = |m|^2 + 2 m2 m3 + m1^2)
template <typename S>
__device__ __forceinline__ void mul_minv(double m1, double m2, double m3, double g, double isg, double isigma,
                                         double v[4]) {
    const double m1s = m1 * m1, m2s = m2 * m2, m3s = m3 * m3;
    double s, is;
    Num<S>::root(2.0 * g + (m2 - m3) * (m2 - m3), s, is);
    const double id = Num<S>::rcp(g + 2.0 * m2 * m3 + m1s);
    const double r1 = m2 + m3, r2 = m2 - m3, r3 = m2s - m3s;
    const double o0 = s * id * (m1 * (v[2] + v[3]) - r1 * v[1]);
    const double o1 = s * isg * id *
                      (m1 * (m3 - m2) * v[1] + (m2 * m3 + m1s + m3s) * v[2] - (m2 * m3 + m1s + m2s) * v[3]);
    const double t = 0.5 * isigma * v[0];
    const double p = 0.5 * isg * id *
                     (m1 * (2.0 * g + 2.0 * m2 * m3 - m2s - m3s) * v[1] + (g * r1 + m1s * r2 + m3 * r3) * v[2] +
                      (g * r1 - m1s * r2 - m2 * r3) * v[3]);
    v[0] = o0; v[1] = o1; v[2] = t + p; v[3] = t - p;
}

// S (-dtau J rh) (rhs_diag_solver.F90:56-72): beta on the pressure row,
// 1 / alpha on the velocity rows
template <typename S>
__device__ __forceinline__ void scaled_rh_vals(const Consts& C, double aj, const double rh[4], const NodeDt& nd,
                                               double v[4]) {
    const double f = -nd.dt * aj;
    const double ia = Num<S>::rcp(nd.alpha);
    v[0] = C.beta * (f * rh[0]);
#pragma unroll
    for (int m = 1; m < 4; m++) v[m] = ia * (f * rh[m]);
}
template <typename S>
__device__ __forceinline__ void scaled_rh(const Fields& F, const Consts& C, long g, const NodeDt& nd, double v[4]) {
    const double rh[4] = {F.rh[0][g], F.rh[1][g], F.rh[2][g], F.rh[3][g]};
    scaled_rh_vals<S>(C, F.aj[g], rh, nd, v);
}

// the metric row of direction D at node g
template <int D>
__device__ __forceinline__ void metric_row(const Fields& F, long g, double& m1, double& m2, double& m3) {
    const double* const* mt = D == 0 ? F.csi : D == 1 ? F.eta : F.zet;
    m1 = mt[0][g]; m2 = mt[1][g]; m3 = mt[2][g];
}

// The modal transform that precedes sweep D (Ma^-1; N1^-1 = Mb^-1 Ma; N2^-1 =
// Mc^-1 Mb, applied factor by factor) of v at a node, from values already
// loaded: its dtau, the metric row a of direction D - 1 (unused for D = 0,
// whose v is S (-dtau J rh)) and the row m of D.  Returns dtau times the
// spectral radius of direction D, dtau theta |grad xi_D|
// (rhs_diag_solver.F90:149-160).
template <int D, typename S>
__device__ __forceinline__ double transform_vals(const NodeDt& nd, const double a[3], const double m[3], double v[4]) {
    if (D > 0) mul_m<S>(a[0], a[1], a[2], nd.sigma, v);
    const double g = m[0] * m[0] + m[1] * m[1] + m[2] * m[2];
    double sg, isg;
    Num<S>::root(g, sg, isg);
    mul_minv<S>(m[0], m[1], m[2], g, isg, nd.isigma, v);
    return nd.dt * (nd.theta * sg);
}
template <typename S>
__device__ __forceinline__ double sd_vals(const NodeDt& nd, const double m[3]) {
    double sg, isg;
    Num<S>::root(m[0] * m[0] + m[1] * m[1] + m[2] * m[2], sg, isg);
    return nd.dt * (nd.theta * sg);
}

template <int D, typename S>
__device__ __forceinline__ double transform_row(const Fields& F, const Consts& C, long g, double v[4]) {
    const NodeDt nd = node_dt<S>(C, F.dtau[g]);
    double a[3] = {0.0, 0.0, 0.0}, m[3];
    if (D > 0) metric_row<(D > 0 ? D - 1 : 0)>(F, g, a[0], a[1], a[2]);
    metric_row<D>(F, g, m[0], m[1], m[2]);
    return transform_vals<D, S>(nd, a, m, v);
}
template <int D, typename S>
__device__ __forceinline__ double row_sd(const Fields& F, const Consts& C, long g) {
    const NodeDt nd = node_dt<S>(C, F.dtau[g]);
    double m[3];
    metric_row<D>(F, g, m[0], m[1], m[2]);
    return sd_vals<S>(nd, m);
}

// the transform of sweep D alone (boundary vectors)
template <int D, typename S>
__device__ __forceinline__ void pre_transform(const Fields& F, const Consts& C, long g, double v[4]) {
    const NodeDt nd = node_dt<S>(C, F.dtau[g]);
    double a[3] = {0.0, 0.0, 0.0}, m[3];
    if (D > 0) metric_row<(D > 0 ? D - 1 : 0)>(F, g, a[0], a[1], a[2]);
    metric_row<D>(F, g, m[0], m[1], m[2]);
    (void)transform_vals<D, S>(nd, a, m, v);
}

// v <- Mc v at global node g (rhs_diag_solver.F90:624-633)
template <typename S>
__device__ __forceinline__ void apply_mc(const Consts& C, double dtau, double z1, double z2, double z3, double v[4]) {
    const NodeDt nd = node_dt<S>(C, dtau);
    mul_m<S>(z1, z2, z3, nd.sigma, v);
}

template <typename S>
struct SweepIO {
    const S* xin[4];  // j and k sweeps: the previous sweep's solution (level-local)
    S* xout[4];       // i and j sweeps: this sweep's solution (level-local)
};

struct SweepShape {
    int n;        // rows per line
    int P;        // segments per line
    int TI;       // lines per workgroup
    int nI;       // i positions of the j and k lines
    long nlines;
};

// values of one segment slot in LDS (the largest phase: 3 Moebius maps, 12
// values) rounded up to an odd count, and a line's slots padded to an odd
// count: the threads of adjacent segments, and the scanning threads of
// adjacent lines, then fall on different LDS banks
constexpr int kSlot = 13;
__host__ __device__ constexpr int line_stride(int P) { return (P * kSlot) | 1; }

// tridiagonal row of matrix mi (eigenvalue 0, +1, -1) from sd = dtau spr of
// the row's node and its two neighbours (rhs_diag_solver.F90:149-189); the
// characteristic-outlet row (ext) couples the +1 eigenvalue upwind only
// (:207-221)
template <typename S>
__device__ __forceinline__ void row_coef(int mi, S sdm, S sd0, S sdp, S h, S h2, S hsq, S epd, bool outlet, S& a,
                                         S& b, S& c) {
    const S lam = mi == 1 ? S(1) : mi == 2 ? S(-1) : S(0);
    if (outlet) {
        a = mi == 1 ? -(sdm * h) : S(0);
        b = mi == 1 ? S(1) + sd0 * h : S(1);
        c = S(0);
        return;
    }
    const S tmp = sd0 * epd * hsq;
    const S dtc = (sd0 == S(0)) ? S(0) : S(1);
    const S ddw = dtc * sdm * h2, dde = dtc * sdp * h2;
    a = -ddw * lam - tmp;
    c = dde * lam - tmp;
    b = S(1) + S(2) * tmp;
}

// matrix of system m: systems 0 and 1 share eigenvalue 0
__host__ __device__ constexpr int mat_of(int m) { return m < 2 ? 0 : m - 1; }

// scale a projective pair or map by a power of two (exact) so that its
// largest entry lies in [0.5, 1)
template <typename S>
__device__ __forceinline__ int pow2_exponent(S mx) {
    int e = 0;
    (void)frexp(mx, &e);
    return e;
}
template <typename S>
__device__ __forceinline__ void scale_map(S (&m)[4]) {
    const int e = -pow2_exponent(fmax(fmax(fabs(m[0]), fabs(m[1])), fmax(fabs(m[2]), fabs(m[3]))));
#pragma unroll
    for (int k = 0; k < 4; k++) m[k] = ldexp(m[k], e);
}
// rows composed between two scalings of a segment's map
template <typename S>
constexpr int kScaleRows = sizeof(S) == 8 ? 4 : 2;

// One direction's DAF line solves on level L.
//   D = 0: rows i = 1 .. ni-2 (+ the outlet plane when ext) of every (j, k)
//          line; input S (-dtau J rh) transformed by Ma^-1, output to xout.
//   D = 1: rows j of every (i, k) line; input xin transformed by N1^-1.
//   D = 2: rows k of every (i, j) line; input xin transformed by N2^-1;
//          the solution times Mc is added to q (and stored in dq_out when
//          given, level-local, 4 SoA).
// use_b1 / use_b2: the semi-explicit boundary vectors brh of the first and
// last rows (fine level, rhs_diag_solver.F90:87-135 and its j/k copies),
// built here by the threads of those rows.
template <int D, int R, typename S>
__device__ __forceinline__ void daf_body(const Level& L, const Fields& F, const Consts& C, const SweepIO<S>& io,
                                         const SweepShape& sh, int use_b1, int use_b2, int b2_full, int ext,
                                         double* dq_out, unsigned bid) {
    extern __shared__ double smem_d[];
    S* lds = reinterpret_cast<S*>(smem_d);
    const int P = sh.P, TI = sh.TI, n = sh.n;
    const int LS = line_stride(P);
    const int tid = (int)threadIdx.x;
    // i lines are contiguous: segments of one line on adjacent lanes; j and k
    // lines: adjacent lines (adjacent i) on adjacent lanes
    const int li = D == 0 ? tid / P : tid % TI;
    const int ps = D == 0 ? tid % P : tid / TI;
    const long t = (long)bid * TI + li;
    const bool act = t < sh.nlines;
    const int ni = L.ni, nj = L.nj, nk = L.nk;
    long base = 0, sD;
    if (D == 0) {
        sD = 1;
        if (act) base = (long)ni * ((1 + t % (nj - 2)) + (long)nj * (1 + t / (nj - 2)));
    } else if (D == 1) {
        sD = ni;
        if (act) base = (1 + t % sh.nI) + (long)ni * nj * (1 + t / sh.nI);
    } else {
        sD = (long)ni * nj;
        if (act) base = (1 + t % sh.nI) + (long)ni * (1 + t / sh.nI);
    }
    const int nd = D == 0 ? ni : D == 1 ? nj : nk;  // nodes along the line
    // the characteristic-outlet row closes the i lines only
    const bool outlet_lines = D == 0 && ext;
    const int s0 = ps * R;
    const int nr = act ? max(0, min(R, n - s0)) : 0;
    const S h = (S)(D == 0 ? L.dc : D == 1 ? L.de : L.dz);
    const S h2 = S(0.5) * h, hsq = h * h, epd = (S)C.ep[0][D];
    auto gnode = [&](int p) { return L.off + base + (long)p * sD; };  // global node at position p

    // ---- load: right-hand sides (transformed) and dtau spr of rows s0-1 .. s0+nr ----
    // window entry w is node position s0 + w (row s0 + w - 1)
    S dv[R][4];
    S sdv[R + 2];
    const int pe = s0 + nr + 1;  // the node after the segment
    if (D == 0) {
        // i lines: a segment's rows and its two window nodes are one run of
        // consecutive nodes, loaded as such (16-byte loads; lanes are R rows
        // apart).  The run of a partial last segment (or an idle thread)
        // reaches past the line's end into the next line or plane of the
        // level; those values are never used.
        double dt[R + 2], m1[R + 2], m2[R + 2], m3[R + 2], aj[R], rh[4][R];
#pragma unroll
        for (int w = 0; w < R + 2; w++) {
            const long g = gnode(s0 + w);
            dt[w] = F.dtau[g];
            m1[w] = F.csi[0][g];
            m2[w] = F.csi[1][g];
            m3[w] = F.csi[2][g];
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            const long g = gnode(s0 + r + 1);
            aj[r] = F.aj[g];
#pragma unroll
            for (int m = 0; m < 4; m++) rh[m][r] = F.rh[m][g];
        }
        // sdw[w]: dtau spr at window entry w; rows r < nr transformed
        double sdw[R + 2];
#pragma unroll
        for (int w = 0; w < R + 2; w++) {
            const NodeDt nd0 = node_dt<S>(C, dt[w]);
            const double mr[3] = {m1[w], m2[w], m3[w]};
            if (w >= 1 && w <= R) {
                const double rv[4] = {rh[0][w - 1], rh[1][w - 1], rh[2][w - 1], rh[3][w - 1]};
                double v[4];
                scaled_rh_vals<S>(C, aj[w - 1], rv, nd0, v);
                sdw[w] = transform_vals<0, S>(nd0, mr, mr, v);
                const bool in = w - 1 < nr;
#pragma unroll
                for (int m = 0; m < 4; m++) dv[w - 1][m] = in ? (S)v[m] : S(0);
            } else {
                sdw[w] = sd_vals<S>(nd0, mr);
            }
        }
        sdv[0] = nr > 0 ? (S)sdw[0] : S(0);
#pragma unroll
        for (int w = 1; w <= R + 1; w++) {
            // rows, then the node after the segment at entry nr + 1
            const bool row = w - 1 < nr;
            const bool after = w == nr + 1 && nr > 0 && pe <= nd - 1;
            sdv[w] = (row || after) ? (S)sdw[w] : S(0);
        }
    } else if (sizeof(S) == 4) {
        // FP32: one branch per row, 125 and 146 VGPRs and three waves per
        // SIMD (loaded ahead as below, 208 VGPRs and two waves, no faster)
#pragma unroll
        for (int r = 0; r < R; r++) {
            sdv[r + 1] = S(0);
#pragma unroll
            for (int m = 0; m < 4; m++) dv[r][m] = S(0);
            if (r < nr) {
                const int p = s0 + r + 1;
                double v[4];
                const long tl = base + (long)p * sD;
#pragma unroll
                for (int m = 0; m < 4; m++) v[m] = (double)io.xin[m][tl];
                sdv[r + 1] = (S)transform_row<D, S>(F, C, gnode(p), v);
#pragma unroll
                for (int m = 0; m < 4; m++) dv[r][m] = (S)v[m];
            }
        }
        sdv[0] = nr > 0 ? (S)row_sd<D, S>(F, C, gnode(s0)) : S(0);
        const S se = (nr > 0 && pe <= nd - 1) ? (S)row_sd<D, S>(F, C, gnode(pe)) : S(0);
        sdv[R + 1] = S(0);
#pragma unroll
        for (int w = 1; w <= R + 1; w++)
            if (w == nr + 1) sdv[w] = se;
    } else {
        // j and k lines: the loads of window entry w + 1 are in flight while
        // entry w is transformed, at addresses clamped to the line (no branch,
        // which would hold back the next row's loads; all rows' loads at once
        // would not fit the registers).  The last entry is the node after the
        // segment's rows, wherever they end.
        struct In {
            double dt, a[3], m[3], x[4];
        };
        auto load = [&](int w, In& o) {
            const long tl = base + (long)min(w <= R ? s0 + w : pe, nd - 1) * sD, g = L.off + tl;
            o.dt = F.dtau[g];
            metric_row<D>(F, g, o.m[0], o.m[1], o.m[2]);
            if (w >= 1 && w <= R) {
                metric_row<(D > 0 ? D - 1 : 0)>(F, g, o.a[0], o.a[1], o.a[2]);
#pragma unroll
                for (int m = 0; m < 4; m++) o.x[m] = (double)io.xin[m][tl];
            }
        };
        In cur, nxt;
        load(0, cur);
#pragma unroll
        for (int w = 0; w < R + 2; w++) {
            if (w + 1 < R + 2) load(w + 1, nxt);
            const NodeDt nd0 = node_dt<S>(C, cur.dt);
            if (w >= 1 && w <= R) {
                const bool in = w - 1 < nr;
                double v[4] = {cur.x[0], cur.x[1], cur.x[2], cur.x[3]};
                const double sd = transform_vals<D, S>(nd0, cur.a, cur.m, v);
                sdv[w] = in ? (S)sd : S(0);
#pragma unroll
                for (int m = 0; m < 4; m++) dv[w - 1][m] = in ? (S)v[m] : S(0);
            } else {
                const S sd = (S)sd_vals<S>(nd0, cur.m);
                if (w == 0) {
                    sdv[0] = nr > 0 ? sd : S(0);
                } else {
                    sdv[R + 1] = S(0);
#pragma unroll
                    for (int q = 1; q <= R + 1; q++)
                        if (q == nr + 1 && nr > 0 && pe <= nd - 1) sdv[q] = sd;
                }
            }
            cur = nxt;
        }
    }
    // semi-explicit boundary vectors of the first and last rows
    const bool first = act && s0 == 0 && nr > 0;
    const bool last = act && nr > 0 && s0 + nr == n;
    if (first && use_b1) {
        double w[4];
        const int b0 = 2 * D;
        if (D == 0) {
            double r1[4], r2[4];
            const long g1 = gnode(1), g2 = gnode(2);
            scaled_rh<S>(F, C, g1, node_dt<S>(C, F.dtau[g1]), r1);
            scaled_rh<S>(F, C, g2, node_dt<S>(C, F.dtau[g2]), r2);
#pragma unroll
            for (int m = 0; m < 4; m++) w[m] = C.sa[b0][m] * r1[m] + C.sb[b0][m] * r2[m];
        } else {
#pragma unroll
            for (int m = 0; m < 4; m++)
                w[m] = C.sa[b0][m] * (double)io.xin[m][base + sD] + C.sb[b0][m] * (double)io.xin[m][base + 2 * sD];
        }
        pre_transform<D, S>(F, C, gnode(0), w);
#pragma unroll
        for (int m = 0; m < 4; m++) {
            S am, bm, cm;
            row_coef<S>(mat_of(m), sdv[0], sdv[1], sdv[2], h, h2, hsq, epd, outlet_lines && n == 1, am, bm, cm);
            dv[0][m] = dv[0][m] - am * (S)w[m];
        }
    }
    if (last && use_b2) {
        double w[4] = {0.0, 0.0, 0.0, 0.0};
        const int b1 = 2 * D + 1;
        if (D == 0) {
            // the fifth product of sa(1:5,1) * rh(1:4, i, ...) (:97) lands in
            // brh(1,2,j,k) when the i = 1 vector is built; nothing else
            // writes brh(:,2) on a single rank (:102, :135), so it is used
            // as it is
            if (use_b1) {
                const long g2 = gnode(2), g3 = gnode(3);
                const double x2 = -F.dtau[g2] * F.rh[0][g2] * F.aj[g2];
                const double x3 = -F.dtau[g3] * F.rh[0][g3] * F.aj[g3];
                w[0] = C.sa[0][4] * (C.beta * x2) + C.sb[0][4] * (C.beta * x3);
            }
        } else if (D == 1 || b2_full) {
#pragma unroll
            for (int m = 0; m < 4; m++)
                w[m] = C.sa[b1][m] * (double)io.xin[m][base + (long)(nd - 2) * sD] +
                       C.sb[b1][m] * (double)io.xin[m][base + (long)(nd - 3) * sD];
            pre_transform<D, S>(F, C, gnode(nd - 1), w);
        } else if (use_b1) {
            // brh(:,2) is not rebuilt when btype(6) == 6 (:467) and keeps
            // the fifth product of the k = 1 build (:462), which reads rh(1)
            // of node i+1: the j sweep's solution there, zero on a boundary
            // node (rh is zeroed on the boundary planes before the DAF)
            const bool on_line = (int)(t % sh.nI) + 2 <= sh.nI;  // i + 1 is a j-line position
            const double x1 = on_line ? (double)io.xin[0][base + sD + 1] : 0.0;
            const double x2 = on_line ? (double)io.xin[0][base + 2 * sD + 1] : 0.0;
            w[0] = C.sa[4][4] * x1 + C.sb[4][4] * x2;
            pre_transform<D, S>(F, C, gnode(nd - 1), w);
        }
        const int r = nr - 1;
#pragma unroll
        for (int rr = 0; rr < R; rr++) {
            if (rr == r) {
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    S am, bm, cm;
                    row_coef<S>(mat_of(m), sdv[rr], sdv[rr + 1], sdv[rr + 2], h, h2, hsq, epd, outlet_lines, am, bm,
                                cm);
                    dv[rr][m] = dv[rr][m] - cm * (S)w[m];
                }
            }
        }
    }
    const bool outlet_row_here = outlet_lines && last;  // row n - 1 is the outlet row
    auto coef = [&](int r, int mi, S& a, S& b, S& c) {
        row_coef<S>(mi, sdv[r], sdv[r + 1], sdv[r + 2], h, h2, hsq, epd, outlet_row_here && r == nr - 1, a, b, c);
    };
    S* slot = lds + li * LS + ps * kSlot;
    const bool scanner = tid < 4 * TI;
    const int sl = tid / 4, sm = tid % 4;
    const bool scan_act = scanner && (long)bid * TI + sl < sh.nlines;
    S* sline = lds + sl * LS;  // the scanned line's slots

    // ---- phase A: Moebius maps of c' over the segment, scanned ----
    {
        S M[3][4];
#pragma unroll
        for (int mi = 0; mi < 3; mi++) { M[mi][0] = S(1); M[mi][1] = S(0); M[mi][2] = S(0); M[mi][3] = S(1); }
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (r < nr) {
#pragma unroll
                for (int mi = 0; mi < 3; mi++) {
                    S a, b, c;
                    coef(r, mi, a, b, c);
                    // [c'; 1] -> [c; b - a c']
                    const S n0 = c * M[mi][2], n1 = c * M[mi][3];
                    const S n2 = b * M[mi][2] - a * M[mi][0], n3 = b * M[mi][3] - a * M[mi][1];
                    M[mi][0] = n0; M[mi][1] = n1; M[mi][2] = n2; M[mi][3] = n3;
                }
            }
            // scaled every few rows: exact, and the entries grow by no more
            // than |a| + |b| + |c| per row (2 rows of FP32: up to 1e19 each)
            if (r % kScaleRows<S> == kScaleRows<S> - 1 || r == R - 1)
#pragma unroll
                for (int mi = 0; mi < 3; mi++) scale_map(M[mi]);
        }
#pragma unroll
        for (int mi = 0; mi < 3; mi++)
#pragma unroll
            for (int e = 0; e < 4; e++) slot[4 * mi + e] = M[mi][e];
    }
    __syncthreads();
    if (scan_act && sm < 3) {
        // projective pair (cn, cd): c' entering the segment is cn / cd
        S cn = S(0), cd = S(1);
        for (int sg0 = 0; sg0 < P; sg0 += 4) {
            S q[4][4];
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (sg0 + u < P)
#pragma unroll
                    for (int e = 0; e < 4; e++) q[u][e] = sline[(sg0 + u) * kSlot + 4 * sm + e];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                if (sg0 + u < P) {
                    // the pair itself: every segment's thread divides for its own
                    sline[(sg0 + u) * kSlot + 4 * sm] = cn;
                    sline[(sg0 + u) * kSlot + 4 * sm + 1] = cd;
                    const S nn = q[u][0] * cn + q[u][1] * cd, dd = q[u][2] * cn + q[u][3] * cd;
                    cn = nn;
                    cd = dd;
                }
            }
            const int e = -pow2_exponent(fmax(fabs(cn), fabs(cd)));
            cn = ldexp(cn, e);
            cd = ldexp(cd, e);
        }
    }
    __syncthreads();
    S cst[3];
#pragma unroll
    for (int mi = 0; mi < 3; mi++) cst[mi] = quot(slot[4 * mi], slot[4 * mi + 1]);

    // ---- phase B: exact c' over the rows (their 1 / den kept); affine maps of d', scanned ----
    S inv[R][3];
    unsigned piv = 0;
    int zrow = 0;  // first row (1-based in the line) with a zero or non-finite pivot
    {
        S U[4], V[4];
#pragma unroll
        for (int m = 0; m < 4; m++) { U[m] = S(0); V[m] = S(1); }
#pragma unroll
        for (int mi = 0; mi < 3; mi++) {
            S cprev = cst[mi];
#pragma unroll
            for (int r = 0; r < R; r++) {
                inv[r][mi] = S(0);
                if (r < nr) {
                    S a, b, c;
                    coef(r, mi, a, b, c);
                    const S den = b - a * cprev;
                    const S iv = recip(den);
                    inv[r][mi] = iv;
                    cprev = c * iv;
                    if (!(den != S(0) && isfinite(den)) && zrow == 0) zrow = s0 + r + 1;
                    // SGTSV's interchange test against the next row's subdiagonal
                    // (a depends on the row's sd and its lower neighbour's only)
                    if (s0 + r + 1 < n) {
                        S an, bn, cn;
                        row_coef<S>(mi, sdv[r + 1], sdv[r + 2], S(0), h, h2, hsq, epd, outlet_lines && s0 + r + 2 == n,
                                    an, bn, cn);
                        if (fabs(den) < fabs(an)) piv += mi == 0 ? 2u : 1u;
                    }
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        if (mat_of(m) == mi) {
                            const S v = -a * iv;
                            U[m] = dv[r][m] * iv + v * U[m];
                            V[m] = v * V[m];
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int m = 0; m < 4; m++) { slot[2 * m] = U[m]; slot[2 * m + 1] = V[m]; }
    }
    __syncthreads();
    if (scan_act) {
        S din = S(0);
        for (int sg0 = 0; sg0 < P; sg0 += 8) {
            S u[8], v[8];
#pragma unroll
            for (int k = 0; k < 8; k++)
                if (sg0 + k < P) { u[k] = sline[(sg0 + k) * kSlot + 2 * sm]; v[k] = sline[(sg0 + k) * kSlot + 2 * sm + 1]; }
#pragma unroll
            for (int k = 0; k < 8; k++) {
                if (sg0 + k < P) {
                    sline[(sg0 + k) * kSlot + 2 * sm] = din;
                    din = u[k] + v[k] * din;
                }
            }
        }
    }
    __syncthreads();

    // ---- phase C: exact d' over the rows; affine maps of x, scanned backwards ----
    {
        S dprev[4];
#pragma unroll
        for (int m = 0; m < 4; m++) dprev[m] = slot[2 * m];
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (r < nr) {
#pragma unroll
                for (int mi = 0; mi < 3; mi++) {
                    S a, b, c;
                    coef(r, mi, a, b, c);
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        if (mat_of(m) == mi) {
                            dprev[m] = (dv[r][m] - a * dprev[m]) * inv[r][mi];
                            dv[r][m] = dprev[m];
                        }
                    }
                }
            }
        }
        S A[4], B[4];
#pragma unroll
        for (int m = 0; m < 4; m++) { A[m] = S(0); B[m] = S(1); }
#pragma unroll
        for (int r = R - 1; r >= 0; r--) {
            if (r < nr) {
#pragma unroll
                for (int mi = 0; mi < 3; mi++) {
                    S a, b, c;
                    coef(r, mi, a, b, c);
                    const S cc = c * inv[r][mi];
                    inv[r][mi] = cc;  // c' from here on
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        if (mat_of(m) == mi) {
                            A[m] = dv[r][m] - cc * A[m];
                            B[m] = -cc * B[m];
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int m = 0; m < 4; m++) { slot[2 * m] = A[m]; slot[2 * m + 1] = B[m]; }
    }
    __syncthreads();
    if (scan_act) {
        S xin = S(0);
        for (int sg1 = P - 1; sg1 >= 0; sg1 -= 8) {
            S u[8], v[8];
#pragma unroll
            for (int k = 0; k < 8; k++)
                if (sg1 - k >= 0) { u[k] = sline[(sg1 - k) * kSlot + 2 * sm]; v[k] = sline[(sg1 - k) * kSlot + 2 * sm + 1]; }
#pragma unroll
            for (int k = 0; k < 8; k++) {
                if (sg1 - k >= 0) {
                    sline[(sg1 - k) * kSlot + 2 * sm] = xin;
                    xin = u[k] + v[k] * xin;
                }
            }
        }
    }
    __syncthreads();

    // ---- phase D: back substitution over the rows and the output ----
    S x[4];
#pragma unroll
    for (int m = 0; m < 4; m++) x[m] = slot[2 * m];
#pragma unroll
    for (int r = R - 1; r >= 0; r--) {
        if (r < nr) {
#pragma unroll
            for (int mi = 0; mi < 3; mi++) {
                const S cc = inv[r][mi];
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    if (mat_of(m) == mi) {
                        x[m] = dv[r][m] - cc * x[m];
                        dv[r][m] = x[m];
                    }
                }
            }
            if (D == 1 || (D == 0 && nr < R)) {
                const long tl = base + (long)(s0 + r + 1) * sD;
#pragma unroll
                for (int m = 0; m < 4; m++) io.xout[m][tl] = dv[r][m];
            }
        }
    }
    if (D == 0 && nr == R) {
        // a whole segment of an i line: one run of consecutive nodes per
        // component
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
            for (int r = 0; r < R; r++) io.xout[m][base + s0 + r + 1] = dv[r][m];
    }
    if (D == 2) {
        // Mc and the q update, four rows at a time: the loads of a group are
        // all in flight, and every value formed, before its first store (rows
        // past the line's end read its last row and are not stored)
#pragma unroll
        for (int r0 = 0; r0 < R; r0 += 4) {
            double v[4][4], qv[4][4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const long g = L.off + base + (long)(min(s0 + r0 + u, n - 1) + 1) * sD;
                const double dt = F.dtau[g], z1 = F.zet[0][g], z2 = F.zet[1][g], z3 = F.zet[2][g];
#pragma unroll
                for (int m = 0; m < 4; m++) qv[u][m] = F.q[m][g];
#pragma unroll
                for (int m = 0; m < 4; m++) v[u][m] = (double)dv[r0 + u][m];
                apply_mc<S>(C, dt, z1, z2, z3, v[u]);
#pragma unroll
                for (int m = 0; m < 4; m++) qv[u][m] = qv[u][m] + v[u][m];
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int r = r0 + u;
                if (r < nr) {
                    const long tl = base + (long)(s0 + r + 1) * sD;
#pragma unroll
                    for (int m = 0; m < 4; m++) F.q[m][L.off + tl] = qv[u][m];
                    if (dq_out) {
#pragma unroll
                        for (int m = 0; m < 4; m++) dq_out[m * L.n + tl] = v[u][m];
                    }
                }
            }
        }
    }
    if (piv) atomicAdd(F.pivots, (unsigned long long)piv);
    if (zrow) atomicMin(F.zero_pivot, (unsigned)zrow);
}

// the boundary-vector flags and the line shape of direction D on level n
// (the i lines take the characteristic-outlet row when ext); P and TI are
// the launch's
struct SweepFlags {
    int use_b1, use_b2, b2_full, ext;
};
__host__ __device__ inline SweepFlags sweep_flags(const Consts& C, int D, int n) {
    SweepFlags f;
    f.use_b1 = (n == 1 && C.btype[2 * D] != 5);
    f.use_b2 = (n == 1 && C.btype[2 * D + 1] != 5);
    f.b2_full = (n == 1 && C.btype[5] != 6);
    // a characteristic outlet at i = ni - 1 joins the fine level's sweeps
    f.ext = (n == 1 && C.btype[1] == DESALM_BC_OUTLET_MOC);
    return f;
}
__host__ __device__ inline int sweep_len(const Level& L, int D, int ext) {
    return D == 0 ? L.ni - 2 + ext : D == 1 ? L.nj - 2 : L.nk - 2;
}
__host__ __device__ inline SweepShape sweep_lines(const Level& L, int D, int ext, int P, int TI) {
    SweepShape sh;
    sh.nI = L.ni - 2 + ext;
    sh.n = sweep_len(L, D, ext);
    sh.nlines = D == 0 ? (long)(L.nj - 2) * (L.nk - 2) : D == 1 ? (long)sh.nI * (L.nk - 2) : (long)sh.nI * (L.nj - 2);
    sh.P = P;
    sh.TI = TI;
    return sh;
}
// segments per line and lines per workgroup for lines of up to len rows
__host__ __device__ inline void sweep_tiles(int D, int len, int R, int& P, int& TI) {
    P = (len + R - 1) / R;
    if (P < 4) P = 4;
    // j and k lines: 16 adjacent i lines per workgroup (128-byte rows; the
    // partial cache lines at a run's ends are shared with the neighbouring
    // workgroups, which run on the same XCD).  A 256-thread workgroup leaves
    // room for a second one on the CU at up to 256 VGPRs.
    TI = D == 0 ? (256 / P > 1 ? 256 / P : 1) : 16;
    while (TI * P > 512 && TI > 1) TI /= 2;
}

// the solution of the i sweep goes to F.dp, of the j sweep to F.cp
// (level-local); the mixed form uses their FP32 counterparts
template <typename S>
__host__ __device__ inline SweepIO<S> sweep_io(const Fields& F, int D);
template <>
__host__ __device__ inline SweepIO<double> sweep_io<double>(const Fields& F, int D) {
    SweepIO<double> io;
    for (int m = 0; m < 4; m++) {
        io.xin[m] = D == 1 ? F.dp[m] : F.cp[m];
        io.xout[m] = D == 0 ? F.dp[m] : F.cp[m];
    }
    return io;
}
template <>
__host__ __device__ inline SweepIO<float> sweep_io<float>(const Fields& F, int D) {
    SweepIO<float> io;
    for (int m = 0; m < 4; m++) {
        io.xin[m] = D == 1 ? F.dpf[m] : F.cpf[m];
        io.xout[m] = D == 0 ? F.dpf[m] : F.cpf[m];
    }
    return io;
}

template <int D, int R, typename S>
__global__ void __launch_bounds__(512) k_daf_sweep(Level L, Fields F, Consts C, SweepIO<S> io, SweepShape sh,
                                                  int use_b1, int use_b2, int b2_full, int ext, double* dq_out) {
    daf_body<D, R, S>(L, F, C, io, sh, use_b1, use_b2, b2_full, ext, dq_out, xcd_block(blockIdx.x, gridDim.x));
}

// every zone of a group in one launch; P and TI are the launch's (from the
// longest line of any zone): a zone's shorter lines leave trailing segments
// empty, which pass the scanned maps through unchanged
template <int D, int R, typename S>
__global__ void __launch_bounds__(512) k_daf_sweep_z(ZoneGrid G, int n, int P, int TI) {
    const ZoneBlock b = zone_block(G);
    const ZoneDesc& Z = G.z[b.z];
    const Level L = Z.lv[n];
    const Fields F = Z.F;
    const Consts C = Z.C;
    const SweepFlags f = sweep_flags(C, D, n);
    daf_body<D, R, S>(L, F, C, sweep_io<S>(F, D), sweep_lines(L, D, f.ext, P, TI), f.use_b1, f.use_b2,
                      f.b2_full, f.ext, nullptr, xcd_block(b.bid, b.nblk));
}

// ---- batched LAPACK SGTSV (src/sgtsv.f:89-259) in FP64, one system per thread ----
//
// A system's rows are consecutive in memory, so the threads of a wave, one
// system each, are n rows apart: read straight from memory every row cost a
// latency of its own and every access a cache line per thread (2048 systems of
// 127 rows: 256 us; 16129 of 191: 485 us).  A wave of 64 systems instead moves
// chunks of kGtRows rows through LDS, in runs of 128 bytes per system, loads
// the next chunk while it eliminates the current one, and keeps the row that
// the next row's elimination changes in registers.  Bound by the serial chain
// of the recurrence (a division and two multiply-adds per row and direction):
// 2048 systems of 127 rows 83 us, 16129 of 191 131 us.
constexpr int kGtRows = 16, kGtLd = kGtRows + 1;

__global__ void __launch_bounds__(64) k_gtsv_batch(int n, int nsys, double* dl, double* d, double* du, double* b,
                                                   int* info) {
    __shared__ double lds[4][64][kGtLd];
    const int lane = (int)threadIdx.x;
    const long s0 = (long)blockIdx.x * 64;
    const bool act = s0 + lane < nsys;
    const int ls = lane / kGtRows, lr = lane % kGtRows;  // system and row of this lane's loads and stores
    constexpr int NQ = kGtRows;
    double* const arr[4] = {dl, d, du, b};
    // rows c0 .. of every system of the wave; past the end the last row or
    // system again
    double v[4][NQ];
    auto load = [&](int c0) {
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            const long sys = min(s0 + ls + 64 / kGtRows * q, (long)nsys - 1);
            const long g = sys * n + max(0, min(c0 + lr, n - 1));
#pragma unroll
            for (int k = 0; k < 4; k++) v[k][q] = arr[k][g];
        }
    };
    auto to_lds = [&] {
#pragma unroll
        for (int q = 0; q < NQ; q++)
#pragma unroll
            for (int k = 0; k < 4; k++) lds[k][ls + 64 / kGtRows * q][lr] = v[k][q];
    };
    // forward elimination: row r - 1 is finished by row r
    int inf = 0;
    double L0 = 0.0, D0 = 0.0, U0 = 0.0, B0 = 0.0;  // row r - 1
    load(0);
    for (int c0 = 0; c0 < n; c0 += kGtRows) {
        to_lds();
        __syncthreads();
        load(c0 + kGtRows);
        const int nr = min(kGtRows, n - c0);
        for (int r = 0; r < nr; r++) {
            const int row = c0 + r;
            const double L1 = lds[0][lane][r];
            double D1 = lds[1][lane][r], U1 = lds[2][lane][r], B1 = lds[3][lane][r];
            if (row > 0) {
                const bool last = row == n - 1;  // the last elimination has no DU of its second row
                if (!inf) {
                    if (fabs(D0) >= fabs(L0)) {
                        if (D0 != 0.0) {
                            const double fact = L0 / D0;
                            D1 = D1 - fact * U0;
                            B1 = B1 - fact * B0;
                            if (!last) L0 = 0.0;
                        } else {
                            inf = row;
                        }
                    } else {
                        const double fact = D0 / L0;
                        D0 = L0;
                        const double td = D1, tb = B0;
                        D1 = U0 - fact * td;
                        if (!last) {
                            L0 = U1;
                            U1 = -fact * L0;
                        }
                        U0 = td;
                        B0 = B1;
                        B1 = tb - fact * B1;
                    }
                }
                if (r > 0) {
                    lds[0][lane][r - 1] = L0;
                    lds[1][lane][r - 1] = D0;
                    lds[2][lane][r - 1] = U0;
                    lds[3][lane][r - 1] = B0;
                } else if (act) {  // the chunk before is stored already, without its last row
                    const long g = (s0 + lane) * n + row - 1;
                    dl[g] = L0;
                    d[g] = D0;
                    du[g] = U0;
                    b[g] = B0;
                }
            }
            L0 = L1;
            D0 = D1;
            U0 = U1;
            B0 = B1;
        }
        const bool end = c0 + nr == n;
        if (end) {
            lds[0][lane][nr - 1] = L0;
            lds[1][lane][nr - 1] = D0;
            lds[2][lane][nr - 1] = U0;
            lds[3][lane][nr - 1] = B0;
        }
        __syncthreads();
        if (lr < (end ? nr : nr - 1)) {
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                const int sys = ls + 64 / kGtRows * q;
                if (s0 + sys < nsys) {
                    const long g = (s0 + sys) * n + c0 + lr;
#pragma unroll
                    for (int k = 0; k < 4; k++) arr[k][g] = lds[k][sys][lr];
                }
            }
        }
        __syncthreads();
    }
    if (!inf && D0 == 0.0) inf = n;
    if (act && info) info[s0 + lane] = inf;
    // back substitution, last chunk first; a system with INFO > 0 keeps its b
    __threadfence_block();
    __syncthreads();
    double x1 = 0.0, x2 = 0.0;  // of rows r + 1 and r + 2
    const int cl = (n - 1) / kGtRows * kGtRows;
    load(cl);
    for (int c0 = cl; c0 >= 0; c0 -= kGtRows) {
        to_lds();
        __syncthreads();
        load(c0 - kGtRows);
        for (int r = min(kGtRows, n - c0) - 1; r >= 0 && !inf; r--) {
            const int row = c0 + r;
            const double Dr = lds[1][lane][r], Br = lds[3][lane][r];
            double x;
            if (row == n - 1) x = Br / Dr;
            else if (row == n - 2) x = (Br - lds[2][lane][r] * x1) / Dr;
            else x = (Br - lds[2][lane][r] * x1 - lds[0][lane][r] * x2) / Dr;
            lds[3][lane][r] = x;
            x2 = x1;
            x1 = x;
        }
        __syncthreads();
        if (c0 + lr < n) {
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                const int sys = ls + 64 / kGtRows * q;
                if (s0 + sys < nsys) b[(s0 + sys) * n + c0 + lr] = lds[3][sys][lr];
            }
        }
        __syncthreads();
    }
}

}  // namespace

template <int D, typename S>
static void daf_sweep(hipStream_t s, const Level& L, const Fields& F, const Consts& C, int n, double* dq_out) {
    const SweepFlags f = sweep_flags(C, D, n);
    const int len = sweep_len(L, D, f.ext);
    // i lines: short segments (their rows are adjacent in memory, so lanes
    // reading row r of adjacent segments are R rows apart)
    const int R = (D == 0 || len <= 64) ? 4 : 8;
    int P = 0, TI = 0;
    sweep_tiles(D, len, R, P, TI);
    const SweepShape sh = sweep_lines(L, D, f.ext, P, TI);
    const unsigned nb = (unsigned)((sh.nlines + sh.TI - 1) / sh.TI);
    const size_t lds = sizeof(S) * (size_t)sh.TI * line_stride(sh.P);
    const SweepIO<S> io = sweep_io<S>(F, D);
    if (R == 4)
        hipLaunchKernelGGL((k_daf_sweep<D, 4, S>), dim3(nb), dim3(sh.TI * sh.P), lds, s, L, F, C, io, sh, f.use_b1,
                           f.use_b2, f.b2_full, f.ext, dq_out);
    else
        hipLaunchKernelGGL((k_daf_sweep<D, 8, S>), dim3(nb), dim3(sh.TI * sh.P), lds, s, L, F, C, io, sh, f.use_b1,
                           f.use_b2, f.b2_full, f.ext, dq_out);
}

template <int D, typename S>
static void daf_sweep_z(hipStream_t s, const ZoneList& Z, int n) {
    int len = 0;
    for (const ZoneDesc& z : Z.host) len = std::max(len, sweep_len(z.lv[n], D, sweep_flags(z.C, D, n).ext));
    const int R = (D == 0 || len <= 64) ? 4 : 8;
    int P = 0, TI = 0;
    sweep_tiles(D, len, R, P, TI);
    unsigned nb = 0;
    const ZoneGrid G = Z.grid(
        [&](const ZoneDesc& z) {
            const SweepShape sh = sweep_lines(z.lv[n], D, sweep_flags(z.C, D, n).ext, P, TI);
            return (unsigned)((sh.nlines + TI - 1) / TI);
        },
        nb);
    const size_t lds = sizeof(S) * (size_t)TI * line_stride(P);
    if (R == 4)
        hipLaunchKernelGGL((k_daf_sweep_z<D, 4, S>), dim3(nb), dim3(TI * P), lds, s, G, n, P, TI);
    else
        hipLaunchKernelGGL((k_daf_sweep_z<D, 8, S>), dim3(nb), dim3(TI * P), lds, s, G, n, P, TI);
}

template <int D>
static void daf_dir(hipStream_t s, const Level& L, const Fields& F, const Consts& C, int n, double* dq_out) {
    if (C.mixed) daf_sweep<D, float>(s, L, F, C, n, dq_out);
    else daf_sweep<D, double>(s, L, F, C, n, dq_out);
}

// the sweep of direction D on level n over every zone of a group in one
// launch (the zones share the precision form)
void launch_daf_z(hipStream_t s, const ZoneList& Z, int n, int D) {
    const bool f = Z.host[0].C.mixed;
    if (D == 0) f ? daf_sweep_z<0, float>(s, Z, n) : daf_sweep_z<0, double>(s, Z, n);
    else if (D == 1) f ? daf_sweep_z<1, float>(s, Z, n) : daf_sweep_z<1, double>(s, Z, n);
    else f ? daf_sweep_z<2, float>(s, Z, n) : daf_sweep_z<2, double>(s, Z, n);
}

void launch_daf_i(hipStream_t s, const Level& L, const Fields& F, const Consts& C, int n) {
    daf_dir<0>(s, L, F, C, n, nullptr);
}

void launch_daf_j(hipStream_t s, const Level& L, const Fields& F, const Consts& C, int n) {
    daf_dir<1>(s, L, F, C, n, nullptr);
}

void launch_daf_k(hipStream_t s, const Level& L, const Fields& F, const Consts& C, int n, double* dq_out) {
    daf_dir<2>(s, L, F, C, n, dq_out);
}

void launch_gtsv_batch(hipStream_t s, int n, int nsys, double* dl, double* d, double* du, double* b, int* info) {
    hipLaunchKernelGGL(k_gtsv_batch, dim3((unsigned)((nsys + 63) / 64)), dim3(64), 0, s, n, nsys, dl, d, du, b, info);
}

}  // namespace desalm
