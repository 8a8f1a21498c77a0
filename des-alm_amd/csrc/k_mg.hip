// k_mg.hip -- FAS multigrid transfers, fine-grid boundary conditions,
// update norms and layout conversion.
//
//   k_inject        mg_inject (src/mg_inject.F90:2-64)
//   k_nlevel        mg_nlevel: injection of q, xnut, qold_mg and the 27-point
//                   restriction of rh into pk (src/mg_nlevel.F90:2-150),
//                   boundary pk zeroed (mg_zero_pk_boundary)
//   k_rs_sweep<D>   rs_sweep constant-coefficient smoothing sweeps
//                   (src/rs_sweep.F90:59-178) with every row on chip; the
//                   i sweep forms mg_prolong's coarse correction q - qold_mg
//                   and its k/j/i linear fills (src/mg_prolong.F90:57-170) as
//                   it loads, the k sweep adds dq to q
//   k_bc_fm         bcond_fm faces (src/bcond_fm.F90:79-306), k_pfix_*
//                   the pinned-pressure shift (:310-322)
//   k_resid_*       mg_residual's L1 update norms (src/mg_residual.F90:58-67)
#include "desalm_internal.h"
#include "seg_sweep.h"

namespace desalm {

namespace {

__device__ __forceinline__ long lidx(const Level& L, int i, int j, int k) {
    return (long)i + (long)L.ni * ((long)j + (long)L.nj * k);
}

inline long lidx_h(const Level& L, int i, int j, int k) { return (long)i + (long)L.ni * ((long)j + (long)L.nj * k); }

// coarse node (i,j,k) -> coincident fine node, 0-based (fine 1-based index
// 2^crs * i - crs of src/mg_nlevel.F90:22-24)
__device__ __forceinline__ int c2f(int i, int crs) { return crs ? 2 * i : i; }

__global__ void k_inject(Level Lc, Level Lf, double* const* comps, int ncomp, int icrs, int jcrs, int kcrs) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= Lc.n) return;
    const int i = (int)(t % Lc.ni), j = (int)((t / Lc.ni) % Lc.nj), k = (int)(t / ((long)Lc.ni * Lc.nj));
    const long gf = Lf.off + lidx(Lf, c2f(i, icrs), c2f(j, jcrs), c2f(k, kcrs));
    const long gc = Lc.off + t;
    for (int m = 0; m < ncomp; m++) comps[m][gc] = comps[m][gf];
}

struct Ptrs {
    double* p[16];
};

__global__ void k_inject_p(Level Lc, Level Lf, Ptrs P, int ncomp, int icrs, int jcrs, int kcrs) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= Lc.n) return;
    const int i = (int)(t % Lc.ni), j = (int)((t / Lc.ni) % Lc.nj), k = (int)(t / ((long)Lc.ni * Lc.nj));
    const long gf = Lf.off + lidx(Lf, c2f(i, icrs), c2f(j, jcrs), c2f(k, kcrs));
    const long gc = Lc.off + t;
    for (int m = 0; m < ncomp; m++) P.p[m][gc] = P.p[m][gf];
}

__device__ __forceinline__ void nlevel_body(const Level& Lc, const Level& Lf, const Fields& F, int icrs, int jcrs,
                                            int kcrs, unsigned bid, unsigned nb) {
    const long t = (long)xcd_block(bid, nb) * blockDim.x + threadIdx.x;
    if (t >= Lc.n) return;
    const int ni = Lc.ni, nj = Lc.nj, nk = Lc.nk;
    const int i = (int)(t % ni), j = (int)((t / ni) % nj), k = (int)(t / ((long)ni * nj));
    const long ll = Lf.off + lidx(Lf, c2f(i, icrs), c2f(j, jcrs), c2f(k, kcrs));
    const long l = Lc.off + t;
    // loads before stores throughout, so that they are in flight together
    double v[4];
#pragma unroll
    for (int m = 0; m < 4; m++) v[m] = F.q[m][ll];
    const double xn = F.xnut[ll];
#pragma unroll
    for (int m = 0; m < 4; m++) {
        F.q[m][l] = v[m];
        F.qold[m][l] = v[m];
    }
    F.xnut[l] = xn;
    if (i == 0 || i == ni - 1 || j == 0 || j == nj - 1 || k == 0 || k == nk - 1) {
        // the reference evaluates these from out-of-level neighbours and then
        // zeroes them (src/mg_driver.F90:134)
#pragma unroll
        for (int m = 0; m < 4; m++) F.pk[m][l] = 0.0;
        return;
    }
    const long ic = 1, ie = Lf.ni, iz = (long)Lf.ni * Lf.nj;
    double pkv[4];
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const double* r = F.rh[m] + ll;
        pkv[m] = (0.25 * r[ic + ie + iz] + 0.5 * r[ic + ie] + 0.25 * r[ic + ie - iz] +
                   0.5 * r[ie + iz] + r[ie] + 0.5 * r[ie - iz] +
                   0.25 * r[-ic + ie + iz] + 0.5 * r[-ic + ie] + 0.25 * r[-ic + ie - iz] +
                   0.5 * r[ic + iz] + r[ic] + 0.5 * r[ic - iz] +
                   r[iz] + 2.0 * r[0] + r[-iz] +
                   0.5 * r[-ic + iz] + r[-ic] + 0.5 * r[-ic - iz] +
                   0.25 * r[ic - ie + iz] + 0.5 * r[ic - ie] + 0.25 * r[ic - ie - iz] +
                   0.5 * r[-ie + iz] + r[-ie] + 0.5 * r[-ie - iz] +
                   0.25 * r[-ic - ie + iz] + 0.5 * r[-ic - ie] + 0.25 * r[-ic - ie - iz]) *
                  (1.0 / 16.0);
    }
#pragma unroll
    for (int m = 0; m < 4; m++) F.pk[m][l] = pkv[m];
}

__global__ void k_zero_pk_boundary(Level L, Fields F) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= L.n) return;
    const int ni = L.ni, nj = L.nj, nk = L.nk;
    const int i = (int)(t % ni), j = (int)((t / ni) % nj), k = (int)(t / ((long)ni * nj));
    if (i == 0 || i == ni - 1 || j == 0 || j == nj - 1 || k == 0 || k == nk - 1) {
#pragma unroll
        for (int m = 0; m < 4; m++) F.pk[m][L.off + t] = 0.0;
    }
}

// ---- prolongation ----
struct ProlongCtx {
    Level Lf, Lc;
    int icrs, jcrs, kcrs;
};

// The coarse correction q - qold_mg (mg_prolong.F90:57-75) filled linearly
// onto R fine nodes i = s0 + 1 .. of the line (jf, kf) for the i sweep: k, then
// j, then i (mg_prolong.F90:82-161).  A fine node coincident with a coarse node
// in a direction takes it, one between two coarse nodes takes half of each: the
// same operands in the same order as the reference's fills (halves are exact,
// so the order alone fixes the bits).  The sweep reads the coarse nodes
// straight (an eighth as many, shared by neighbouring lines in L2) instead of
// a filled field that a launch of its own wrote: prolongation 197 -> 188 us on
// 193x129x129, and one launch less per level.
template <int R>
__device__ __forceinline__ void fill_rows(const ProlongCtx& P, const Fields& F, int jf, int kf, int s0, double (&w)[R][4]) {
    const Level& Lc = P.Lc;
    const bool jodd = P.jcrs && (jf & 1), kodd = P.kcrs && (kf & 1);
    const int jl = P.jcrs ? jf >> 1 : jf, kl = P.kcrs ? kf >> 1 : kf;
    const long sJ = Lc.ni, sK = (long)Lc.ni * Lc.nj;
    const long line = Lc.off + sJ * jl + sK * kl;
    // coarse node c of the row, j and k filled
    auto node = [&](int c, double (&f)[4]) {
        const long l = line + min(c, Lc.ni - 1);
        auto corr = [&](long g, double (&v)[4]) {
#pragma unroll
            for (int m = 0; m < 4; m++) v[m] = F.q[m][g] - F.qold[m][g];
        };
        auto kfill = [&](long g, double (&v)[4]) {
            corr(g, v);
            if (kodd) {
                double h[4];
                corr(g + sK, h);
#pragma unroll
                for (int m = 0; m < 4; m++) v[m] = 0.5 * h[m] + 0.5 * v[m];
            }
        };
        kfill(l, f);
        if (jodd) {
            double h[4];
            kfill(l + sJ, h);
#pragma unroll
            for (int m = 0; m < 4; m++) f[m] = 0.5 * h[m] + 0.5 * f[m];
        }
    };
    if (P.icrs) {
        // rows i = s0 + 1 (between), s0 + 2 (coincident), ...: coarse nodes
        // s0 / 2 .. (s0 + R) / 2 (s0 and R are even)
        double f[R / 2 + 1][4];
#pragma unroll
        for (int u = 0; u <= R / 2; u++) node(s0 / 2 + u, f[u]);
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int m = 0; m < 4; m++)
                w[r][m] = r % 2 == 0 ? 0.5 * f[r / 2 + 1][m] + 0.5 * f[r / 2][m] : f[r / 2 + 1][m];
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) node(s0 + 1 + r, w[r]);
    }
}

// rs_sweep in direction D on the interior of a level (src/rs_sweep.F90:59-178):
// the constant system (-ep, 1+2ep, -ep) applied to the four components of dq
// (F.dp, level-local) with every row on chip (seg_sweep.h), solved in place;
// D = 2 adds the result to q instead.  The reference calls SGTSV with four
// right-hand sides; this is its non-interchanging elimination.
template <int D, int R>
__device__ __forceinline__ void rs_sweep_body(const ProlongCtx& PC, const Fields& F, const SegShape& sh, double epn,
                                              unsigned bid) {
    const Level& L = PC.Lf;
    extern __shared__ double smem_rs[];
    const int P = sh.P, TI = sh.TI, n = sh.n;
    const int tid = (int)threadIdx.x;
    const int li = D == 0 ? tid / P : tid % TI;
    const int ps = D == 0 ? tid % P : tid / TI;
    const long line0 = (long)bid * TI;
    const long t = line0 + li;
    const bool act = t < sh.nlines;
    const int ni = L.ni, nj = L.nj;
    long base = 0, sD;
    if (D == 0) {
        sD = 1;
        if (act) base = (long)ni * ((1 + t % (nj - 2)) + (long)nj * (1 + t / (nj - 2)));
    } else if (D == 1) {
        sD = ni;
        if (act) base = (1 + t % (ni - 2)) + (long)ni * nj * (1 + t / (ni - 2));
    } else {
        sD = (long)ni * nj;
        if (act) base = (1 + t % (ni - 2)) + (long)ni * (1 + t / (ni - 2));
    }
    const int s0 = ps * R;
    const int nr = act ? max(0, min(R, n - s0)) : 0;
    double a[R], b[R], c[R], d[R][4];
#pragma unroll
    for (int r = 0; r < R; r++) {
        a[r] = -epn;
        b[r] = 1.0 + 2.0 * epn;
        c[r] = -epn;
    }
    if (D == 0) {
        // i lines: the coarse correction, filled here
        double w[R][4];
        fill_rows<R>(PC, F, act ? (int)(1 + t % (nj - 2)) : 1, act ? (int)(1 + t / (nj - 2)) : 1, s0, w);
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int m = 0; m < 4; m++) d[r][m] = r < nr ? w[r][m] : 0.0;
    } else {
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int m = 0; m < 4; m++) d[r][m] = r < nr ? F.dp[m][base + (long)(s0 + r + 1) * sD] : 0.0;
    }
    unsigned piv = 0;
    int zrow = 0;
    seg_solve<R, 4, double>(a, b, c, d, -epn, nr, n, s0, smem_rs, P, TI, sh.nlines, line0, li, ps, piv, zrow);
    if (D == 2) {
        // every q of the segment is loaded, and every sum formed, before
        // the first store: the loads are in flight together and the stores
        // wait for nothing
        double qv[R][4];
#pragma unroll
        for (int r = 0; r < R; r++) {
            const long g = L.off + base + (long)(min(s0 + r, n - 1) + 1) * sD;
#pragma unroll
            for (int m = 0; m < 4; m++) qv[r][m] = F.q[m][g];
        }
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int m = 0; m < 4; m++) qv[r][m] = qv[r][m] + d[r][m];
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (r < nr) {
                const long g = L.off + base + (long)(s0 + r + 1) * sD;
#pragma unroll
                for (int m = 0; m < 4; m++) F.q[m][g] = qv[r][m];
            }
        }
    } else if (D == 0 && nr == R) {
        // a whole segment of an i line: one run of consecutive nodes per
        // component
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
            for (int r = 0; r < R; r++) F.dp[m][base + s0 + r + 1] = d[r][m];
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (r < nr) {
                const long tl = base + (long)(s0 + r + 1) * sD;
#pragma unroll
                for (int m = 0; m < 4; m++) F.dp[m][tl] = d[r][m];
            }
        }
    }
    if (piv) atomicAdd(F.pivots, (unsigned long long)piv);
    if (zrow) atomicMin(F.zero_pivot, (unsigned)zrow);
}

// ---- grid ratios of the inflow faces (init_outlet_bc, init.F90:2750-2891) ----
// Face b (0..3: i = 1, i = img, j = 1, j = jmg), node t of the face plane
// (i faces: j + nj k, j faces: i + ni k): the spacing of the first node pair
// off the face over that of the second, along coordinate dir (bdir - 1).
__global__ void k_outlet_ratio(Level L, Fields F, int b, int dir) {
    const int ni = L.ni, nj = L.nj, nk = L.nk;
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long np = b < 2 ? (long)nj * nk : (long)ni * nk;
    if (t >= np) return;
    const long sJ = ni, sK = (long)ni * nj;
    long l0, st;
    if (b < 2) {
        const long base = sJ * (t % nj) + sK * (t / nj);
        l0 = b == 0 ? base : base + ni - 1;
        st = b == 0 ? 1 : -1;
    } else {
        const long base = (t % ni) + sK * (t / ni);
        l0 = b == 2 ? base : base + sJ * (nj - 1);
        st = b == 2 ? sJ : -sJ;
    }
    const double* c = F.x[dir] + L.off;
    const double c0 = c[l0], c1 = c[l0 + st], c2 = c[l0 + 2 * st];
    F.rat[b][t] = (b % 2 == 0) ? (c1 - c0) / (c2 - c1) : (c0 - c1) / (c1 - c2);
}

// ---- bcond_fm faces ----
// The reference sets the i faces, then the j faces, then the k faces, each
// over boundary nodes too, so an edge node reads face nodes of the direction
// before.  One launch does all three: the value a node has after direction E
// is formed from the values its one or two source nodes have after direction
// E - 1, down to nodes that no face writes (bc_value), and a node is stored by
// the thread of its last direction alone.  A node that another thread's chain
// reads from memory is stored by no thread (a node inside the block), or its
// own chain is the identity in every component that the reader uses: faces of
// types 0 and 5, type 8 but on the high i face, i faces of type 6, the source
// plane of a two-sided copy, the velocities of an inflow face.  Its owner
// stores such a component with the bits it read, so the reader gets the same
// from before and after that store; a rule that would change one needs a
// launch of its own.  (Three launches in sequence: 15 us on a level
// of 33^3 nodes, where each is little more than its launch; 8.4 us in one.)
// Exception: a plane copy (btype 6) on one face of a direction only reads the
// opposite plane that its own rule overwrites; then every direction has its
// own launch (E0 = E1), whose threads hold both faces of a line.
// Inflow (btype 4) on a k face uses ratio 0: the reference fills its table
// only where btype == 4 .and. btype == 5 (init.F90:2855, :2874), i.e. never,
// and the table is zero as allocated.
// (The rule of a face is first reduced to at most three source positions, so
// that one level of the recursion has three call sites and not one per rule.)
template <int E0, int E>
struct BcValue {
    // q(1:4) after directions E0 .. E at node p
    static __device__ __forceinline__ void get(const Level& L, const Fields& F, const Consts& C, const int (&p)[3],
                                               double (&v)[4]) {
        const int nd = E == 0 ? L.ni : E == 1 ? L.nj : L.nk;
        // the rule at p: a copy of s0, or a combination of s1 and s2 (all of q,
        // or the pressure alone with the rest as in a copy)
        bool high = p[E] == nd - 1;
        const bool face = p[E] == 0 || high;
        int bt = face ? (high ? C.btype[2 * E + 1] : C.btype[2 * E]) : 0;
        if (E > 0 && high && bt == 6) {  // the low plane as it is by now
            high = false;
            bt = C.btype[2 * E];
        }
        int s0 = face ? (high ? nd - 1 : 0) : p[E];
        if (bt == 6 && E > 0) s0 = nd - 1;  // plane copy from the opposite boundary plane (not done for i)
        if (bt == 7) s0 = high ? 1 : nd - 2;  // periodic wrap: the image of the opposite interior plane
        if (bt == 8 && E == 0 && high) s0 = nd - 2;
        const bool lin = bt >= 1 && bt <= 3, inflow = bt == 4;
        int s[3] = {p[0], p[1], p[2]};
        double a[4] = {}, c[4] = {};
        if (!lin) {
            s[E] = s0;
            BcValue<E0, E - 1>::get(L, F, C, s, v);
        }
        if (lin || inflow) {
            s[E] = high ? nd - 2 : 1;
            BcValue<E0, E - 1>::get(L, F, C, s, a);
            s[E] = high ? nd - 3 : 2;
            BcValue<E0, E - 1>::get(L, F, C, s, c);
        }
        if (lin) {
#pragma unroll
            for (int m = 0; m < 4; m++) {
                const double sa = high ? C.sa[2 * E + 1][m] : C.sa[2 * E][m];
                const double sb = high ? C.sb[2 * E + 1][m] : C.sb[2 * E][m];
                v[m] = fma(sa, a[m], sb * c[m]);
            }
        }
        if (inflow) {  // pressure extrapolated on the grid ratio (bcond_fm.F90:95-102)
            double r = 0.0;
            if (E < 2) {
                const double* rat = high ? F.rat[E < 2 ? 2 * E + 1 : 0] : F.rat[E < 2 ? 2 * E : 0];
                r = E == 0 ? rat[p[1] + (long)L.nj * p[2]] : rat[p[0] + (long)L.ni * p[2]];
            }
            v[0] = fma(1.0 + r, a[0], -(r * c[0]));
        }
    }
};
// before the first direction: memory
template <int E0>
struct BcBase {
    static __device__ __forceinline__ void get(const Level& L, const Fields& F, const Consts&, const int (&p)[3],
                                               double (&v)[4]) {
        const long g = L.off + lidx(L, p[0], p[1], p[2]);
#pragma unroll
        for (int m = 0; m < 4; m++) v[m] = F.q[m][g];
    }
};
template <>
struct BcValue<0, -1> : BcBase<0> {};
template <>
struct BcValue<1, 0> : BcBase<1> {};
template <>
struct BcValue<2, 1> : BcBase<2> {};

// workgroups of the faces of directions E0 .. E1 (a workgroup has one
// direction); in one launch each side its own, then one for the pinned node
__host__ __device__ inline unsigned face_blocks(const Level& L, int E) {
    const long n = E == 0 ? (long)L.nj * L.nk : E == 1 ? (long)L.ni * L.nk : (long)L.ni * L.nj;
    return (unsigned)((n + 255) / 256);
}
__host__ __device__ inline unsigned face_blocks(const Level& L, int E0, int E1) {
    unsigned n = 0;
    for (int e = E0; e <= E1; e++) n += face_blocks(L, e);
    return E0 == E1 ? n : 2 * n + 1;
}
// line t of direction e: position of its low node; false past the last line
__device__ __forceinline__ bool face_line(const Level& L, int e, long t, int (&p)[3]) {
    const int n0 = e == 0 ? L.nj : L.ni, n1 = e == 2 ? L.nj : L.nk;
    if (t >= (long)n0 * n1) return false;
    const int a = (int)(t % n0), b = (int)(t / n0);
    p[0] = e == 0 ? 0 : a;
    p[1] = e == 0 ? a : e == 1 ? 0 : b;
    p[2] = e == 2 ? 0 : b;
    return true;
}

// side: 0 low face, 1 high face (one launch for all directions: adjacent
// workgroups, so that an edge node's chain of reads is that of one side), 2
// both
template <int E0, int E, int E1>
__device__ __forceinline__ void bc_store(const Level& L, const Fields& F, const Consts& C, int (&p)[3], int side,
                                         long nfix) {
    const int nd[3] = {L.ni, L.nj, L.nk};
    // nodes on a later direction's face belong to its threads
    for (int e = E + 1; e <= E1; e++)
        if (p[e] == 0 || p[e] == nd[e] - 1) return;
    double a[4];
    if (side != 2) {
        if (side) p[E] = nd[E] - 1;
        BcValue<E0, E>::get(L, F, C, p, a);
        const long g = L.off + lidx(L, p[0], p[1], p[2]);
#pragma unroll
        for (int m = 0; m < 4; m++) F.q[m][g] = a[m];
        return;
    }
    double b[4];
    BcValue<E0, E>::get(L, F, C, p, a);
    const long lo = L.off + lidx(L, p[0], p[1], p[2]);
    p[E] = nd[E] - 1;
    BcValue<E0, E>::get(L, F, C, p, b);
    const long hi = L.off + lidx(L, p[0], p[1], p[2]);
    // one launch per direction: the pinned node's pressure comes from the
    // thread of its k line, since a one-sided plane copy to it reads the plane
    // that this line's other end overwrites
    if (E == 2 && lo - L.off == nfix % ((long)L.ni * L.nj)) {
        const long g = L.off + nfix;
        *F.pfix = g == lo ? a[0] : g == hi ? b[0] : F.q[0][g];
    }
#pragma unroll
    for (int m = 0; m < 4; m++) {
        F.q[m][lo] = a[m];
        F.q[m][hi] = b[m];
    }
}

// faces of directions E0 .. E1; with the last direction also the pressure of
// the pinned node after it (bcond_fm.F90:310-322) into F.pfix
template <int E0, int E1>
__device__ __forceinline__ void bc_fm_body(const Level& L, const Fields& F, const Consts& C, long nfix, unsigned bid,
                                           unsigned nblk) {
    if (E0 != E1 && bid == nblk - 1) {
        if (threadIdx.x != 0) return;
        const int p[3] = {(int)(nfix % L.ni), (int)((nfix / L.ni) % L.nj), (int)(nfix / ((long)L.ni * L.nj))};
        double v[4];
        BcValue<E0, E1>::get(L, F, C, p, v);
        *F.pfix = v[0];
        return;
    }
    int p[3];
    const int side = E0 == E1 ? 2 : (int)(bid & 1u);
    unsigned b = E0 == E1 ? bid : bid >> 1;
    if constexpr (E0 == 0) {
        const unsigned n = face_blocks(L, 0);
        if (b < n) {
            if (face_line(L, 0, (long)b * 256 + threadIdx.x, p)) bc_store<E0, 0, E1>(L, F, C, p, side, nfix);
            return;
        }
        b -= n;
    }
    if constexpr (E0 <= 1 && E1 >= 1) {
        const unsigned n = face_blocks(L, 1);
        if (b < n) {
            if (face_line(L, 1, (long)b * 256 + threadIdx.x, p)) bc_store<E0, 1, E1>(L, F, C, p, side, nfix);
            return;
        }
        b -= n;
    }
    if constexpr (E1 == 2) {
        if (face_line(L, 2, (long)b * 256 + threadIdx.x, p)) bc_store<E0, 2, E1>(L, F, C, p, side, nfix);
    }
}

// whether a direction copies planes on one face only
inline bool one_sided_copy(const Consts& C) {
    for (int e = 1; e < 3; e++)
        if ((C.btype[2 * e] == 6) != (C.btype[2 * e + 1] == 6)) return true;
    return false;
}

__device__ __forceinline__ void pfix_sub_body(const Level& L, const Fields& F, unsigned bid) {
    const long t = (long)bid * blockDim.x + threadIdx.x;
    if (t >= L.n) return;
    const double pf = *F.pfix;
    F.q[0][L.off + t] = F.q[0][L.off + t] - pf;
}

// ---- mg_residual: deterministic two-stage L1 sums ----
// pfix: first subtract the pinned pressure F.pfix from p at every node (the
// last step of bcond_fm, deferred to this pass when it follows directly)
__device__ __forceinline__ void resid_part_body(const Level& L, const Fields& F, int save, int pfix, unsigned bid,
                                                unsigned nb) {
    __shared__ double sh[5][256];
    double acc[5] = {0, 0, 0, 0, 0};
    const int ni = L.ni, nj = L.nj, nk = L.nk;
    const double pf = pfix ? *F.pfix : 0.0;
    for (long t = (long)bid * blockDim.x + threadIdx.x; t < L.n; t += (long)nb * blockDim.x) {
        const int i = (int)(t % ni), j = (int)((t / ni) % nj), k = (int)(t / ((long)ni * nj));
        const long g = L.off + t;
        const bool in = !(i == 0 || i == ni - 1 || j == 0 || j == nj - 1 || k == 0 || k == nk - 1);
        // all ten loads before the first store
        double qv[5], qo[5];
#pragma unroll
        for (int m = 0; m < 5; m++) {
            qv[m] = F.q[m][g];
            qo[m] = F.qold[m][g];
        }
        if (pfix) {
            qv[0] = qv[0] - pf;
            F.q[0][g] = qv[0];
        }
#pragma unroll
        for (int m = 0; m < 5; m++) {
            if (in) acc[m] += fabs(qv[m] - qo[m]);
            if (save) F.qold[m][g] = qv[m];
        }
    }
#pragma unroll
    for (int m = 0; m < 5; m++) sh[m][threadIdx.x] = acc[m];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int m = 0; m < 5; m++) sh[m][threadIdx.x] += sh[m][threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
#pragma unroll
        for (int m = 0; m < 5; m++) F.resid_part[bid * 5 + m] = sh[m][0];
    }
}

__device__ __forceinline__ void resid_final_body(const Fields& F, int nblocks) {
    __shared__ double sh[5][256];
    double acc[5] = {0, 0, 0, 0, 0};
    for (int b = threadIdx.x; b < nblocks; b += blockDim.x)
#pragma unroll
        for (int m = 0; m < 5; m++) acc[m] += F.resid_part[b * 5 + m];
#pragma unroll
    for (int m = 0; m < 5; m++) sh[m][threadIdx.x] = acc[m];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int m = 0; m < 5; m++) sh[m][threadIdx.x] += sh[m][threadIdx.x + w];
        }
        __syncthreads();
    }
    // the sums stay on the device and go, with the zero-pivot word, straight
    // to the host memory that the driver reads after the pseudo-iteration (a
    // copy command of its own cost 4 us on the stream)
    if (threadIdx.x == 0) {
#pragma unroll
        for (int m = 0; m < 5; m++) {
            F.resid[m] = sh[m][0];
            F.host_sums[m] = sh[m][0];
        }
        *reinterpret_cast<unsigned*>(F.host_sums + 5) = *F.zero_pivot;
    }
}

__global__ void __launch_bounds__(256) k_resid_final(Fields F, int nblocks) { resid_final_body(F, nblocks); }

__global__ void k_copy_qold(Level L, Fields F) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= L.n) return;
#pragma unroll
    for (int m = 0; m < 5; m++) F.qold[m][L.off + t] = F.q[m][L.off + t];
}

__global__ void k_aos_to_soa(const double* aos, int ncomp, long n, Ptrs P) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    for (int m = 0; m < ncomp; m++) P.p[m][t] = aos[t * ncomp + m];
}

__global__ void k_soa_to_aos(Ptrs P, int ncomp, long n, double* aos) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    for (int m = 0; m < ncomp; m++) aos[t * ncomp + m] = P.p[m][t];
}

__global__ void __launch_bounds__(256) k_nlevel(Level Lc, Level Lf, Fields F, int icrs, int jcrs, int kcrs) {
    nlevel_body(Lc, Lf, F, icrs, jcrs, kcrs, blockIdx.x, gridDim.x);
}
__global__ void __launch_bounds__(256) k_nlevel_z(ZoneGrid G, int n) {
    const ZoneBlock b = zone_block(G);
    const ZoneDesc& Z = G.z[b.z];
    const Level Lc = Z.lv[n], Lf = Z.lv[n - 1];
    const Fields F = Z.F;
    const int ic = Z.icrs, jc = Z.jcrs, kc = Z.kcrs;
    nlevel_body(Lc, Lf, F, ic, jc, kc, b.bid, b.nblk);
}
template <int D, int R>
__global__ void __launch_bounds__(512) k_rs_sweep(ProlongCtx P, Fields F, SegShape sh, double epn) {
    rs_sweep_body<D, R>(P, F, sh, epn, xcd_block(blockIdx.x, gridDim.x));
}
template <int D, int R>
__global__ void __launch_bounds__(512) k_rs_sweep_z(ZoneGrid G, int n, int P, int TI) {
    const ZoneBlock b = zone_block(G);
    const ZoneDesc& Z = G.z[b.z];
    const ProlongCtx PC{Z.lv[n], Z.lv[n + 1], Z.icrs, Z.jcrs, Z.kcrs};
    const Fields F = Z.F;
    rs_sweep_body<D, R>(PC, F, seg_lines(PC.Lf, D, P, TI), Z.C.ep[1][D], xcd_block(b.bid, b.nblk));
}
template <int E0, int E1>
__global__ void __launch_bounds__(256) k_bc_fm(Level L, Fields F, Consts C, long nfix) {
    bc_fm_body<E0, E1>(L, F, C, nfix, blockIdx.x, gridDim.x);
}
template <int E0, int E1>
__global__ void __launch_bounds__(256) k_bc_fm_z(ZoneGrid G) {
    const ZoneBlock b = zone_block(G);
    const ZoneDesc& Z = G.z[b.z];
    const Level L = Z.lv[1];
    const Fields F = Z.F;
    const Consts C = Z.C;
    bc_fm_body<E0, E1>(L, F, C, Z.pfix - L.off, b.bid, b.nblk);
}
__global__ void __launch_bounds__(256) k_pfix_sub(Level L, Fields F) { pfix_sub_body(L, F, blockIdx.x); }
__global__ void __launch_bounds__(256) k_pfix_sub_z(ZoneGrid G) {
    const ZoneBlock b = zone_block(G);
    const Level L = G.z[b.z].lv[1];
    const Fields F = G.z[b.z].F;
    pfix_sub_body(L, F, b.bid);
}
__global__ void __launch_bounds__(256) k_resid_part(Level L, Fields F, int save, int pfix) {
    resid_part_body(L, F, save, pfix, blockIdx.x, gridDim.x);
}
__global__ void __launch_bounds__(256) k_resid_part_z(ZoneGrid G, int save) {
    const ZoneBlock b = zone_block(G);
    const Level L = G.z[b.z].lv[1];
    const Fields F = G.z[b.z].F;
    resid_part_body(L, F, save, 0, b.bid, b.nblk);
}
// one workgroup per zone
__global__ void __launch_bounds__(256) k_resid_final_z(const ZoneDesc* __restrict__ z) {
    resid_final_body(z[blockIdx.x].F, resid_blocks(z[blockIdx.x].lv[1].n));
}

inline unsigned nblk(long n, int b) { return (unsigned)((n + b - 1) / b); }

}  // namespace

void launch_inject(hipStream_t s, const Level* lv, int ng, int icrs, int jcrs, int kcrs, double* const* comps,
                   int ncomp) {
    Ptrs P{};
    for (int m = 0; m < ncomp && m < 16; m++) P.p[m] = comps[m];
    for (int n = 2; n <= ng; n++) {
        const Level& Lc = lv[n];
        const Level& Lf = lv[n - 1];
        hipLaunchKernelGGL(k_inject_p, dim3(nblk(Lc.n, 256)), dim3(256), 0, s, Lc, Lf, P, ncomp, icrs, jcrs, kcrs);
    }
}

void launch_nlevel(hipStream_t s, const Level& Lc, const Level& Lf, const Fields& F, int icrs, int jcrs, int kcrs) {
    hipLaunchKernelGGL(k_nlevel, dim3(nblk(Lc.n, 256)), dim3(256), 0, s, Lc, Lf, F, icrs, jcrs, kcrs);
}

void launch_zero_pk_boundary(hipStream_t s, const Level& L, const Fields& F) {
    hipLaunchKernelGGL(k_zero_pk_boundary, dim3(nblk(L.n, 256)), dim3(256), 0, s, L, F);
}

// the smoothing sweep of direction D over the interior lines of level L
template <int D>
static void rs_sweep(hipStream_t s, const ProlongCtx& P, const Fields& F, double ep) {
    const Level& L = P.Lf;
    const int n = D == 0 ? L.ni - 2 : D == 1 ? L.nj - 2 : L.nk - 2;
    const long nl = D == 0 ? (long)(L.nj - 2) * (L.nk - 2) : D == 1 ? (long)(L.ni - 2) * (L.nk - 2)
                                                                    : (long)(L.ni - 2) * (L.nj - 2);
    // i lines: short segments (their rows are adjacent in memory, so lanes
    // reading row r of adjacent segments are R rows apart)
    const int R = (D == 0 || n <= 64) ? 4 : 8;
    const SegShape sh = seg_shape(n, nl, R, D == 0);
    const unsigned nb = (unsigned)((sh.nlines + sh.TI - 1) / sh.TI);
    const size_t lds = seg_lds_bytes(sh, 4);
    if (R == 4)
        hipLaunchKernelGGL((k_rs_sweep<D, 4>), dim3(nb), dim3(sh.TI * sh.P), lds, s, P, F, sh, ep);
    else
        hipLaunchKernelGGL((k_rs_sweep<D, 8>), dim3(nb), dim3(sh.TI * sh.P), lds, s, P, F, sh, ep);
}

void launch_prolong(hipStream_t s, const Level& Lf, const Level& Lc, const Fields& F, const Consts& C, int icrs,
                    int jcrs, int kcrs) {
    ProlongCtx P{Lf, Lc, icrs, jcrs, kcrs};
    rs_sweep<0>(s, P, F, C.ep[1][0]);
    rs_sweep<1>(s, P, F, C.ep[1][1]);
    rs_sweep<2>(s, P, F, C.ep[1][2]);
}

void launch_outlet_ratios(hipStream_t s, const Level& L, const Fields& F, const int* btype, const int* bdir) {
    for (int b = 0; b < 4; b++) {
        if (btype[b] != DESALM_BC_INFLOW && btype[b] != DESALM_BC_OUTLET_MOC) continue;
        const long np = b < 2 ? (long)L.nj * L.nk : (long)L.ni * L.nk;
        hipLaunchKernelGGL(k_outlet_ratio, dim3(nblk(np, 256)), dim3(256), 0, s, L, F, b, bdir[b] - 1);
    }
}

void launch_bcond_fm(hipStream_t s, const Level& L, const Fields& F, const Consts& C, int ifix, int jfix, int kfix,
                     bool pfix_deferred) {
    const long nfix = lidx_h(L, ifix - 1, jfix - 1, kfix - 1);
    if (one_sided_copy(C)) {
        hipLaunchKernelGGL((k_bc_fm<0, 0>), dim3(face_blocks(L, 0, 0)), dim3(256), 0, s, L, F, C, nfix);
        hipLaunchKernelGGL((k_bc_fm<1, 1>), dim3(face_blocks(L, 1, 1)), dim3(256), 0, s, L, F, C, nfix);
        hipLaunchKernelGGL((k_bc_fm<2, 2>), dim3(face_blocks(L, 2, 2)), dim3(256), 0, s, L, F, C, nfix);
    } else {
        hipLaunchKernelGGL((k_bc_fm<0, 2>), dim3(face_blocks(L, 0, 2)), dim3(256), 0, s, L, F, C, nfix);
    }
    if (!pfix_deferred) hipLaunchKernelGGL(k_pfix_sub, dim3(nblk(L.n, 256)), dim3(256), 0, s, L, F);
}

// Partial sums of (q - qn)^2 over the fine interior (real_residual,
// src/main.F90:214-300), deterministic like k_resid_part; k_resid_final adds
// the parts into F.resid
__global__ void __launch_bounds__(256) k_real_part(Level L, Fields F) {
    __shared__ double sh[5][256];
    double acc[5] = {0, 0, 0, 0, 0};
    const int ni = L.ni, nj = L.nj, nk = L.nk;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < L.n; t += (long)gridDim.x * blockDim.x) {
        const int i = (int)(t % ni), j = (int)((t / ni) % nj), k = (int)(t / ((long)ni * nj));
        if (i == 0 || i == ni - 1 || j == 0 || j == nj - 1 || k == 0 || k == nk - 1) continue;
        const long g = L.off + t;
#pragma unroll
        for (int m = 0; m < 5; m++) {
            const double d = F.q[m][g] - F.qn[m][g];
            acc[m] += d * d;
        }
    }
#pragma unroll
    for (int m = 0; m < 5; m++) sh[m][threadIdx.x] = acc[m];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int m = 0; m < 5; m++) sh[m][threadIdx.x] += sh[m][threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
#pragma unroll
        for (int m = 0; m < 5; m++) F.resid_part[blockIdx.x * 5 + m] = sh[m][0];
    }
}

// q(1:5) and xnut at n fine-level nodes (level-local index node[p]) into
// out[6 p .. 6 p + 5]
__global__ void k_probe(Fields F, int n, const long* node, double* out) {
    const int p = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (p >= n) return;
    const long g = node[p];
#pragma unroll
    for (int m = 0; m < 5; m++) out[6 * p + m] = F.q[m][g];
    out[6 * p + 5] = F.xnut[g];
}

void launch_real_residual(hipStream_t s, const Level& L, const Fields& F) {
    const int nb = resid_blocks(L.n);
    hipLaunchKernelGGL(k_real_part, dim3(nb), dim3(256), 0, s, L, F);
    hipLaunchKernelGGL(k_resid_final, dim3(1), dim3(256), 0, s, F, nb);
}

void launch_probe(hipStream_t s, const Fields& F, int n, const long* node, double* out) {
    if (n > 0) hipLaunchKernelGGL(k_probe, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, s, F, n, node, out);
}

void launch_resid_and_save(hipStream_t s, const Level& L, const Fields& F, int save, bool pfix) {
    const int nb = resid_blocks(L.n);
    hipLaunchKernelGGL(k_resid_part, dim3(nb), dim3(256), 0, s, L, F, save, pfix ? 1 : 0);
    hipLaunchKernelGGL(k_resid_final, dim3(1), dim3(256), 0, s, F, nb);
}

// ---- every zone of a group in one launch per kernel ----
void launch_nlevel_z(hipStream_t s, const ZoneList& Z, int n) {
    unsigned nb = 0;
    const ZoneGrid G = Z.grid([&](const ZoneDesc& z) { return nblk(z.lv[n].n, 256); }, nb);
    hipLaunchKernelGGL(k_nlevel_z, dim3(nb), dim3(256), 0, s, G, n);
}

template <int D>
static void rs_sweep_z(hipStream_t s, const ZoneList& Z, int n) {
    int len = 0;
    for (const ZoneDesc& z : Z.host) len = std::max(len, seg_lines(z.lv[n], D, 1, 1).n);
    const int R = (D == 0 || len <= 64) ? 4 : 8;
    const SegShape sh = seg_shape(len, 1, R, D == 0);
    unsigned nb = 0;
    const ZoneGrid G = Z.grid(
        [&](const ZoneDesc& z) { return (unsigned)((seg_lines(z.lv[n], D, sh.P, sh.TI).nlines + sh.TI - 1) / sh.TI); },
        nb);
    const size_t lds = seg_lds_bytes(sh, 4);
    if (R == 4)
        hipLaunchKernelGGL((k_rs_sweep_z<D, 4>), dim3(nb), dim3(sh.TI * sh.P), lds, s, G, n, sh.P, sh.TI);
    else
        hipLaunchKernelGGL((k_rs_sweep_z<D, 8>), dim3(nb), dim3(sh.TI * sh.P), lds, s, G, n, sh.P, sh.TI);
}

// prolongation from level n + 1 onto level n
void launch_prolong_z(hipStream_t s, const ZoneList& Z, int n) {
    rs_sweep_z<0>(s, Z, n);
    rs_sweep_z<1>(s, Z, n);
    rs_sweep_z<2>(s, Z, n);
}

// bcond_fm faces and the pinned-pressure shift of every zone's fine level
void launch_bcond_fm_z(hipStream_t s, const ZoneList& Z) {
    unsigned gn = 0;
    bool split = false;
    for (const ZoneDesc& z : Z.host) split = split || one_sided_copy(z.C);
    auto faces = [&](auto kernel, int e0, int e1) {
        unsigned nf = 0;
        const ZoneGrid G = Z.grid([&](const ZoneDesc& z) { return face_blocks(z.lv[1], e0, e1); }, nf);
        hipLaunchKernelGGL(kernel, dim3(nf), dim3(256), 0, s, G);
    };
    if (split) {
        faces(k_bc_fm_z<0, 0>, 0, 0);
        faces(k_bc_fm_z<1, 1>, 1, 1);
        faces(k_bc_fm_z<2, 2>, 2, 2);
    } else {
        faces(k_bc_fm_z<0, 2>, 0, 2);
    }
    const ZoneGrid Gn = Z.grid([&](const ZoneDesc& z) { return nblk(z.lv[1].n, 256); }, gn);
    hipLaunchKernelGGL(k_pfix_sub_z, dim3(gn), dim3(256), 0, s, Gn);
}

// update norms of every zone's fine level into its F.resid, then qold <- q
void launch_resid_and_save_z(hipStream_t s, const ZoneList& Z, int save) {
    unsigned nb = 0;
    const ZoneGrid G = Z.grid([&](const ZoneDesc& z) { return (unsigned)resid_blocks(z.lv[1].n); }, nb);
    hipLaunchKernelGGL(k_resid_part_z, dim3(nb), dim3(256), 0, s, G, save);
    hipLaunchKernelGGL(k_resid_final_z, dim3(Z.nz()), dim3(256), 0, s, (const ZoneDesc*)Z.dev);
}

void launch_copy_qold(hipStream_t s, const Level& L, const Fields& F) {
    hipLaunchKernelGGL(k_copy_qold, dim3(nblk(L.n, 256)), dim3(256), 0, s, L, F);
}

void launch_aos_to_soa(hipStream_t s, const double* aos, int ncomp, long n, double* const* soa) {
    Ptrs P{};
    for (int m = 0; m < ncomp && m < 16; m++) P.p[m] = soa[m];
    hipLaunchKernelGGL(k_aos_to_soa, dim3(nblk(n, 256)), dim3(256), 0, s, aos, ncomp, n, P);
}

void launch_soa_to_aos(hipStream_t s, double* const* soa, int ncomp, long n, double* aos) {
    Ptrs P{};
    for (int m = 0; m < ncomp && m < 16; m++) P.p[m] = soa[m];
    hipLaunchKernelGGL(k_soa_to_aos, dim3(nblk(n, 256)), dim3(256), 0, s, P, ncomp, n, aos);
}

}  // namespace desalm
