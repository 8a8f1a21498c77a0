// k_mlp.hip -- learned warm start of a physical time step.
//
// The reference starts every physical step's pseudo-iterations from the
// previous step's solution (mg_driver.F90:48-51: qn <- q, q unchanged).  The
// warm start replaces that initial guess on the fine level's interior by a
// two-step extrapolation in physical time whose coefficients are predicted
// per node and per variable,
//   q(0) = q^n + a d1 + b d2,  d1 = q^n - q^(n-1),  d2 = q^(n-1) - q^(n-2),
// with (a - 1, b) the outputs of a multilayer perceptron (zero outputs give
// linear extrapolation).  Its inputs are scale-free: for each of the five
// variables, the 18 time differences d1, d2 at the node and its eight
// neighbours (the six face neighbours and the second neighbours along i, the
// inflow direction; clamped to the block) divided by their root mean square,
// plus q^n at the node.  The
// pseudo-iterations then run to the same tolerance as from any other start,
// so the warm start only changes how many of them are needed.
//
// Everything is FP32 and written here: the feature gather, the layers on tiles
// of 64 rows that stay in LDS from the input to the output gradient, weight
// gradients as per-chunk partial products summed in a fixed order, the loss
// and Adam.
// Every layer's weights are one (K + 1) x N row-major matrix whose last row
// is the bias, and every activation matrix carries a trailing column of ones,
// so a layer is a single product.
#include "desalm_internal.h"

namespace desalm {

namespace {

constexpr int kBM = 64;     // rows (samples) per tile
constexpr int kKMax = 96;   // largest K + 1 a layer may have
constexpr int kWgRows = 512;  // rows per weight-gradient partial

// 64-bit mix of (seed, a, b) -> uniform index source (splitmix64 finaliser)
__device__ __forceinline__ unsigned long long mix3(unsigned long long s, unsigned long long a,
                                                   unsigned long long b) {
    unsigned long long z = s + 0x9E3779B97F4A7C15ull * (a + 1) + 0xBF58476D1CE4E5B9ull * (b + 1);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// interior node (level-local index) of interior ordinal r, i fastest
__device__ __forceinline__ long interior_node(const Level& L, long r) {
    const long ni = L.ni - 2, nj = L.nj - 2;
    const long i = 1 + r % ni, j = 1 + (r / ni) % nj, k = 1 + r / (ni * nj);
    return i + (long)L.ni * (j + (long)L.nj * k);
}

// Features and (optionally) training target of level-local node t.
// Feature order: for component c, for stencil point s (node, -i, +i, -j,
// +j, -k, +k, -2i, +2i; the second neighbours clamped to i = 0 and ni - 1):
// d1, d2, each divided by the root mean square of the component's 18 (0
// when they are all zero); then q^n(c) at the node.
// mu / isd standardise the features when non-null.  Target: per component
// r = q - 2 q^n + q^(n-1), then d1 and d2 at the node (raw).
__device__ void ws_row(const Level& L, const Fields& F, double* const* qnm2, long t, float* x, float* y,
                       const float* mu, const float* isd) {
    const long g = L.off + t;
    const int i = (int)(t % L.ni);
    const long st[kWsPts] = {0, -1, 1, -(long)L.ni, (long)L.ni, -(long)L.ni * L.nj, (long)L.ni * L.nj,
                             i >= 2 ? -2 : -(long)i, i + 2 <= L.ni - 1 ? 2 : (long)(L.ni - 1 - i)};
    int f = 0;
    for (int c = 0; c < kWsComp; c++) {
        const double* a = F.qn[c];
        const double* b = F.qnm1[c];
        const double* d = qnm2[c];
        double v[2 * kWsPts];
        double ss = 0.0;
#pragma unroll
        for (int s = 0; s < kWsPts; s++) {
            const long p = g + st[s];
            const double bp = b[p];
            v[2 * s] = a[p] - bp;
            v[2 * s + 1] = bp - d[p - L.off];
            ss += v[2 * s] * v[2 * s] + v[2 * s + 1] * v[2 * s + 1];
        }
        const double rms = sqrt(ss / (2 * kWsPts));
#pragma unroll
        for (int e = 0; e < 2 * kWsPts; e++) {
            float w = rms > 0.0 ? (float)(v[e] / rms) : 0.0f;
            if (mu) w = (w - mu[f]) * isd[f];
            x[f++] = w;
        }
    }
    for (int c = 0; c < kWsComp; c++) {
        float w = (float)F.qn[c][g];
        if (mu) w = (w - mu[f]) * isd[f];
        x[f++] = w;
    }
    x[f] = 1.0f;  // bias column
    if (y) {
        for (int c = 0; c < kWsComp; c++) {
            const double qn = F.qn[c][g], qm = F.qnm1[c][g];
            y[c] = (float)(F.q[c][g] - 2.0 * qn + qm);
            y[kWsComp + c] = (float)(qn - qm);
            y[2 * kWsComp + c] = (float)(qm - qnm2[c][g - L.off]);
        }
    }
}

// record: m rows sampled from the interior with replacement (seeded),
// raw features into X (ld kWsIn + 1) and targets into T (ld kWsTgt)
__global__ void k_ws_sample(Level L, Fields F, WsQ Q, float* X, float* T, long m, unsigned long long seed,
                            long step) {
    const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= m) return;
    const long nint = (long)(L.ni - 2) * (L.nj - 2) * (L.nk - 2);
    const long t = interior_node(L, (long)(mix3(seed, (unsigned long long)step, (unsigned long long)r) % nint));
    ws_row(L, F, Q.q, t, X + r * (kWsIn + 1), T + r * kWsTgt, nullptr, nullptr);
}

// inference features of interior ordinals r0 .. r0 + m - 1, standardised
// when stats is not null
__global__ void k_ws_features(Level L, Fields F, WsQ Q, float* X, long r0, long m, const float* stats) {
    const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= m) return;
    ws_row(L, F, Q.q, interior_node(L, r0 + r), X + r * (kWsIn + 1), nullptr, stats,
           stats ? stats + kWsIn : nullptr);
}

// linear extrapolation 2 q^n - q^(n-1) on the interior; nu~ keeps the floor
// of the SA update (rhs_sa_bcond.F90:283-287)
__global__ void k_ws_extrap(Level L, Fields F, long m) {
    const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= m) return;
    const long g = L.off + interior_node(L, r);
    for (int c = 0; c < kWsComp; c++) {
        double v = 2.0 * F.qn[c][g] - F.qnm1[c][g];
        if (c == 4) v = fmax(1.0e-07, v);
        F.q[c][g] = v;
    }
}

// ---- the network on tiles of 64 rows ----
// A workgroup keeps a tile's activations and the weights of all three layers
// in LDS, so a training step is three launches: k_mlp_tile (batch gather,
// forward pass, loss, data gradients), k_wgrad (weight gradients of all
// layers) and k_grad_sum (their partials summed, Adam).  As one launch per
// layer and direction (fourteen) a step of 16384 rows, 32 hidden units, took
// 400 us: 92 us for each of three weight gradients, whose 32 workgroups
// (one per 512 rows) left seven eighths of the CUs idle, and 4.5 us or more
// for each launch; in three launches it takes 51 us (29, 18 and 5), most of it
// latency: one tile per CU walks its layers in sequence.  Every sum keeps its
// order (products over k ascending; rows ascending inside a part of 512,
// parts ascending), so results are the same bits.
constexpr int kLd = kBM + 4;  // row stride of the transposed activations [k][row]: float4 reads, few bank conflicts

// floats of LDS: activations of the input and of both hidden layers, and the
// weights of the three layers with rows padded to an odd count (the backward
// pass reads them along k).  The gradients of the outputs and of the second
// hidden layer reuse the input's space.
struct MlpLds {
    int ld, w1, w2, w3, a1, a2, total;
    __host__ __device__ explicit MlpLds(int nh) {
        ld = nh | 1;
        w1 = kKMax * kLd;
        w2 = w1 + (kWsIn + 1) * ld;
        w3 = w2 + (nh + 1) * ld;
        a1 = (w3 + (nh + 1) * (kWsOut | 1) + 3) & ~3;
        a2 = a1 + (nh + 1) * kLd;
        total = a2 + (nh + 1) * kLd;
    }
};
static_assert((kWsOut + kWsMaxHidden) * kLd <= kKMax * kLd, "gradients fit the input's space");

// acc[u][v] = sum over k < K1 of A[k][4 tr + u] W[k][CT tc + v], k ascending
template <int CT>
__device__ __forceinline__ void tile_product(const float* A, int K1, const float* W, int ld, int N, int tr, int tc,
                                             float (&acc)[4][CT]) {
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
        for (int v = 0; v < CT; v++) acc[u][v] = 0.0f;
    int col[CT];
#pragma unroll
    for (int v = 0; v < CT; v++) col[v] = min(tc * CT + v, N - 1);
#pragma unroll 8
    for (int k = 0; k < K1; k++) {
        const float4 a = *reinterpret_cast<const float4*>(A + k * kLd + 4 * tr);
        float w[CT];
#pragma unroll
        for (int v = 0; v < CT; v++) w[v] = W[k * ld + col[v]];
#pragma unroll
        for (int v = 0; v < CT; v++) {
            acc[0][v] = fmaf(a.x, w[v], acc[0][v]);
            acc[1][v] = fmaf(a.y, w[v], acc[1][v]);
            acc[2][v] = fmaf(a.z, w[v], acc[2][v]);
            acc[3][v] = fmaf(a.w, w[v], acc[3][v]);
        }
    }
}

// B[n][row] = tanh(A W), n < N, and the ones column B[N]
template <int CT>
__device__ __forceinline__ void tile_layer(const float* A, int K1, const float* W, int ld, int N, float* B, int tid) {
    const int tr = tid / 16, tc = tid % 16;
    float acc[4][CT];
    tile_product<CT>(A, K1, W, ld, N, tr, tc, acc);
#pragma unroll
    for (int v = 0; v < CT; v++) {
        const int n = tc * CT + v;
        if (n < N)
            *reinterpret_cast<float4*>(B + n * kLd + 4 * tr) =
                make_float4(tanhf(acc[0][v]), tanhf(acc[1][v]), tanhf(acc[2][v]), tanhf(acc[3][v]));
    }
    if (tc == 0) *reinterpret_cast<float4*>(B + N * kLd + 4 * tr) = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
}

// G[k][row] = (sum over n of Z[n][row] W[k][n], n ascending) (1 - A[k][row]^2)
// for k < K: the gradient through a layer (without its bias row) and the tanh
// that produced A; also stored row-major in Gg (ld K).  G null: Gg only.
template <int CT>
__device__ __forceinline__ void tile_back(const float* Z, int N, const float* W, int ld, int K, const float* A,
                                          float* G, float* Gg, int r0, int M, int tid) {
    const int tr = tid / 16, tc = tid % 16;
    int row[CT];
#pragma unroll
    for (int v = 0; v < CT; v++) row[v] = min(tc * CT + v, K - 1) * ld;
    float acc[4][CT] = {};
#pragma unroll 8
    for (int n = 0; n < N; n++) {
        const float4 z = *reinterpret_cast<const float4*>(Z + n * kLd + 4 * tr);
#pragma unroll
        for (int v = 0; v < CT; v++) {
            const float w = W[row[v] + n];
            acc[0][v] = fmaf(z.x, w, acc[0][v]);
            acc[1][v] = fmaf(z.y, w, acc[1][v]);
            acc[2][v] = fmaf(z.z, w, acc[2][v]);
            acc[3][v] = fmaf(z.w, w, acc[3][v]);
        }
    }
#pragma unroll
    for (int v = 0; v < CT; v++) {
        const int k = tc * CT + v;
        if (k >= K) continue;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const float ap = A[k * kLd + 4 * tr + u];
            const float g = acc[u][v] * (1.0f - ap * ap);
            if (G) G[k * kLd + 4 * tr + u] = g;
            if (r0 + 4 * tr + u < M) Gg[(long)(r0 + 4 * tr + u) * K + k] = g;
        }
    }
}

// 64 rows [64 blockIdx, ...) of M through the network.
//   kTileForward: rows A.A0 -> outputs A.Y
//   kTileLoss:    rows A.A0, scaled targets A.Tb -> activations and gradients of every layer (for k_wgrad),
//                 loss partial of the tile
//   kTileTrain:   the same on rows drawn from the first nsrc rows of the sample buffer (X, T; standardised
//                 here, the drawn rows stored in A.A0)
// Loss: e_c = y_a,c d1_c + y_b,c d2_c - r_c in units of the per-component
// scale, mean over rows and components of e^2; dZ3 = d loss / d y.
enum { kTileForward, kTileLoss, kTileTrain };
template <int MODE, int CT>
__global__ void __launch_bounds__(256) k_mlp_tile(MlpBuf A, const float* w, int nh, int M, const float* X,
                                                  const float* T, long nsrc, unsigned long long seed, long it,
                                                  const float* stats) {
    extern __shared__ __align__(16) float smem_mlp[];
    __shared__ long s_src[kBM];
    __shared__ double s_red[256];
    const MlpLds O(nh);
    float* s0 = smem_mlp;
    const int tid = (int)threadIdx.x;
    const int r0 = (int)blockIdx.x * kBM;
    constexpr int K1 = kWsIn + 1;
    if (MODE == kTileTrain) {
        if (tid < kBM)
            s_src[tid] = (long)(mix3(seed ^ 0x5851F42D4C957F2Dull, (unsigned long long)it,
                                     (unsigned long long)(r0 + tid)) % (unsigned long long)nsrc);
        __syncthreads();
    }
    constexpr int kLossPer = (kBM * kWsComp + 255) / 256;
    float tgt[kLossPer][3], tsc[kLossPer];
    // the rows: 32 threads along a row, 8 rows at a time, every load issued
    // before the first use
    {
        constexpr int NC = K1 / 32, NR = kBM / 8;
        static_assert(K1 % 32 == 0, "whole groups of 32 columns");
        const int cx = tid % 32, rx = tid / 32;
        float v[NR][NC];
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int row = rx + 8 * r;
            const bool in = r0 + row < M;
            const float* src = MODE == kTileTrain ? X + s_src[row] * K1 : A.A0 + (long)(in ? r0 + row : 0) * K1;
#pragma unroll
            for (int c = 0; c < NC; c++) v[r][c] = src[cx + 32 * c];
        }
        // the targets of this thread's (row, component) pairs as well
        if (MODE != kTileForward) {
#pragma unroll
            for (int q = 0; q < kLossPer; q++) {
                const int e = tid + 256 * q, row = e % kBM, c = min(e / kBM, kWsComp - 1);
                const float* t = MODE == kTileTrain ? T + s_src[row] * kWsTgt
                                                    : A.Tb + (long)min(r0 + row, M - 1) * kWsTgt;
#pragma unroll
                for (int u = 0; u < 3; u++) tgt[q][u] = t[u * kWsComp + c];
                if (MODE == kTileTrain) tsc[q] = stats[2 * kWsIn + c];
            }
        }
        float mu[NC], isd[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int col = min(cx + 32 * c, kWsIn - 1);
            mu[c] = MODE == kTileTrain ? stats[col] : 0.0f;
            isd[c] = MODE == kTileTrain ? stats[kWsIn + col] : 0.0f;
        }
        for (int k = rx; k < K1; k += 8)
            for (int n = cx; n < nh; n += 32) smem_mlp[O.w1 + k * O.ld + n] = w[k * nh + n];
        const float* w2 = w + K1 * nh;
        const float* w3 = w2 + (nh + 1) * nh;
        for (int k = rx; k <= nh; k += 8) {
            for (int n = cx; n < nh; n += 32) smem_mlp[O.w2 + k * O.ld + n] = w2[k * nh + n];
            if (cx < kWsOut) smem_mlp[O.w3 + k * (kWsOut | 1) + cx] = w3[k * kWsOut + cx];
        }
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const int row = rx + 8 * r;
            const bool in = r0 + row < M;
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const int col = cx + 32 * c;
                float x = v[r][c];
                if (MODE == kTileTrain) {
                    x = col < kWsIn ? (x - mu[c]) * isd[c] : 1.0f;
                    if (in) A.A0[(long)(r0 + row) * K1 + col] = x;
                }
                s0[col * kLd + row] = in ? x : 0.0f;
            }
        }
    }
    __syncthreads();
    tile_layer<CT>(s0, K1, smem_mlp + O.w1, O.ld, nh, smem_mlp + O.a1, tid);
    __syncthreads();
    tile_layer<CT>(smem_mlp + O.a1, nh + 1, smem_mlp + O.w2, O.ld, nh, smem_mlp + O.a2, tid);
    __syncthreads();
    // the output layer: y into the input's space (dead by now), [c][row]
    {
        const int tr = tid / 16, tc = tid % 16;
        float acc[4][1];
        tile_product<1>(smem_mlp + O.a2, nh + 1, smem_mlp + O.w3, kWsOut | 1, kWsOut, tr, tc, acc);
        if (tc < kWsOut) {
#pragma unroll
            for (int u = 0; u < 4; u++) {
                if (MODE == kTileForward) {
                    if (r0 + 4 * tr + u < M) A.Y[(long)(r0 + 4 * tr + u) * kWsOut + tc] = acc[u][0];
                } else {
                    s0[tc * kLd + 4 * tr + u] = acc[u][0];
                }
            }
        }
    }
    if (MODE == kTileForward) return;
    // activations of the hidden layers for k_wgrad
    for (int row = tid / 32; row < kBM && r0 + row < M; row += 8)
        for (int col = tid % 32; col <= nh; col += 32) {
            A.A1[(long)(r0 + row) * (nh + 1) + col] = smem_mlp[O.a1 + col * kLd + row];
            A.A2[(long)(r0 + row) * (nh + 1) + col] = smem_mlp[O.a2 + col * kLd + row];
        }
    __syncthreads();
    double s = 0.0;
    const float scale = 2.0f / (float)((long)M * kWsComp);
#pragma unroll
    for (int q = 0; q < kLossPer; q++) {
        const int e = tid + 256 * q, row = e % kBM, c = e / kBM;
        if (c >= kWsComp) continue;
        float za = 0.0f, zb = 0.0f;
        if (r0 + row < M) {
            const float r = MODE == kTileTrain ? tgt[q][0] / tsc[q] : tgt[q][0];
            const float d1 = MODE == kTileTrain ? tgt[q][1] / tsc[q] : tgt[q][1];
            const float d2 = MODE == kTileTrain ? tgt[q][2] / tsc[q] : tgt[q][2];
            const float err = fmaf(s0[c * kLd + row], d1, s0[(kWsComp + c) * kLd + row] * d2) - r;
            za = scale * err * d1;
            zb = scale * err * d2;
            s += (double)err * (double)err;
            A.dZ3[(long)(r0 + row) * kWsOut + c] = za;
            A.dZ3[(long)(r0 + row) * kWsOut + kWsComp + c] = zb;
        }
        // only this thread reads or writes these two entries before the barrier
        s0[c * kLd + row] = za;
        s0[(kWsComp + c) * kLd + row] = zb;
    }
    s_red[tid] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (tid < h) s_red[tid] += s_red[tid + h];
        __syncthreads();
    }
    if (tid == 0) A.lpart[blockIdx.x] = s_red[0];
    tile_back<CT>(s0, kWsOut, smem_mlp + O.w3, kWsOut | 1, nh, smem_mlp + O.a2, s0 + kWsOut * kLd, A.dZ2, r0, M, tid);
    __syncthreads();
    tile_back<CT>(s0 + kWsOut * kLd, nh, smem_mlp + O.w2, O.ld, nh, smem_mlp + O.a1, nullptr, A.dZ1, r0, M, tid);
}

// Partial weight gradients of rows [kWgRows blockIdx.x, ...) of all three
// layers: P[part][offset of the layer + k N + n] = sum_r act[r][k] dZ[r][n]
// (the ones column gives the bias row).  blockIdx.y walks the layers' tiles of
// kWgK x kWgN outputs, so a batch of 16384 rows is 384 workgroups.
constexpr int kWgK = 16, kWgN = 32, kWgTile = 128;
__host__ __device__ inline int wg_tiles(int K1, int N) { return ((K1 + kWgK - 1) / kWgK) * ((N + kWgN - 1) / kWgN); }
__global__ void __launch_bounds__(128) k_wgrad(MlpBuf A, int nh, int M, int np) {
    __shared__ float As[kWgTile][kWgK];
    __shared__ float Zs[kWgTile][kWgN];
    int tile = (int)blockIdx.y;
    const int n1 = wg_tiles(kWsIn + 1, nh), n2 = wg_tiles(nh + 1, nh);
    const float *act, *dz;
    int K1, N, base;
    if (tile < n1) {
        act = A.A0; dz = A.dZ1; K1 = kWsIn + 1; N = nh; base = 0;
    } else if (tile < n1 + n2) {
        tile -= n1;
        act = A.A1; dz = A.dZ2; K1 = nh + 1; N = nh; base = (kWsIn + 1) * nh;
    } else {
        tile -= n1 + n2;
        act = A.A2; dz = A.dZ3; K1 = nh + 1; N = kWsOut; base = (kWsIn + 1 + nh + 1) * nh;
    }
    const int tk = (K1 + kWgK - 1) / kWgK;
    const int k0 = (tile % tk) * kWgK, n0 = (tile / tk) * kWgN;
    const int tid = (int)threadIdx.x;
    const int kx = 2 * (tid / 16), nx = 2 * (tid % 16);
    const int rbeg = (int)blockIdx.x * kWgRows, rend = min(M, rbeg + kWgRows);
    // the next tile's rows are loaded while the current one is summed, at
    // clamped addresses (no branch around a load)
    constexpr int QA = kWgTile * kWgK / 128, QZ = kWgTile * kWgN / 128;
    float av[QA], zv[QZ];
    const int ka = k0 + tid % kWgK, nz = n0 + tid % kWgN;  // columns of this thread's loads
    const float* ap = act + min(ka, K1 - 1);
    const float* zp = dz + min(nz, N - 1);
    const int ra = tid / kWgK, rz = tid / kWgN;
    auto load = [&](int rt) {
#pragma unroll
        for (int q = 0; q < QA; q++) av[q] = ap[(long)min(rt + ra + 128 / kWgK * q, rend - 1) * K1];
#pragma unroll
        for (int q = 0; q < QZ; q++) zv[q] = zp[(long)min(rt + rz + 128 / kWgN * q, rend - 1) * N];
    };
    float acc[2][2] = {};
    load(rbeg);
    for (int rt = rbeg; rt < rend; rt += kWgTile) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < QA; q++) (&As[0][0])[tid + 128 * q] = rt + ra + 128 / kWgK * q < rend ? av[q] : 0.0f;
#pragma unroll
        for (int q = 0; q < QZ; q++) (&Zs[0][0])[tid + 128 * q] = rt + rz + 128 / kWgN * q < rend ? zv[q] : 0.0f;
        load(rt + kWgTile);
        __syncthreads();
        // rows past the part's end are zero on both sides
#pragma unroll 16
        for (int r = 0; r < kWgTile; r++) {
            const float2 a = *reinterpret_cast<const float2*>(&As[r][kx]);
            const float2 z = *reinterpret_cast<const float2*>(&Zs[r][nx]);
            acc[0][0] = fmaf(a.x, z.x, acc[0][0]);
            acc[0][1] = fmaf(a.x, z.y, acc[0][1]);
            acc[1][0] = fmaf(a.y, z.x, acc[1][0]);
            acc[1][1] = fmaf(a.y, z.y, acc[1][1]);
        }
    }
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int v = 0; v < 2; v++)
            if (k0 + kx + u < K1 && n0 + nx + v < N)
                A.P[(long)blockIdx.x * np + base + (k0 + kx + u) * N + n0 + nx + v] = acc[u][v];
}

struct AdamArgs {
    float *w, *m, *v;  // null w: no update
    float lr, b1, b2, eps, c1, c2;
};

// g[o] = sum over the parts, ascending, then the Adam update of parameter o;
// the last workgroup sums the loss partials of the row tiles into loss
__global__ void __launch_bounds__(256) k_grad_sum(const float* P, int nparts, int np, float* g, AdamArgs a,
                                                  const double* lpart, int ntiles, double* loss) {
    if (blockIdx.x == gridDim.x - 1) {
        __shared__ double s_red[256];
        double s = 0.0;
        for (int b = (int)threadIdx.x; b < ntiles; b += 256) s += lpart[b];
        s_red[threadIdx.x] = s;
        __syncthreads();
        for (int h = 128; h > 0; h >>= 1) {
            if ((int)threadIdx.x < h) s_red[threadIdx.x] += s_red[threadIdx.x + h];
            __syncthreads();
        }
        if (threadIdx.x == 0) *loss = s_red[0];
        return;
    }
    const int o = (int)(blockIdx.x * 256 + threadIdx.x);
    if (o >= np) return;
    float s = 0.0f;
    int p = 0;
    for (; p + 8 <= nparts; p += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = P[(long)(p + u) * np + o];
#pragma unroll
        for (int u = 0; u < 8; u++) s += v[u];
    }
    for (; p < nparts; p++) s += P[(long)p * np + o];
    g[o] = s;
    if (!a.w) return;
    const float mi = a.b1 * a.m[o] + (1.0f - a.b1) * s;
    const float vi = a.b2 * a.v[o] + (1.0f - a.b2) * s * s;
    a.m[o] = mi;
    a.v[o] = vi;
    a.w[o] -= a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
}

// The learned start of the whole interior in one launch: features of a tile
// of TM nodes into LDS, the three layers on the tile (4 x 4 outputs per
// thread, weights resident in LDS), and
//   q(0) = q^n + (1 + y_a) d1 + y_b d2,  nu~ >= 1e-7,
// written from there.  A workgroup walks a contiguous run of tiles, so the
// weights are staged once and the j neighbours of a tile come from its L2.
// Bound by FP32 and FP64 arithmetic (4458 multiply-adds, 64 tanh and 90 FP64
// divisions per node with 32 hidden units).  As a feature pass, three layer
// passes and an apply pass over chunks of 131072 nodes the rows crossed HBM
// five times and the feature rows were written 96 words apart by adjacent
// threads: 17 ms for the 9.3 M interior nodes of a 257x193x193 block, 4.1 ms
// here.  TM = 128 for up to 32 hidden units (8 column groups of 4), 64 above (16): the
// tile's rows times its column groups fill 256 threads either way.
// Products run over k ascending and features are rounded as in ws_row.
template <int TM>
__device__ __forceinline__ void infer_product(const float* A, int K1, const float* W, int ld, int tr, int tc,
                                              float (&acc)[4][4]) {
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) acc[u][v] = 0.0f;
#pragma unroll 4
    for (int k = 0; k < K1; k++) {
        const float4 a = *reinterpret_cast<const float4*>(A + k * (TM + 4) + 4 * tr);
        const float4 w = *reinterpret_cast<const float4*>(W + k * ld + 4 * tc);
        const float av[4] = {a.x, a.y, a.z, a.w}, wv[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int v = 0; v < 4; v++) acc[u][v] = fmaf(av[u], wv[v], acc[u][v]);
    }
}

template <int TM>
struct InferLds {
    static constexpr int NC = TM == 128 ? 32 : 64;  // padded hidden width
    static constexpr int LA = TM + 4;
    static constexpr int act = 0;                                // [kKMax][LA]; later both hidden layers and y
    static constexpr int w1 = kKMax * LA;                        // [96][NC]
    static constexpr int w2 = w1 + (kWsIn + 1) * NC;             // [NC + 1][NC]
    static constexpr int w3 = w2 + (NC + 1) * NC;                // [NC + 1][12]
    static constexpr int total = w3 + (NC + 1) * 12;
};
static_assert(2 * 33 + kWsOut <= kKMax, "both hidden layers and y fit the input's rows (32 units)");

template <int TM>
__global__ void __launch_bounds__(256) k_ws_infer(Level L, Fields F, WsQ Q, const float* w, int nh, const float* stats,
                                                  long m, int ntiles) {
    extern __shared__ __align__(16) float smem_mlp[];
    using O = InferLds<TM>;
    constexpr int K1 = kWsIn + 1, LA = O::LA, NC = O::NC;
    __shared__ int s_node[TM];
    const int tid = (int)threadIdx.x;
    float* act = smem_mlp + O::act;
    // weights, columns and rows past the network's zero
    for (int e = tid; e < K1 * NC; e += 256) {
        const int k = e / NC, n = e % NC;
        smem_mlp[O::w1 + e] = n < nh ? w[k * nh + n] : 0.0f;
    }
    const float* g2 = w + K1 * nh;
    const float* g3 = g2 + (nh + 1) * nh;
    for (int e = tid; e < (nh + 1) * NC; e += 256) {
        const int k = e / NC, n = e % NC;
        smem_mlp[O::w2 + e] = n < nh ? g2[k * nh + n] : 0.0f;
    }
    for (int e = tid; e < (nh + 1) * 12; e += 256) {
        const int k = e / 12, n = e % 12;
        smem_mlp[O::w3 + e] = n < kWsOut ? g3[k * kWsOut + n] : 0.0f;
    }
    const int tr = tid / (NC / 4), tc = tid % (NC / 4);
    // this workgroup's run of tiles
    const unsigned lb = xcd_block(blockIdx.x, gridDim.x);
    const int t0 = (int)((long)ntiles * lb / gridDim.x), t1 = (int)((long)ntiles * (lb + 1) / gridDim.x);
    for (int tile = t0; tile < t1; tile++) {
        const long r0 = (long)tile * TM;
        __syncthreads();  // the weights, and y of the tile before
        if (tid < TM) s_node[tid] = (int)interior_node(L, min(r0 + tid, m - 1));
        __syncthreads();
        // features: one component of one node per thread and turn (whole
        // waves share a component)
        for (int e = tid; e < TM * kWsComp; e += 256) {
            const int row = e % TM, c = __builtin_amdgcn_readfirstlane(e / TM);
            const int t = s_node[row], i = t % L.ni;
            const int st[kWsPts] = {0, -1, 1, -L.ni, L.ni, -L.ni * L.nj, L.ni * L.nj,
                                    i >= 2 ? -2 : -i, i + 2 <= L.ni - 1 ? 2 : L.ni - 1 - i};
            const double* a = F.qn[c] + L.off;
            const double* b = F.qnm1[c] + L.off;
            const double* d = Q.q[c];
            double av[kWsPts], bv[kWsPts], dv[kWsPts];
#pragma unroll
            for (int s = 0; s < kWsPts; s++) {
                av[s] = a[t + st[s]];
                bv[s] = b[t + st[s]];
                dv[s] = d[t + st[s]];
            }
            double v[2 * kWsPts];
            double ss = 0.0;
#pragma unroll
            for (int s = 0; s < kWsPts; s++) {
                v[2 * s] = av[s] - bv[s];
                v[2 * s + 1] = bv[s] - dv[s];
                ss += v[2 * s] * v[2 * s] + v[2 * s + 1] * v[2 * s + 1];
            }
            const double rms = sqrt(ss / (2 * kWsPts));
            const int f0 = c * 2 * kWsPts, fq = kWsComp * 2 * kWsPts + c;
#pragma unroll
            for (int q = 0; q < 2 * kWsPts; q++) {
                const float x = rms > 0.0 ? (float)(v[q] / rms) : 0.0f;
                act[(f0 + q) * LA + row] = (x - stats[f0 + q]) * stats[kWsIn + f0 + q];
            }
            act[fq * LA + row] = ((float)av[0] - stats[fq]) * stats[kWsIn + fq];
            if (c == 0) act[kWsIn * LA + row] = 1.0f;
        }
        __syncthreads();
        float acc[4][4];
        infer_product<TM>(act, K1, smem_mlp + O::w1, NC, tr, tc, acc);
        __syncthreads();  // the input is dead: rows 0 .. nh hold the first hidden layer
        auto store_layer = [&](float* B) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int n = 4 * tc + v;
                if (n < nh)
                    *reinterpret_cast<float4*>(B + n * LA + 4 * tr) =
                        make_float4(tanhf(acc[0][v]), tanhf(acc[1][v]), tanhf(acc[2][v]), tanhf(acc[3][v]));
            }
            if (tc == 0) *reinterpret_cast<float4*>(B + nh * LA + 4 * tr) = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
        };
        store_layer(act);
        __syncthreads();
        infer_product<TM>(act, nh + 1, smem_mlp + O::w2, NC, tr, tc, acc);
        // the second hidden layer beside the first where both fit, else over it
        constexpr int second = TM == 128 ? 33 : 0;
        if (second == 0) __syncthreads();
        float* B2 = act + second * LA;
        store_layer(B2);
        __syncthreads();
        float* y = act + (TM == 128 ? 66 : 65) * LA;  // [10][LA]
        if (tc < 3) {
            infer_product<TM>(B2, nh + 1, smem_mlp + O::w3, 12, tr, tc, acc);
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (4 * tc + v < kWsOut)
                    *reinterpret_cast<float4*>(y + (4 * tc + v) * LA + 4 * tr) =
                        make_float4(acc[0][v], acc[1][v], acc[2][v], acc[3][v]);
        }
        __syncthreads();
        for (int e = tid; e < TM * kWsComp; e += 256) {
            const int row = e % TM, c = __builtin_amdgcn_readfirstlane(e / TM);
            if (r0 + row >= m) continue;
            const int t = s_node[row];
            const long g = L.off + t;
            const double qn = F.qn[c][g], qm = F.qnm1[c][g];
            const double d1 = qn - qm, d2 = qm - Q.q[c][t];
            double v = qn + (1.0 + (double)y[c * LA + row]) * d1 + (double)y[(kWsComp + c) * LA + row] * d2;
            if (c == 4) v = fmax(1.0e-07, v);
            F.q[c][g] = v;
        }
    }
}

// per-column sum and sum of squares over n rows (ld columns, first nc used),
// partial per block: part[blockIdx][2 nc]
__global__ void __launch_bounds__(256) k_colstats(const float* X, int ld, int nc, long n, double* part) {
    __shared__ double sh[256];
    const int c = (int)blockIdx.y;
    double s = 0.0, s2 = 0.0;
    for (long r = (long)blockIdx.x * 256 + threadIdx.x; r < n; r += (long)gridDim.x * 256) {
        const double v = X[r * ld + c];
        s += v;
        s2 += v * v;
    }
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[((long)blockIdx.x * nc + c) * 2] = sh[0];
    __syncthreads();
    sh[threadIdx.x] = s2;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[((long)blockIdx.x * nc + c) * 2 + 1] = sh[0];
}

unsigned nblk(long n, int b) { return (unsigned)((n + b - 1) / b); }

}  // namespace

// ---- launchers ----

void launch_ws_sample(hipStream_t s, const Level& L, const Fields& F, const WsQ& Q, float* X, float* T, long m,
                      unsigned long long seed, long step) {
    hipLaunchKernelGGL(k_ws_sample, dim3(nblk(m, 128)), dim3(128), 0, s, L, F, Q, X, T, m, seed, step);
}

void launch_ws_features(hipStream_t s, const Level& L, const Fields& F, const WsQ& Q, float* X, long r0, long m,
                        const float* stats) {
    hipLaunchKernelGGL(k_ws_features, dim3(nblk(m, 128)), dim3(128), 0, s, L, F, Q, X, r0, m, stats);
}

void launch_ws_extrap(hipStream_t s, const Level& L, const Fields& F, long m) {
    hipLaunchKernelGGL(k_ws_extrap, dim3(nblk(m, 256)), dim3(256), 0, s, L, F, m);
}

template <int TM>
static hipError_t ws_infer(hipStream_t s, const Level& L, const Fields& F, const WsQ& Q, const float* w, int nh,
                           const float* stats, long m) {
    const int lds = (int)sizeof(float) * InferLds<TM>::total;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_ws_infer<TM>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    const int ntiles = (int)((m + TM - 1) / TM);
    // two workgroups per CU (69 KB of LDS each with TM = 128)
    const unsigned grid = (unsigned)(ntiles < 512 ? ntiles : 512);
    hipLaunchKernelGGL(k_ws_infer<TM>, dim3(grid), dim3(256), lds, s, L, F, Q, w, nh, stats, m, ntiles);
    return hipGetLastError();
}

hipError_t launch_ws_infer(hipStream_t s, const Level& L, const Fields& F, const WsQ& Q, const float* w, int nh,
                           const float* stats, long m) {
    return nh <= 32 ? ws_infer<128>(s, L, F, Q, w, nh, stats, m) : ws_infer<64>(s, L, F, Q, w, nh, stats, m);
}

// the tile kernel in one of its modes; the hidden width picks the columns per
// thread (16 column groups)
template <int MODE>
static hipError_t mlp_tile(hipStream_t s, const MlpBuf& A, const float* w, int nh, int M, const float* X,
                           const float* T, long nsrc, unsigned long long seed, long it, const float* stats) {
    const int lds = (int)sizeof(float) * MlpLds(nh).total;
    const dim3 grid(nblk(M, kBM)), block(256);
    auto go = [&](auto kernel) {
        if (lds > 64 * 1024) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(kernel, grid, block, lds, s, A, w, nh, M, X, T, nsrc, seed, it, stats);
        return hipGetLastError();
    };
    return nh <= 32 ? go(k_mlp_tile<MODE, 2>) : go(k_mlp_tile<MODE, 4>);
}

hipError_t launch_mlp_forward(hipStream_t s, const MlpBuf& A, const float* w, int nh, int M) {
    return mlp_tile<kTileForward>(s, A, w, nh, M, nullptr, nullptr, 1, 0, 0, nullptr);
}

hipError_t launch_mlp_loss(hipStream_t s, const MlpBuf& A, const float* w, int nh, int M) {
    return mlp_tile<kTileLoss>(s, A, w, nh, M, nullptr, nullptr, 1, 0, 0, nullptr);
}

hipError_t launch_mlp_train(hipStream_t s, const MlpBuf& A, const float* w, int nh, int M, const float* X,
                            const float* T, long nsrc, unsigned long long seed, long it, const float* stats) {
    return mlp_tile<kTileTrain>(s, A, w, nh, M, X, T, nsrc, seed, it, stats);
}

int wgrad_parts(int M) { return (int)nblk(M, kWgRows); }
int mlp_tiles(int M) { return (int)nblk(M, kBM); }

void launch_mlp_grad(hipStream_t s, const MlpBuf& A, int nh, int M, int np, float* g, double* loss, float* w, float* m,
                     float* v, float lr, float b1, float b2, float eps, float c1, float c2) {
    const int parts = wgrad_parts(M);
    const int tiles = wg_tiles(kWsIn + 1, nh) + wg_tiles(nh + 1, nh) + wg_tiles(nh + 1, kWsOut);
    hipLaunchKernelGGL(k_wgrad, dim3(parts, tiles), dim3(128), 0, s, A, nh, M, np);
    const AdamArgs a{w, m, v, lr, b1, b2, eps, c1, c2};
    hipLaunchKernelGGL(k_grad_sum, dim3(nblk(np, 256) + 1), dim3(256), 0, s, A.P, parts, np, g, a, A.lpart,
                       mlp_tiles(M), loss);
}

void launch_colstats(hipStream_t s, const float* X, int ld, int nc, long n, double* part, int nparts) {
    hipLaunchKernelGGL(k_colstats, dim3(nparts, nc), dim3(256), 0, s, X, ld, nc, n, part);
}

}  // namespace desalm
