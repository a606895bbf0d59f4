// Kernels of the block responses (blocks.h).
#include "blocks.h"
#include "launch.h"

#include <algorithm>
#include <cmath>

namespace parode {
namespace k {

// The kernels that hold a whole map in one work-group's LDS.
constexpr int kBN = 64;             // states (n_a), outputs a step
constexpr int kBP = kBN + 1;        // LDS pitch
constexpr int kBM = 32;             // inputs

// ------------------------------------------------------------------ products
// One 16 x 16 tile of X Y from LDS (v_mfma_f64_16x16x4f64): lane l holds
// X[i0 + l%16][k + l/16] and Y[k + l/16][j0 + l%16] (YT: Y given transposed);
// D: register v of lane l is row i0 + 4v + l/16, column j0 + l%16.
template <bool YT>
__device__ __forceinline__ doublex4 lds_tile(const double* X, int px, const double* Y, int py,
                                             int i0, int j0, int kk)
{
    const int l16 = threadIdx.x & 15, q4 = (threadIdx.x >> 4) & 3;
    doublex4 acc = {0.0, 0.0, 0.0, 0.0};
    const double* xr = X + (i0 + l16) * px + q4;
    const double* yr = YT ? Y + (j0 + l16) * py + q4 : Y + q4 * py + j0 + l16;
    const int ys = YT ? 1 : py;
    // (kk: whole 16; a chunk's operands are read before its products: one LDS round
    // trip for four)
#pragma unroll 1
    for (int k = 0; k < kk; k += 16) {
        double x[4], y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            x[u] = xr[k + 4 * u];
            y[u] = yr[(k + 4 * u) * ys];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[u], y[u], acc, 0, 0, 0);
    }
    return acc;
}

// ------------------------------------------------------------------- the map
struct BlkTables {
    BlockShape s;
    double h;
    Rk4Coef rk;
    AbmCoef ab;
    const float *A, *B, *C, *D, *x0;
    const void* U;
    double *PT, *QT, *OT, *Ht, *DL, *seed;
    float* Y;
    int ni, nq;   // steps of a slice of OT (and Ht), of a slice of QT
    long gx;
};
// LDS of a work-group (doubles): P = P_l (transposed power, [n16][kBP]), the rows R of
// its slice and the input block G ([s m] rows); the map's own arrays lie in R's and
// G's places (RK4) or behind them (ABM)
constexpr int kTabR = kBN * kBP, kTabG = 2 * kBN * kBP, kTabMap = 3 * kBN * kBP;
constexpr int kTabLds = kTabMap + 5280;
static_assert(2 * kBN * kBP + 4 * kBN * (kBM + 1) <= kTabLds, "room for the RK4 map");


// Z = X Y with the reference's rounding: float products, sequential float sums.
__device__ __forceinline__ void lds_mul_seq(int r, int kk, int c, const float* X, int px,
                                            const float* Y, int py, float* Z, int pz)
{
#pragma clang fp contract(off)
    for (int t = threadIdx.x; t < r * c; t += 1024) {
        const int i = t / c, j = t - i * c;
        float v = 0.0f;
        for (int q = 0; q < kk; ++q) {
            const float pr = X[i * px + q] * Y[q * py + j];
            v = v + pr;
        }
        Z[i * pz + j] = v;
    }
}

// A work-group makes a small system's map (n_a <= 64, m <= 32) in LDS, P_0 and G to
// its tables' places, and (store) to memory: the step map M, the block input G, the direct terms F and the state's shift D
// (blocks.h).  RK4 by Horner's scheme, M = I + hA (I + hA/2 (I + hA/3 (I +
// hA/4))), beside the products A^k B; with the reference's rounding by its own
// products A^2, A^3, A^4.  A chain of a few dependent 64 x 64 products: latency.
__device__ __forceinline__ void d_blk_map_rk4(const BlkTables& a, double* lds, bool store)
{
#pragma clang fp contract(off)
    const BlockShape& s = a.s;
    const int n = s.n, m = s.m, p = s.p, tid = threadIdx.x, wave = tid >> 6;
    const int n16 = (n + 15) & ~15, m16 = (m + 15) & ~15, nt = n16 / 16, mt = m16 / 16;
    constexpr int KP = kBM + 1;
    double* As = lds;
    double* Ts = lds + kBN * kBP;
    double* Kb[4];
    for (int q = 0; q < 4; ++q) Kb[q] = lds + 2 * kBN * kBP + q * kBN * KP;
    const int l16 = tid & 15, q4 = (tid >> 4) & 3;
    for (int t = tid; t < n16 * m16; t += 1024) {
        const int i = t / m16, j = t - i * m16;
        const bool in = i < n && j < m;
        Kb[0][i * KP + j] = in ? (double)a.B[(long)i * m + j] : 0.0;
        for (int q = 1; q < 4; ++q) Kb[q][i * KP + j] = 0.0;
    }
    if (s.mirror) {
        float* A1 = reinterpret_cast<float*>(As);
        float* A2 = A1 + kBN * kBP;
        float* A3 = reinterpret_cast<float*>(Ts);
        float* A4 = A3 + kBN * kBP;
        float* Bf = reinterpret_cast<float*>(Kb[0]);   // B, AB, A2B, A3B in float
        for (int t = tid; t < n * n; t += 1024) A1[t / n * kBP + t % n] = a.A[t];
        __syncthreads();
        for (int t = tid; t < n * m; t += 1024) Bf[t / m * KP + t % m] = a.B[t];
        __syncthreads();
        float* AB = Bf + kBN * KP;
        float* A2B = AB + kBN * KP;
        float* A3B = A2B + kBN * KP;
        lds_mul_seq(n, n, n, A1, kBP, A1, kBP, A2, kBP);
        lds_mul_seq(n, n, m, A1, kBP, Bf, KP, AB, KP);
        __syncthreads();
        lds_mul_seq(n, n, n, A2, kBP, A1, kBP, A3, kBP);
        lds_mul_seq(n, n, m, A2, kBP, Bf, KP, A2B, KP);
        __syncthreads();
        lds_mul_seq(n, n, n, A1, kBP, A3, kBP, A4, kBP);
        lds_mul_seq(n, n, m, A3, kBP, Bf, KP, A3B, KP);
        __syncthreads();
        // the combinations (RungeKutta4thOrder.cpp:48-57), in registers first:
        // the float products share their LDS with what follows
        double mv[4], bv[2][3];
        for (int u = 0; u < 4; ++u) {
            const int t = tid + u * 1024;
            mv[u] = 0.0;
            if (t >= n * n) continue;
            const int i = t / n, j = t - i * n, x = i * kBP + j;
            double v = ((i == j) ? 1.0 : 0.0) + a.rk.h * (double)A1[x];
            v = v + a.rk.c2 * (double)A2[x];
            v = v + a.rk.c3 * (double)A3[x];
            v = v + a.rk.c4 * (double)A4[x];
            mv[u] = (double)(float)v;
        }
        for (int u = 0; u < 2; ++u) {
            const int t = tid + u * 1024;
            if (t >= n * m) continue;
            const int x = t / m * KP + t % m;
            const double b = Bf[x], ab = AB[x], a2b = A2B[x], a3b = A3B[x];
            bv[u][0] = (double)(float)((1.0 / 6.0) * (((a.rk.h * b + a.rk.s1 * ab) + a.rk.s2 * a2b) + a.rk.s3 * a3b));
            bv[u][1] = (double)(float)((1.0 / 6.0) * ((a.rk.t0 * b + a.rk.t1 * ab) + a.rk.t2 * a2b));
            bv[u][2] = (double)(float)(a.rk.u0 * b);
        }
        __syncthreads();
        for (int t = tid; t < n16 * n16; t += 1024) Ts[t / n16 * kBP + t % n16] = 0.0;
        for (int t = tid; t < n16 * m16; t += 1024)
            for (int q = 0; q < 4; ++q) Kb[q][t / m16 * KP + t % m16] = 0.0;
        __syncthreads();
        for (int u = 0; u < 4; ++u) {
            const int t = tid + u * 1024;
            if (t < n * n) Ts[t / n * kBP + t % n] = mv[u];
        }
        for (int u = 0; u < 2; ++u) {
            const int t = tid + u * 1024;
            if (t >= n * m) continue;
            const int x = t / m * KP + t % m;
            for (int q = 0; q < 3; ++q) Kb[q == 2 ? 3 : q][x] = bv[u][q];
        }
        __syncthreads();
    } else {
        for (int t = tid; t < n16 * n16; t += 1024) {
            const int i = t / n16, j = t - i * n16;
            const double v = (i < n && j < n) ? (double)a.A[(long)i * n + j] : 0.0;
            As[i * kBP + j] = v;
            Ts[i * kBP + j] = (i == j ? 1.0 : 0.0) + (a.h / 4.0) * v;
        }
        __syncthreads();
        for (int st = 3; st >= 1; --st) {
            // tiles of A T, then of A (A^k B); a wave has at most two items
            doublex4 acc[2];
            const int items = nt * nt + nt * mt;
            for (int u = 0; u < 2; ++u) {
                const int w = wave + 16 * u;
                if (w < nt * nt)
                    acc[u] = lds_tile<false>(As, kBP, Ts, kBP, w / nt * 16, w % nt * 16, n16);
                else if (w < items)
                    acc[u] = lds_tile<false>(As, kBP, Kb[3 - st], KP, (w - nt * nt) / mt * 16,
                                             (w - nt * nt) % mt * 16, n16);
            }
            __syncthreads();
            const double c = a.h / (double)st;
            for (int u = 0; u < 2; ++u) {
                const int w = wave + 16 * u;
                if (w < nt * nt) {
                    for (int v = 0; v < 4; ++v) {
                        const int i = w / nt * 16 + 4 * v + q4, j = w % nt * 16 + l16;
                        Ts[i * kBP + j] = (i == j ? 1.0 : 0.0) + c * acc[u][v];
                    }
                } else if (w < items) {
                    for (int v = 0; v < 4; ++v) {
                        const int i = (w - nt * nt) / mt * 16 + 4 * v + q4;
                        const int j = (w - nt * nt) % mt * 16 + l16;
                        Kb[4 - st][i * KP + j] = acc[u][v];
                    }
                }
            }
            __syncthreads();
        }
        for (int t = tid; t < n16 * m16; t += 1024) {
            const int x = t / m16 * KP + t % m16;
            const double b = Kb[0][x], ab = Kb[1][x], a2b = Kb[2][x], a3b = Kb[3][x];
            Kb[0][x] = (1.0 / 6.0) * (((a.rk.h * b + a.rk.s1 * ab) + a.rk.s2 * a2b) + a.rk.s3 * a3b);
            Kb[1][x] = (1.0 / 6.0) * ((a.rk.t0 * b + a.rk.t1 * ab) + a.rk.t2 * a2b);
            Kb[3][x] = a.rk.u0 * b;
        }
        __syncthreads();
    }
    // Ts = M; Kb[0], Kb[1], Kb[3] = the three input blocks of a step.
    // G = [B1 + M B3 | B2], the shift and the direct term from B3
    const int gi = wave / mt * 16, gj = wave % mt * 16;
    const bool mine = wave < nt * mt;   // (at most 4 x 2 tiles)
    double g1[4], g2[4];
    if (mine) {
        const doublex4 acc = lds_tile<false>(Ts, kBP, Kb[3], KP, gi, gj, n16);
        for (int v = 0; v < 4; ++v) {
            const int x = (gi + 4 * v + q4) * KP + gj + l16;
            g1[v] = Kb[0][x] + acc[v];
            g2[v] = Kb[1][x];
        }
    }
    for (int t = tid; t < n16 * n16; t += 1024) {
        const int r = t / n16, c = t - r * n16;
        const double v = r < n && c < n ? Ts[c * kBP + r] : 0.0;
        As[r * kBP + c] = v;   // (P)
        if (store && r < n && c < n) a.PT[(long)r * n + c] = v;
    }
    if (store) {
        for (int t = tid; t < m * n; t += 1024) a.DL[t] = Kb[3][(t % n) * KP + t / n];
        double* F = a.Ht + (long)s.s * (s.T - 1) * m * p;
        for (int t = tid; t < m * p; t += 1024) {
            const int j = t / p, o = t - j * p;
            double v = 0.0;
            if (s.useC)
                for (int i = 0; i < n; ++i) v = fma((double)a.C[(long)o * n + i], Kb[3][i * KP + j], v);
            else
                v = Kb[3][o * KP + j];
            F[t] = v + (s.useD ? (double)a.D[(long)o * m + j] : 0.0);
        }
    }
    __syncthreads();
    double* G = lds + kTabG;
    double* GT = a.QT + (long)s.s * (s.T - 1) * m * n;
    for (int t = tid; t < kBN * n16; t += 1024) G[t / n16 * kBP + t % n16] = 0.0;
    __syncthreads();
    if (!mine) return;
    for (int v = 0; v < 4; ++v) {
        const int i = gi + 4 * v + q4, j = gj + l16;
        if (i >= n || j >= m) continue;
        G[j * kBP + i] = g1[v];
        G[(m + j) * kBP + i] = g2[v];
        if (store) {
            GT[(long)j * n + i] = g1[v];
            GT[(long)(m + j) * n + i] = g2[v];
        }
    }
}

// The ABM companion of a small system (n <= 16): its dense block row R, the
// blocks V_0 = B_4, V_t = B_{4-t} + sum_{i < t} M_{4-t+i} V_i (M_b: R's blocks,
// oldest first; B_q: the step's input blocks), which give
// G = [V_1; V_2; V_3; V_4], D_r = [0 (r blocks); V_0 .. V_{3-r}], F_r = C V_{3-r}.
__device__ __forceinline__ void d_blk_map_abm(const BlkTables& a, double* lds, bool store)
{
#pragma clang fp contract(off)
    const BlockShape& s = a.s;
    const int n = s.n, m = s.m, p = s.p, na = s.na, tid = threadIdx.x;
    constexpr int AP = 17, KP = kBM + 1;
    double* A1 = lds + kTabMap;        // [16][AP]
    double* A2 = A1 + 16 * AP;
    double* B1 = A2 + 16 * AP;         // [16][KP]
    double* AB = B1 + 16 * KP;
    double* R = AB + 16 * KP;          // [16][kBP]
    double* V = R + 16 * kBP;          // [5][16][KP]
    for (int t = tid; t < n * n; t += 1024) A1[t / n * AP + t % n] = a.A[t];
    for (int t = tid; t < n * m; t += 1024) B1[t / m * KP + t % m] = a.B[t];
    __syncthreads();
    for (int t = tid; t < n * (n + m); t += 1024) {
        const int i = t / (n + m), j = t - i * (n + m);
        const double* y = j < n ? A1 + j : B1 + (j - n);
        const int py = j < n ? AP : KP;
        double v = 0.0;
        if (s.mirror) {
            float f = 0.0f;
            for (int q = 0; q < n; ++q) {
                const float pr = (float)A1[i * AP + q] * (float)y[q * py];
                f = f + pr;
            }
            v = f;
        } else {
#pragma unroll 4
            for (int q = 0; q < n; ++q) v = fma(A1[i * AP + q], y[q * py], v);
        }
        if (j < n)
            A2[i * AP + j] = v;
        else
            AB[i * KP + j - n] = v;
    }
    __syncthreads();
    auto rnd = [&](double v) { return s.mirror ? (double)(float)v : v; };
    const AbmCoef& c = a.ab;
    for (int t = tid; t < n * n; t += 1024) {
        const int i = t / n, j = t - i * n;
        const double id = (i == j) ? 1.0 : 0.0, x = A1[i * AP + j], x2 = A2[i * AP + j];
        R[i * kBP + j] = rnd(c.a3A2 * x2);
        R[i * kBP + n + j] = rnd(c.a2A * x + c.a2A2 * x2);
        R[i * kBP + 2 * n + j] = rnd(c.a1A * x + c.a1A2 * x2);
        R[i * kBP + 3 * n + j] = rnd((id + c.a0A * x) + c.a0A2 * x2);
    }
    auto bq = [&](int q, int i, int j) {   // the step's input block q
        const double b = B1[i * KP + j], ab = AB[i * KP + j];
        return q == 0 ? rnd(c.b3AB * ab) : q == 1 ? rnd(c.b2B * b + c.b2AB * ab)
             : q == 2 ? rnd(c.b1B * b + c.b1AB * ab) : q == 3 ? rnd(c.b0B * b + c.b0AB * ab)
             : rnd(c.bm1 * b);
    };
    for (int st = 0; st < 5; ++st) {
        __syncthreads();
        for (int t = tid; t < n * m; t += 1024) {
            const int i = t / m, j = t - i * m;
            double v = bq(4 - st, i, j);
            for (int b = 0; b < st; ++b)
#pragma unroll 4
                for (int q = 0; q < n; ++q)
                    v = fma(R[i * kBP + (4 - st + b) * n + q], V[(b * 16 + q) * KP + j], v);
            V[(st * 16 + i) * KP + j] = v;
        }
    }
    __syncthreads();
    const int n16 = (na + 15) & ~15;
    for (int t = tid; t < n16 * n16; t += 1024) {
        const int j = t / n16, i = t - j * n16;   // PT[j][i] = M[i][j]
        double v = 0.0;
        if (i < na && j < na) v = i < 3 * n ? (j == i + n ? 1.0 : 0.0) : R[(i - 3 * n) * kBP + j];
        lds[j * kBP + i] = v;
        if (store && i < na && j < na) a.PT[(long)j * na + i] = v;
    }
    double* GT = a.QT + (long)(s.T - 1) * m * na;
    for (int t = tid; t < kBN * n16; t += 1024) {
        const int j = t / n16, x = t - j * n16, b = x / n, i = x - b * n;
        const double v = j < m && x < na ? V[((b + 1) * 16 + i) * KP + j] : 0.0;
        lds[kTabG + j * kBP + x] = v;
        if (store && j < m && x < na) GT[(long)j * na + x] = v;
    }
    if (!store) return;
    for (int t = tid; t < 4 * m * na; t += 1024) {
        const int rj = t / na, x = t - rj * na, r = rj / m, j = rj - r * m, b = x / n, i = x - b * n;
        a.DL[t] = b >= r ? V[((b - r) * 16 + i) * KP + j] : 0.0;
    }
    double* F = a.Ht + (long)(s.T - 1) * m * p;
    for (int t = tid; t < 4 * m * p; t += 1024) {
        const int rj = t / p, o = t - rj * p, r = rj / m, j = rj - r * m;
        double v = 0.0;
        if (s.useC) {
#pragma unroll 4
            for (int i = 0; i < n; ++i)
                v = fma((double)a.C[(long)o * n + i], V[((3 - r) * 16 + i) * KP + j], v);
        } else {
            v = V[((3 - r) * 16 + o) * KP + j];
        }
        F[t] = v + (r == 3 && s.useD ? (double)a.D[(long)o * m + j] : 0.0);
    }
}

// The outputs of the ABM start-up states x_0, x_1, x_2 (inputs: rows 0, 2, 4 of
// the h/2 grid; AdamsMoulton.cpp:106-116), FP64 sums.
template <typename TU>
__device__ __forceinline__ void d_start_outputs(const BlockShape& s, const float* C, const float* D,
                                                const double* X0, const TU* U, float* Y)
{
    for (int t = threadIdx.x; t < 3 * s.p; t += blockDim.x) {
        const int e = t / s.p, o = t - e * s.p;
        double v = 0.0;
        if (s.useC)
            for (int i = 0; i < s.n; ++i) v = fma((double)C[(long)o * s.n + i], X0[e * s.n + i], v);
        else
            v = X0[e * s.n + o];
        if (s.useD)
            for (int j = 0; j < s.m; ++j)
                v = fma((double)D[(long)o * s.m + j], (double)U[(long)2 * e * s.m + j], v);
        Y[t] = (float)v;
    }
}
template <typename TU>
__global__ __launch_bounds__(1024) void k_blk_start_outputs(BlockShape s, const float* C,
                                                            const float* D, const double* X0,
                                                            const TU* U, float* Y)
{
    d_start_outputs<TU>(s, C, D, X0, U, Y);
}

// The seed of a plan's solve (a work-group of its own): x0, or the ABM start-up states
// and the outputs of the first three (inputs: rows 0, 2, 4 of the h/2 grid).
template <typename TU>
__device__ __forceinline__ void d_blk_seed(const BlkTables& a)
{
    const BlockShape& s = a.s;
    const TU* U = static_cast<const TU*>(a.U);
    if (s.method == 0) {
        for (int i = threadIdx.x; i < s.n; i += 1024) a.seed[i] = (double)a.x0[i];
        return;
    }
    startup_rows<TU, 4>(s.mirror, s.n, s.m, a.h, a.A, a.B, a.x0, U, a.seed);
    __syncthreads();
    d_start_outputs<TU>(s, a.C, a.D, a.seed, U, a.Y);
}

// ---------------------------------------------------------------- the tables
// P <- P^2 in LDS (and, with R, the rows of R by P or P^T): every tile from the
// old values, a barrier, the new values, a barrier.  Sixteen waves, two tiles
// of P^2 and rows each.  from/to: the rows of R that are read and written.
template <bool ROWS, bool YT>
__device__ __forceinline__ void lds_step(double* P, int n16, double* R, int from, int to, int rows,
                                         bool square)
{
    const int wave = threadIdx.x >> 6, l16 = threadIdx.x & 15, q4 = (threadIdx.x >> 4) & 3;
    const int nt = n16 / 16, sq = square ? nt * nt : 0, rt = (rows + 15) / 16;
    const int items = sq + (ROWS ? rt * nt : 0);
    doublex4 acc[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int w = wave + 16 * u;
        if (w < sq)
            acc[u] = lds_tile<false>(P, kBP, P, kBP, w / nt * 16, w % nt * 16, n16);
        else if (w < items)
            acc[u] = lds_tile<YT>(R + from * kBP, kBP, P, kBP, (w - sq) / nt * 16,
                                  (w - sq) % nt * 16, n16);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int w = wave + 16 * u;
        if (w >= items) continue;
        const bool isR = w >= sq;
        const int x = isR ? w - sq : w, i0 = x / nt * 16, j = x % nt * 16 + l16;
        for (int v = 0; v < 4; ++v) {
            const int i = i0 + 4 * v + q4;
            if (!isR)
                P[i * kBP + j] = acc[u][v];
            else if (i < rows)
                R[(to + i) * kBP + j] = acc[u][v];
        }
    }
    __syncthreads();
}

// Map and tables of a small system (n_a, p, s m <= 64).  Every work-group makes the
// map for itself (a launch of its own for it cost 5 us more).  Work-group 0 squares P_0 up
// to P_lb; the others each make a slice of OT and Ht (ni steps) or of QT (nq
// steps) and square P_l for themselves, since passing it between work-groups
// would cost a launch per level; the last, if the solve's start is known, its
// seed.  A slice of steps [i0, i0 + 2^a) takes the levels below a by doubling its
// rows and the others by the bits of i0 (the powers commute).  Time: the map and
// lb dependent products of 64 x 64 in one compute unit.
template <typename TU>
__device__ __forceinline__ void d_blk_tables(const VBlock vb, const BlkTables& a, double* lds)
{
    const BlockShape& s = a.s;
    const int na = s.na, n16 = (na + 15) & ~15, tid = threadIdx.x, m = s.m, p = s.p;
    const int sm = s.s * m, nO = s.T / a.ni;
    const long nn = (long)na * na;
    if (a.x0 && vb.x == a.gx - 1) {
        d_blk_seed<TU>(a);
        return;
    }
    if (s.method == 0)
        d_blk_map_rk4(a, lds, vb.x == 0);
    else
        d_blk_map_abm(a, lds, vb.x == 0);
    __syncthreads();
    double* P = lds;
    double* G = lds + kTabG;
    if (vb.x == 0) {
        for (int l = 0; l < s.lb; ++l) {
            lds_step<false, false>(P, n16, nullptr, 0, 0, 0, true);
            double* out = a.PT + (l + 1) * nn;
            for (int t = tid; t < nn; t += 1024) out[t] = P[t / na * kBP + t % na];
        }
        return;
    }
    const bool isO = vb.x <= nO;
    const int w = (int)vb.x - 1 - (isO ? 0 : nO);
    const int ns = isO ? a.ni : a.nq, per = isO ? p : sm, i0 = w * ns, rows = ns * per;
    const int off = na - s.n;
    // the rows of step 0: those of C E, or G itself
    double* R = isO ? lds + kTabR : G;
    if (isO)
        for (int t = tid; t < kBN * n16; t += 1024) {
            const int r = t / n16, c = t - r * n16;
            double v = 0.0;
            if (r < per && c >= off && c < na)
                v = s.useC ? (double)a.C[(long)r * s.n + c - off] : (c - off == r ? 1.0 : 0.0);
            R[r * kBP + c] = v;
        }
    __syncthreads();
    for (int l = 0; l < s.lb; ++l) {
        const bool more = l + 1 < s.lb;
        const bool dbl = (1 << l) < ns;
        const bool mul = dbl || ((i0 >> l) & 1);
        const int cnt = dbl ? per << l : rows;
        // rows of OT are multiplied by P_l (PT transposed), rows of QT by P_l^T
        if (!mul)
            lds_step<false, false>(P, n16, nullptr, 0, 0, 0, more);
        else if (isO)
            lds_step<true, true>(P, n16, R, 0, dbl ? cnt : 0, cnt, more);
        else
            lds_step<true, false>(P, n16, R, 0, dbl ? cnt : 0, cnt, more);
    }
    if (!isO) {
        for (int t = tid; t < rows * na; t += 1024) {
            const int r = t / na, c = t - r * na, i = r / sm;
            if (i0 + i > 0)   // (step 0 is G itself, which the map made)
                a.QT[((long)(s.T - 1 - i0 - i) * sm + (r - i * sm)) * na + c] = R[r * kBP + c];
        }
        return;
    }
    const long cols = (long)s.T * p;
    for (int t = tid; t < rows * na; t += 1024) {
        const int c = t / rows, r = t - c * rows;
        a.OT[c * cols + (long)i0 * p + r] = R[r * kBP + c];
    }
    // Ht of step k: (C E M^k) G, [s m][p], for a lag of k + 1 steps
    const int wave = tid >> 6, l16 = tid & 15, q4 = (tid >> 4) & 3;
    const int ct = (sm + 15) / 16, rt = (rows + 15) / 16;
    for (int x = wave; x < rt * ct; x += 16) {
        const doublex4 acc = lds_tile<true>(R, kBP, G, kBP, x / ct * 16, x % ct * 16, n16);
        const int j = x % ct * 16 + l16;
        for (int v = 0; v < 4; ++v) {
            const int r = x / ct * 16 + 4 * v + q4, i = r / p, k = i0 + i;
            if (r < rows && j < sm && k <= s.T - 2)
                a.Ht[((long)(s.T - 2 - k) * sm + j) * p + (r - i * p)] = acc[v];
        }
    }
}

template <typename TU>
__global__ __launch_bounds__(1024) void k_blk_tables(const BlkTables a)
{
    __shared__ double lds[kTabLds];
    d_blk_tables<TU>(VBlock{(long)blockIdx.x, (long)blockIdx.y, (long)gridDim.x}, a, lds);
}

// ---------------------------------------------------------------- the passes
// Pass 1 (OUT false): Z[b][:] = window of block b times QT.
// Pass 2 (OUT true):  Y[b T p ...] = [Z_b, window of block b] times [OT; Ht].
// Both are products of Nb rows; the window part of pass 2 is causal: column
// (i, o) takes the window's first (s i + taps) m values only.
struct BlkPass {
    int na, m, p, s, T, taps;
    int cols, kz, ku;       // columns; K of the state part and of the window part
    long nb, nReal;
    const void* U;
    long blockU;            // samples between blocks' windows
    int gm;                 // samples skipped after each window row
    unsigned magic;         // of m (k / m by multiply-high; m = 1: k itself)
    long last;              // last window row that is there
    const double *Z, *OT, *BU;   // BU: QT or Ht
    double* S;              // pass 1's output
    float* Y;               // pass 2's output
    const double* seed;     // pass 2, RK4: the first state, and D (or null)
    const float* D;
    double* PT;             // pass 1: work-group gx * gy squares P_lb .. P_{L-2}
    int lb, L;
    long gx, gy;
};

__device__ __forceinline__ bool not_finite(double v) { return !(fabs(v) <= 1.7976931348623157e308); }

// offset of window value k of a block (its samples start at u)
__device__ __forceinline__ long win(const BlkPass& a, int k)
{
    if (a.gm == 0) return k;
    const int r = a.m == 1 ? k : (int)__umulhi((unsigned)k, a.magic);
    return k + (long)r * a.gm;
}
// window values of block b that are there
__device__ __forceinline__ int win_len(const BlkPass& a, long b)
{
    const long rows = a.last + 1 - b * a.s * a.T;
    const long k = (rows < 0 ? 0 : rows) * a.m;
    return k < a.ku ? (int)k : a.ku;
}

// RK4's first outputs depend on x_0 alone (and u_0 through D)
__device__ __forceinline__ bool first_output(const BlkPass& a, long b, int col)
{
    return a.taps == 1 && b == 0 && col < a.p;
}

// One output of pass 2, term by term and only over the samples it depends on:
// for tiles that hold a sample that is not finite, which the tile's products
// would carry (times zero) into the outputs before it.
template <typename TU>
__device__ double blk_output(const BlkPass& a, long b, int col)
{
    const int i = col / a.p, o = col - i * a.p;
    double y = 0.0;
    const TU* u = static_cast<const TU*>(a.U) + b * a.blockU;
    if (first_output(a, b, col)) {   // from x_0 itself, not from x_0 less a shift by u_0
        for (int k = 0; k < a.kz; ++k) y = fma(a.seed[k], a.OT[(long)k * a.cols + col], y);
        if (a.D)
            for (int k = 0; k < a.m; ++k) y = fma((double)u[k], (double)a.D[(long)o * a.m + k], y);
        return y;
    }
    for (int k = 0; k < a.kz; ++k) y = fma(a.Z[b * a.na + k], a.OT[(long)k * a.cols + col], y);
    const double* h = a.BU + (long)a.s * (a.T - 1 - i) * a.m * a.p + o;
    int ke = (a.s * i + a.taps) * a.m;
    const int kl = win_len(a, b);
    ke = ke < kl ? ke : kl;
    for (int k = 0; k < ke; ++k) y = fma((double)u[win(a, k)], h[(long)k * a.p], y);
    return y;
}

__device__ __forceinline__ void blk_store(const BlkPass& a, bool out, long b, int col, double v)
{
    if (!out) {
        a.S[b * a.na + col] = v;
    } else if (b * a.T + col / a.p < a.nReal) {
        a.Y[b * a.cols + col] = (float)v;
    }
}

// Few tiles: 16 R x 16 R tiles whose K is split over NW waves, operands straight
// from the caches, 16 loads of a wave in flight; the waves' partial tiles meet
// in LDS.  Bound by the latency of those loads and by the caches (R = 2 halves
// its bytes per product); used while the 64 x 64 tiles would not fill the
// compute units.
template <typename TU, bool OUT, int NW, int R>
__device__ __forceinline__ void d_blk_split(const VBlock vb, const BlkPass& a, double* part,
                                            int* bad)
{
    constexpr int kT = 16 * R, kW = 256 * R * R;   // tile side, values of a partial tile
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15, q4 = lane >> 4;
    const long b0 = vb.y * kT;
    const int j0 = (int)vb.x * kT;
    // a lane's rows and columns (those past the last repeat it): row 16 r + l16
    // from u[r], its samples zero from k = kl[r] on; the factors of column
    // 16 r + l16 from h[r], zero from k = kcol[r] on
    const TU* u[R];
    const double* h[R];
    int kl[R], kcol[R], col[R];
    long row[R];
    int kEnd = a.ku, kMin = a.ku, stride = a.na;
    if (OUT) {
        const int jl = j0 + kT - 1 < a.cols ? j0 + kT - 1 : a.cols - 1;
        kEnd = (a.s * (jl / a.p) + a.taps) * a.m;
        kMin = (a.s * (j0 / a.p) + a.taps) * a.m;
        stride = a.p;
        if (threadIdx.x == 0) *bad = 0;
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        row[r] = b0 + 16 * r + l16 < a.nb ? b0 + 16 * r + l16 : a.nb - 1;
        col[r] = j0 + 16 * r + l16 < a.cols ? j0 + 16 * r + l16 : a.cols - 1;
        u[r] = static_cast<const TU*>(a.U) + row[r] * a.blockU;
        const int w = win_len(a, row[r]);
        kl[r] = w < kEnd ? w : kEnd;
        kcol[r] = a.ku;
        h[r] = a.BU + col[r];
        if (OUT) {
            const int i = col[r] / a.p;
            kcol[r] = (a.s * i + a.taps) * a.m;
            h[r] = a.BU + (long)a.s * (a.T - 1 - i) * a.m * a.p + (col[r] - i * a.p);
        }
    }
    const int zs = OUT ? (a.kz + 3) / 4 : 0, us = (kEnd + 3) / 4, per = (zs + us + NW - 1) / NW;
    const int kb = wave * per, ke = kb + per < zs + us ? kb + per : zs + us;
    doublex4 acc[R][R];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int c = 0; c < R; ++c) acc[r][c] = doublex4{0.0, 0.0, 0.0, 0.0};
    constexpr int UN = 8 / R;
    double x[UN][R], y[UN][R];
    auto multiply = [&] {
#pragma unroll
        for (int t = 0; t < UN; ++t)
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int c = 0; c < R; ++c)
                    acc[r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[t][r], y[t][c], acc[r][c], 0,
                                                                     0, 0);
    };
    int k = kb;
    if (OUT) {
        const int kz = ke < zs ? ke : zs;
        for (; k < kz; k += UN) {
#pragma unroll
            for (int t = 0; t < UN; ++t) {
                const int j = (k + t) * 4 + q4;
                const bool in = k + t < kz && j < a.kz;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    x[t][r] = in ? a.Z[row[r] * a.na + j] : 0.0;
                    y[t][r] = in ? a.OT[(long)j * a.cols + col[r]] : 0.0;
                }
            }
            multiply();
        }
        k = kb > zs ? kb : zs;
    }
    bool nf = false;
    if (OUT && first_output(a, b0, j0)) kMin = 0;
    for (; k < ke; k += UN) {
#pragma unroll
        for (int t = 0; t < UN; ++t) {
            const int j = (k - zs + t) * 4 + q4;
            const bool in = k + t < ke;
            const int at = win(a, j);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                x[t][r] = (in && j < kl[r]) ? (double)u[r][at] : 0.0;
                y[t][r] = (in && j < kcol[r]) ? h[r][(long)j * stride] : 0.0;
                if (OUT) nf = nf || (j >= kMin && not_finite(x[t][r]));
            }
        }
        multiply();
    }
    if (OUT && nf) *bad = 1;
    // D[i][j] is in lane j + 16 (i % 4), register i / 4
    if (R > 1 || wave > 0) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < R; ++c)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    part[(R > 1 ? wave : wave - 1) * kW + (16 * r + 4 * v + q4) * kT + 16 * c + l16] =
                        acc[r][c][v];
    }
    __syncthreads();
    if (OUT && *bad) {
        for (int t = threadIdx.x; t < kW; t += NW * 64) {
            const long bb = b0 + t / kT;
            const int cc = j0 + t % kT;
            if (bb < a.nb && cc < a.cols) blk_store(a, true, bb, cc, blk_output<TU>(a, bb, cc));
        }
        return;
    }
    if (R > 1) {   // a value's parts are added in wave order, each by one thread
        for (int t = threadIdx.x; t < kW; t += NW * 64) {
            double v = part[t];
#pragma unroll
            for (int g = 1; g < NW; ++g) v += part[g * kW + t];
            const long bb = b0 + t / kT;
            const int cc = j0 + t % kT;
            if (bb < a.nb && cc < a.cols) blk_store(a, OUT, bb, cc, v);
        }
        return;
    }
    if (wave > 0) return;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        double t = acc[0][0][v];
#pragma unroll
        for (int g = 1; g < NW; ++g) t += part[(g - 1) * kW + (4 * v + q4) * kT + l16];
        const long bb = b0 + 4 * v + q4;
        if (bb < a.nb && j0 + l16 < a.cols) blk_store(a, OUT, bb, j0 + l16, t);
    }
}

// Many tiles: 64 x 64 tiles, four waves of 2 x 2 matrix-core tiles, K in slices
// of 16 (first the states, then the window) staged in LDS and double buffered.
constexpr int kPT = 64, kPK = 16;
struct BlkStage {
    double A[2][kPT][kPK + 1];
    double B[2][kPK][kPT + 8];
};
template <int KS>
struct BlkTileLds {
    BlkStage stage[KS];
    int bad;
};

template <typename TU, bool OUT, int KS>
__device__ __forceinline__ void d_blk_tile(const VBlock vb, const BlkPass& a, BlkTileLds<KS>& Ls)
{
    const int grp = KS > 1 ? (int)threadIdx.x >> 8 : 0;
    BlkStage& L = Ls.stage[grp];
    const int tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, q4 = lane >> 4;
    const int wr = wave >> 1, wc = wave & 1;
    const long b0 = vb.y * kPT;
    const int j0 = (int)vb.x * kPT;
    const int ar = tid >> 2, ak = (tid & 3) * 4;     // A slice: row, first of four k
    const int bk = tid >> 4, bj = (tid & 15) * 4;    // B slice: k, first of four columns
    // rows past nb repeat the last one (their products are not stored)
    const long ab = b0 + ar < a.nb ? b0 + ar : a.nb - 1;
    const TU* u = static_cast<const TU*>(a.U) + ab * a.blockU;
    const int kz = OUT ? a.kz : 0, zs = (kz + kPK - 1) / kPK;
    int kl = win_len(a, ab), kEnd = a.ku, kMin = a.ku, stride = a.na;
    // the thread's four columns (those past the last repeat it): their factors
    // in BU at hb[q] + k stride, zero from k = kcol[q] on
    int kcol[4];
    long hb[4];
    const bool cols4 = j0 + bj + 4 <= a.cols;
    const int c0 = cols4 ? j0 + bj : a.cols - 1;
    bool run4 = cols4;                               // one run of four factors
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int col = j0 + bj + q < a.cols ? j0 + bj + q : a.cols - 1;
        kcol[q] = a.ku;
        hb[q] = col + (long)bk * stride;
        if (OUT) {
            const int i = col / a.p;
            kcol[q] = (a.s * i + a.taps) * a.m;
            hb[q] = ((long)a.s * (a.T - 1 - i) * a.m + bk) * a.p + (col - i * a.p);
        }
        run4 = run4 && hb[q] == hb[0] + q && kcol[q] == kcol[0];
    }
    if (OUT) {
        const int jl = j0 + kPT - 1 < a.cols ? j0 + kPT - 1 : a.cols - 1;
        kEnd = (a.s * (jl / a.p) + a.taps) * a.m;
        kMin = (a.s * (j0 / a.p) + a.taps) * a.m;
        if (first_output(a, b0, j0)) kMin = 0;
        stride = a.p;
        kl = kl < kEnd ? kl : kEnd;   // (the last slice may reach past the tile's samples)
        if (threadIdx.x == 0) Ls.bad = 0;
    }
    const int slices = zs + (kEnd + kPK - 1) / kPK;
    // window rows lie in a row of samples when four values never cross one
    // (one 16-byte load for four floats, two for four doubles: abm n = 64 from float
    // samples, 2^20 points, 876 us a solve with four loads, 806 with one)
    const bool wide4 = a.gm == 0 || (a.m & 3) == 0;
    const double* z = OUT ? a.Z + ab * a.na + ak : nullptr;
    const double* ot = OUT ? a.OT + (long)bk * a.cols : nullptr;
    bool nf = false;
    double ra[4], rb[4];
    auto load = [&](int sl) {
        if (OUT && sl < zs) {
            const int k0 = sl * kPK;
            const double* o = ot + (long)k0 * a.cols;
            if (k0 + kPK <= kz) {
                load4(z + k0, ra);
                if (cols4) {
                    load4(o + c0, rb);
                } else {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        rb[q] = o[j0 + bj + q < a.cols ? j0 + bj + q : a.cols - 1];
                }
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    ra[q] = k0 + ak + q < kz ? z[k0 + q] : 0.0;
                    rb[q] = k0 + bk < kz ? o[j0 + bj + q < a.cols ? j0 + bj + q : a.cols - 1] : 0.0;
                }
            }
            return;
        }
        const int k0 = (sl - zs) * kPK, k = k0 + ak;
        if (wide4 && k + 4 <= kl) {
            load4(u + win(a, k), ra);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) ra[q] = k + q < kl ? (double)u[win(a, k + q)] : 0.0;
        }
        const double* h = a.BU + (long)k0 * stride;
        if (k0 + kPK <= kMin || (!OUT && k0 + kPK <= kEnd)) {   // every factor is there
            if (run4) {
                load4(h + hb[0], rb);
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) rb[q] = h[hb[q]];
            }
            return;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (OUT) nf = nf || not_finite(ra[q]);
            rb[q] = k0 + bk < kcol[q] ? h[hb[q]] : 0.0;
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            L.A[buf][ar][ak + q] = ra[q];
            L.B[buf][bk][bj + q] = rb[q];
        }
    };
    doublex4 acc[2][2];
#pragma unroll
    for (int ti = 0; ti < 2; ++ti)
#pragma unroll
        for (int tj = 0; tj < 2; ++tj) acc[ti][tj] = doublex4{0.0, 0.0, 0.0, 0.0};
    // group g takes the slices g, g + KS, ...
    const int rounds = (slices + KS - 1) / KS;
    if (grp < slices) {
        load(grp);
        store(0);
    }
    __syncthreads();
    int buf = 0;
    for (int t0 = 0; t0 < rounds; ++t0) {
        const int sl = t0 * KS + grp;
        const bool more = sl + KS < slices;
        if (more) load(sl + KS);
        if (sl < slices) {
#pragma unroll
            for (int ks = 0; ks < kPK; ks += 4) {
                double x[2], y[2];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    x[t] = L.A[buf][wr * 32 + t * 16 + l16][ks + q4];
                    y[t] = L.B[buf][ks + q4][wc * 32 + t * 16 + l16];
                }
#pragma unroll
                for (int ti = 0; ti < 2; ++ti)
#pragma unroll
                    for (int tj = 0; tj < 2; ++tj)
                        acc[ti][tj] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[ti], y[tj],
                                                                          acc[ti][tj], 0, 0, 0);
            }
        }
        if (more) store(buf ^ 1);
        __syncthreads();
        buf ^= 1;
    }
    if (OUT) {
        if (nf) Ls.bad = 1;
        __syncthreads();
        if (Ls.bad) {
            for (int t = threadIdx.x; t < kPT * kPT; t += 256 * KS) {
                const long bb = b0 + t / kPT;
                const int cc = j0 + t % kPT;
                if (bb < a.nb && cc < a.cols)
                    blk_store(a, true, bb, cc, blk_output<TU>(a, bb, cc));
            }
            return;
        }
    }
    if (KS > 1) {   // the groups' partial tiles, added in group order
        if (grp > 0) {
            double* part = &L.A[0][0][0];            // 16 values a thread
#pragma unroll
            for (int ti = 0; ti < 2; ++ti)
#pragma unroll
                for (int tj = 0; tj < 2; ++tj)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        part[((ti * 2 + tj) * 4 + v) * 256 + tid] = acc[ti][tj][v];
        }
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int g = 1; g < KS; ++g) {
            const double* pg = &Ls.stage[g].A[0][0][0];
#pragma unroll
            for (int ti = 0; ti < 2; ++ti)
#pragma unroll
                for (int tj = 0; tj < 2; ++tj)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        acc[ti][tj][v] += pg[((ti * 2 + tj) * 4 + v) * 256 + tid];
        }
    }
#pragma unroll
    for (int tj = 0; tj < 2; ++tj) {
        const int col = j0 + wc * 32 + tj * 16 + l16;
        if (col >= a.cols) continue;
#pragma unroll
        for (int ti = 0; ti < 2; ++ti)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const long bb = b0 + wr * 32 + ti * 16 + 4 * v + q4;
                if (bb < a.nb) blk_store(a, OUT, bb, col, acc[ti][tj][v]);
            }
    }
}

// P_{l+1} = P_l^2 for l = lb .. L-2 of a small system, beside pass 1's tiles.
template <int NW>
__device__ __forceinline__ void d_blk_powers(int na, int lb, int L, double* PT, double* P)
{
    const int n16 = (na + 15) & ~15, nt = n16 / 16, tid = threadIdx.x, wave = tid >> 6;
    const int l16 = tid & 15, q4 = (tid >> 4) & 3;
    const long nn = (long)na * na;
    for (int t = tid; t < n16 * n16; t += NW * 64) {
        const int r = t / n16, c = t - r * n16;
        P[r * kBP + c] = (r < na && c < na) ? PT[lb * nn + (long)r * na + c] : 0.0;
    }
    __syncthreads();
    constexpr int U = 16 / NW < 1 ? 1 : 16 / NW;
    for (int l = lb; l + 1 < L; ++l) {
        doublex4 acc[U];
#pragma unroll
        for (int q = 0; q < U; ++q) {
            const int w = wave + NW * q;
            if (w < nt * nt)
                acc[q] = lds_tile<false>(P, kBP, P, kBP, w / nt * 16, w % nt * 16, n16);
        }
        __syncthreads();
        double* out = PT + (l + 1) * nn;
#pragma unroll
        for (int q = 0; q < U; ++q) {
            const int w = wave + NW * q;
            if (w >= nt * nt) continue;
            for (int v = 0; v < 4; ++v) {
                const int r = w / nt * 16 + 4 * v + q4, c = w % nt * 16 + l16;
                P[r * kBP + c] = acc[q][v];
                if (r < na && c < na) out[(long)r * na + c] = acc[q][v];
            }
        }
        __syncthreads();
    }
}

// The work-group's tile: consecutive work-groups go to different XCDs, each
// with its own L2, so the tiles of one row block (which read the same samples)
// are given to one XCD.  Row blocks past the last full eight keep plain order.
__device__ __forceinline__ VBlock blk_place(long idx, long gx, long gy)
{
    const long full = gy / 8 * 8 * gx;
    if (idx >= full) return VBlock{idx % gx, idx / gx, gx};
    const long t = idx / 8;
    return VBlock{t % gx, t / gx * 8 + idx % 8, gx};
}

template <typename TU, bool OUT, int NW, int R>
__global__ __launch_bounds__(NW * 64) void k_blk_split(const BlkPass a)
{
    constexpr int kPart = R > 1 ? NW * 256 * R * R : (NW - 1) * 256;
    constexpr int kLds = OUT || kPart > kBN * kBP ? kPart : kBN * kBP;
    __shared__ double lds[kLds];
    __shared__ int bad;
    if (!OUT && (long)blockIdx.x == a.gx * a.gy) {
        d_blk_powers<NW>(a.na, a.lb, a.L, a.PT, lds);
        return;
    }
    d_blk_split<TU, OUT, NW, R>(blk_place(blockIdx.x, a.gx, a.gy), a, lds, &bad);
}

template <typename TU, bool OUT, int KS>
__global__ __launch_bounds__(256 * KS, 4) void k_blk_tile(const BlkPass a)
{
    __shared__ BlkTileLds<KS> L;
    static_assert(sizeof(BlkStage) >= kBN * kBP * sizeof(double), "room for the powers");
    if (!OUT && (long)blockIdx.x == a.gx * a.gy) {
        d_blk_powers<4 * KS>(a.na, a.lb, a.L, a.PT, &L.stage[0].A[0][0][0]);
        return;
    }
    d_blk_tile<TU, OUT, KS>(blk_place(blockIdx.x, a.gx, a.gy), a, L);
}

// ------------------------------------------------------------------ the scan
// Start states of Nb blocks: E_0 = Z_0, E_{b+1} = P E_b + S_b with P = P_l0.
// The blocks are taken as up to 16 R groups of Lg consecutive ones, one group a
// row of the matrix-core tiles; a wave holds 16 columns of P in registers.
//   kScanAll  (one work-group): every group from zero; then the groups' start
//             states by doubling, y_g += P_{l0 + lg + k} y_{g - 2^k}; then every
//             group from its start state, writing E (in place of S)
//   kScanUp   the groups' responses from zero to Zg (work-groups of 16 groups)
//   kScanDown the groups from their start states in Zg, writing E
// E[Nb] is the state after the last block.  Bound by the chain of 2 Lg + log2
// steps, each a 16 x n_a x n_a product and an exchange through LDS.
enum { kScanAll, kScanUp, kScanDown };
struct BlkScan {
    int na, l0, lg, L;
    long nb;
    const double* PT;
    double *E, *Zg;
    // the seed in X and its shift to Z (kScanAll)
    const double *seed, *DL;
    const void* U;
    bool uDouble;
    int km, m, gm;          // taps m; samples skipped after each window row
    unsigned magic;
    long last;
    int R;                  // row tiles of a work-group
    long gx;
};

// Z_0 = X_0 - sum_r D_r u_r
__device__ __forceinline__ double blk_shift(const BlkScan& a, long row0, long at, int i)
{
    double v = 0.0;
    const double* Ud = static_cast<const double*>(a.U);
    const float* Uf = static_cast<const float*>(a.U);
#pragma unroll 1
    for (int k = 0; k < a.km; ++k) {
        const int r = a.m == 1 ? k : (int)__umulhi((unsigned)k, a.magic);
        if (row0 + r > a.last) break;
        const long o = at + k + (long)r * a.gm;
        v = fma(a.DL[(long)k * a.na + i], a.uDouble ? Ud[o] : (double)Uf[o], v);
    }
    return v;
}

// Loads are unconditional (clamped, and selected where their value is used): a
// branch around one makes every wait a wait for all of them, and then each step
// takes a memory latency (2 us at n_a = 48, of which its products are 0.3).
template <int MODE, int NK>   // NK = (n_a + 15) / 16 * 4 steps of the products
__device__ __forceinline__ void d_blk_scan_n(const VBlock vb, const BlkScan& a, double* lds)
{
    constexpr int nct = NK / 4, pitch = 4 * NK + 1;
    const int na = a.na;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, q4 = lane >> 4;
    const int rt = wave / nct, ct = wave - rt * nct, rows = 16 * a.R;
    if (rt >= a.R) return;   // (a grouped launch has waves for its widest system)
    const long Lg = 1L << a.lg, g0 = vb.x * rows;
    double* x0 = lds;                       // [rows][pitch], double buffered
    double* x1 = lds + rows * pitch;
    const long nn = (long)na * na;
    const int col = ct * 16 + l16, ccol = col < na ? col : na - 1;
    double p[NK];
    auto fetch_p = [&](int l, double* to) {
        const double* P = a.PT + l * nn + ccol;
#pragma unroll
        for (int u = 0; u < NK; ++u) {
            const int k = 4 * u + q4;
            to[u] = P[(long)(k < na ? k : na - 1) * na];
        }
    };
    auto use_p = [&](const double* from) {
#pragma unroll
        for (int u = 0; u < NK; ++u) p[u] = 4 * u + q4 < na && col < na ? from[u] : 0.0;
        // (arrived before any loop that reads them: else its every step waits for all loads)
#pragma unroll
        for (int u = 0; u < NK; ++u) asm volatile("" : "+v"(p[u]));
    };
    // rows of x (this wave's row tile shifted up by d rows, zero above) times P:
    // CH operands are read before the first of their products (one LDS round
    // trip, not one for each)
    auto product = [&](const double* x, doublex4 acc, int d) {
        constexpr int CH = MODE == kScanAll && NK > 8 ? 8 : NK;   // (16 waves: 128 registers each)
        const int r = rt * 16 + l16 - d;
        const double* xr = x + (r > 0 ? r : 0) * pitch + q4;
#pragma unroll
        for (int u0 = 0; u0 < NK; u0 += CH) {
            double v[CH];
#pragma unroll
            for (int u = 0; u < CH; ++u) v[u] = u0 + u < NK ? xr[4 * (u0 + u)] : 0.0;
#pragma unroll
            for (int u = 0; u < CH; ++u)
                if (u0 + u < NK)
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(r >= 0 ? v[u] : 0.0, p[u0 + u], acc,
                                                               0, 0, 0);
        }
        return acc;
    };
    // this lane's groups are rows rt 16 + 4 v + q4; its element of block j of
    // group v is at at(v, j), the last block's at lim
    const long g1 = g0 + rt * 16 + q4, first = (g1 << a.lg) * na + ccol;
    const long lim = (a.nb - 1) * na + ccol;
    auto at = [&](int v, long j) { return first + (((long)(4 * v) << a.lg) + j) * na; };
    auto fetch = [&](doublex4& to, long j) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const long o = at(v, j);
            to[v] = a.E[o < lim ? o : lim];
        }
    };
    auto select = [&](doublex4 y, long j) {
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (col >= na || at(v, j) > lim) y[v] = 0.0;
        return y;
    };
    auto put = [&](double* x, int v, double y) { x[(rt * 16 + 4 * v + q4) * pitch + col] = y; };
    double* cur = x0;
    double* nxt = x1;
    auto flip = [&]() {
        __syncthreads();
        double* t = cur;
        cur = nxt;
        nxt = t;
    };
    // the elements of D steps are on their way (D divides L_g: groups over several
    // work-groups have 16 blocks or more)
    constexpr int D = MODE == kScanAll ? 1 : 2;
    doublex4 s[D];
#pragma unroll
    for (int q = 0; q < D; ++q) fetch(s[q], q);
    fetch_p(a.l0, p);
    use_p(p);
    if (MODE != kScanDown) {
        // from zero
#pragma unroll
        for (int v = 0; v < 4; ++v) put(cur, v, 0.0);
        __syncthreads();
#pragma unroll 1
        for (long j0 = 0; j0 < Lg; j0 += D) {
#pragma unroll
            for (int q = 0; q < D; ++q) {
                const doublex4 e = select(s[q], j0 + q);
                fetch(s[q], j0 + q + D);
                const doublex4 y = product(cur, e, 0);
#pragma unroll
                for (int v = 0; v < 4; ++v) put(nxt, v, y[v]);
                flip();
            }
        }
        if (MODE == kScanUp) {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (col < na && at(v, 0) <= lim)
                    a.Zg[(g1 + 4 * v) * na + col] = cur[(rt * 16 + 4 * v + q4) * pitch + col];
            return;
        }
#pragma unroll
        for (int q = 0; q < D; ++q) fetch(s[q], q);
        // the groups' start states: row g holds the response of group g - 1,
        // row 0 the seed
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int g = rt * 16 + 4 * v + q4;
            double y = 0.0;
            if (g > 0) y = cur[(g - 1) * pitch + col];
            if (g == 0 && col < na) y = a.seed[col] - blk_shift(a, 0, 0, col);
            put(nxt, v, y);
        }
        flip();
        const long groups = (a.nb + Lg - 1) / Lg;
        // the next step's power is on its way (16 waves at NK = 16 have no room for it)
        constexpr bool kAhead = NK < 16;
        double pn[kAhead ? NK : 1];
        if (kAhead && groups > 1) fetch_p(a.l0 + a.lg, pn);
#pragma unroll 1
        for (int k = 0; (1L << k) < groups; ++k) {
            if (kAhead) {
                use_p(pn);
                fetch_p((2L << k) < groups ? a.l0 + a.lg + k + 1 : a.l0, pn);
            } else {
                fetch_p(a.l0 + a.lg + k, p);
                use_p(p);
            }
            doublex4 y;
#pragma unroll
            for (int v = 0; v < 4; ++v) y[v] = cur[(rt * 16 + 4 * v + q4) * pitch + col];
            // (the first 2^k groups have their start states: a power that has
            // overflowed would add infinity times their zero neighbours)
            const doublex4 z = product(cur, y, 1 << k);
#pragma unroll
            for (int v = 0; v < 4; ++v) put(nxt, v, rt * 16 + 4 * v + q4 < (1 << k) ? y[v] : z[v]);
            flip();
        }
        if (kAhead) {
            if (groups > 1) use_p(pn);
        } else {
            fetch_p(a.l0, p);
            use_p(p);
        }
    } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
            put(cur, v, col < na && at(v, 0) <= lim ? a.Zg[(g1 + 4 * v) * na + col] : 0.0);
        __syncthreads();
    }
    // from the start states: E_e over S_e, each read before it is written
    doublex4 x;
#pragma unroll
    for (int v = 0; v < 4; ++v) x[v] = cur[(rt * 16 + 4 * v + q4) * pitch + col];
#pragma unroll 1
    for (long j0 = 0; j0 < Lg; j0 += D) {
#pragma unroll
        for (int q = 0; q < D; ++q) {
            const long j = j0 + q;
            const doublex4 y = select(s[q], j);
            fetch(s[q], j + D);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const long o = at(v, j);
                if (col < na && o <= lim) a.E[o] = x[v];
            }
            x = product(cur, y, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (col < na && at(v, j) == lim) a.E[lim + na] = x[v];
                put(nxt, v, x[v]);
            }
            flip();
        }
    }
}

template <int MODE>
__device__ __forceinline__ void d_blk_scan(const VBlock vb, const BlkScan& a, double* lds)
{
    switch ((a.na + 15) / 16) {
    case 1: return d_blk_scan_n<MODE, 4>(vb, a, lds);
    case 2: return d_blk_scan_n<MODE, 8>(vb, a, lds);
    case 3: return d_blk_scan_n<MODE, 12>(vb, a, lds);
    default: return d_blk_scan_n<MODE, 16>(vb, a, lds);
    }
}

template <int MODE, int NK>
__global__ __launch_bounds__(MODE != kScanAll ? 16 * NK : NK == 12 ? 768 : 1024) void k_blk_scan(const BlkScan a)
{
    extern __shared__ double scan_lds[];
    d_blk_scan_n<MODE, NK>(VBlock{(long)blockIdx.x, (long)blockIdx.y, (long)gridDim.x}, a, scan_lds);
}

__global__ void k_blk_carry(const BlkScan a, long row0, long at, double* out)
{
    for (int i = threadIdx.x; i < a.na; i += blockDim.x)
        out[i] = a.E[a.nb * a.na + i] + blk_shift(a, row0, at, i);
}

// wide maps: the first state at the tree's top is the seed, shifted.  16 states to
// a work-group, a state's taps m terms over 16 lanes (one after the other in one
// work-group: 37 us at 812 states, 100 terms).
__device__ __forceinline__ void d_blk_root(const VBlock vb, const BlkScan& a, double* E)
{
    __shared__ double part[16][17];
    const int c = threadIdx.x & 15, g = threadIdx.x >> 4, i = (int)vb.x * 16 + c;
    double v = 0.0;
    if (i < a.na) {
        const double* Ud = static_cast<const double*>(a.U);
        const float* Uf = static_cast<const float*>(a.U);
        for (int k = g; k < a.km; k += 16) {
            const int r = a.m == 1 ? k : (int)__umulhi((unsigned)k, a.magic);
            if (r > a.last) break;
            const long o = k + (long)r * a.gm;
            v = fma(a.DL[(long)k * a.na + i], a.uDouble ? Ud[o] : (double)Uf[o], v);
        }
    }
    part[g][c] = v;
    __syncthreads();
    if (g || i >= a.na) return;
#pragma unroll
    for (int q = 1; q < 16; ++q) v += part[q][c];
    E[i] = a.seed[i] - v;
}
__global__ __launch_bounds__(256) void k_blk_root(const BlkScan a, double* E)
{
    d_blk_root(VBlock{(long)blockIdx.x, 0, (long)gridDim.x}, a, E);
}
// The state after all blocks (every node is whole): z P + S from the last node of
// the tree's top, shifted back.
__global__ __launch_bounds__(256) void k_blk_carry_wide(const BlkScan a, const double* P,
                                                        const double* e, const double* S,
                                                        long row0, long at, double* out)
{
    extern __shared__ double z[];
    for (int i = threadIdx.x; i < a.na; i += 256) z[i] = e[i];
    __syncthreads();
    const int i = (int)blockIdx.x * 256 + threadIdx.x;
    if (i >= a.na) return;
    double v = S[i] + blk_shift(a, row0, at, i);
    for (int k = 0; k < a.na; ++k) v = fma(P[(long)k * a.na + i], z[k], v);
    out[i] = v;
}

// ---------------------------------------------------------------- wide maps
// The element-wise stages between the products: FP64 copies and the transposed
// outputs (prep), the step's combinations (comb; RungeKutta4thOrder.cpp:48-57,
// AdamsMoulton.cpp:258-316), the ABM block input and shift (asm).
template <typename TI>
__device__ __forceinline__ void blk_comb(const BlkElem& a, long x)
{
#pragma clang fp contract(off)
    const BlockShape& s = a.s;
    const int n = s.n, m = s.m, na = s.na;
    // with the reference's rounding the products are floats, and A, B the inputs
    const TI* A = s.mirror ? reinterpret_cast<const TI*>(a.A) : reinterpret_cast<const TI*>(a.A64);
    const TI* B = s.mirror ? reinterpret_cast<const TI*>(a.B) : reinterpret_cast<const TI*>(a.B64);
    const TI *A2 = reinterpret_cast<const TI*>(a.A2), *A3 = reinterpret_cast<const TI*>(a.A3),
             *A4 = reinterpret_cast<const TI*>(a.A4), *AB = reinterpret_cast<const TI*>(a.AB),
             *A2B = reinterpret_cast<const TI*>(a.A2B), *A3B = reinterpret_cast<const TI*>(a.A3B);
    auto rnd = [&](double v) { return s.mirror ? (double)(float)v : v; };
    const long np = (long)na * na;
    if (s.method == 0) {
        const Rk4Coef& k = a.rk;
        if (x < np) {
            const int j = (int)(x / n), i = (int)(x - (long)j * n);
            const long t = (long)i * n + j;
            double v = ((i == j) ? 1.0 : 0.0) + k.h * (double)A[t];
            v = v + k.c2 * (double)A2[t];
            v = v + k.c3 * (double)A3[t];
            v = v + k.c4 * (double)A4[t];
            a.PT[x] = rnd(v);
            return;
        }
        x -= np;
        const int j = (int)(x / n), i = (int)(x - (long)j * n);
        const long t = (long)i * m + j;
        const double b = B[t], ab = AB[t], a2b = A2B[t], a3b = A3B[t];
        a.B1[x] = rnd((1.0 / 6.0) * (((k.h * b + k.s1 * ab) + k.s2 * a2b) + k.s3 * a3b));
        a.QT[((long)s.s * (s.T - 1) * m + m + j) * n + i] =
            rnd((1.0 / 6.0) * ((k.t0 * b + k.t1 * ab) + k.t2 * a2b));
        a.DL[x] = rnd(k.u0 * b);
        return;
    }
    const AbmCoef& c = a.ab;
    if (x < np) {
        const int j = (int)(x / na), i = (int)(x - (long)j * na);   // PT[j][i] = M[i][j]
        double v;
        if (i < 3 * n) {
            v = j == i + n ? 1.0 : 0.0;
        } else {
            const int r = i - 3 * n, b = j / n, q = j - b * n;
            const double y = A[(long)r * n + q], y2 = A2[(long)r * n + q], id = r == q ? 1.0 : 0.0;
            v = b == 0 ? rnd(c.a3A2 * y2) : b == 1 ? rnd(c.a2A * y + c.a2A2 * y2)
              : b == 2 ? rnd(c.a1A * y + c.a1A2 * y2) : rnd((id + c.a0A * y) + c.a0A2 * y2);
        }
        a.PT[x] = v;
        return;
    }
    x -= np;
    const int j = (int)(x / n), i = (int)(x - (long)j * n);
    const long t = (long)i * m + j, mn = (long)m * n;
    const double b = B[t], ab = AB[t];
    a.B1[x] = rnd(c.b3AB * ab);
    a.B1[mn + x] = rnd(c.b2B * b + c.b2AB * ab);
    a.B1[2 * mn + x] = rnd(c.b1B * b + c.b1AB * ab);
    a.B1[3 * mn + x] = rnd(c.b0B * b + c.b0AB * ab);
    a.VT[(long)j * 5 * n + i] = rnd(c.bm1 * b);
}

__device__ __forceinline__ void d_blk_elem(const VBlock vb, const BlkElem& a)
{
    const BlockShape& s = a.s;
    const int n = s.n, m = s.m, p = s.p, na = s.na;
    for (long x = vb.x * 256 + threadIdx.x; x < a.count; x += vb.gx * 256) {
        if (a.stage == BlkElem::kComb) {
            if (s.mirror)
                blk_comb<float>(a, x);
            else
                blk_comb<double>(a, x);
        } else if (a.stage == BlkElem::kPrep) {
            long t = x;
            if (t < (long)n * n) {
                a.A64[t] = (double)a.A[t];
                continue;
            }
            t -= (long)n * n;
            if (t < (long)n * m) {
                a.B64[t] = (double)a.B[t];
                continue;
            }
            t -= (long)n * m;
            if (t < (long)m * p) {
                a.DT[t] = s.useD ? (double)a.D[(t % p) * m + t / p] : 0.0;
                continue;
            }
            t -= (long)m * p;
            if (t < (long)na * p) {     // O of step 0, and C^T
                const int k = (int)(t / p), o = (int)(t - (long)k * p), i = k - (na - n);
                double v = 0.0;
                if (i >= 0) {
                    v = s.useC ? (double)a.C[(long)o * n + i] : (i == o ? 1.0 : 0.0);
                    a.CT[(long)i * p + o] = v;
                }
                a.OT[(long)k * s.T * p + o] = v;
                continue;
            }
            t -= (long)na * p;
            a.seed[t] = (double)a.x0[t];
        } else {
            long t = x;
            if (t < (long)m * na) {
                const int j = (int)(t / na), i = (int)(t - (long)j * na);
                a.QT[(long)(s.T - 1) * m * na + t] = a.VT[(long)j * 5 * n + n + i];
                continue;
            }
            t -= (long)m * na;
            const int rj = (int)(t / na), y = (int)(t - (long)rj * na);
            const int r = rj / m, j = rj - r * m, b = y / n, i = y - b * n;
            a.DL[t] = b >= r ? a.VT[(long)j * 5 * n + (b - r) * n + i] : 0.0;
        }
    }
}

__global__ __launch_bounds__(256) void k_blk_elem(const BlkElem a)
{
    d_blk_elem(VBlock{(long)blockIdx.x, (long)blockIdx.y, (long)gridDim.x}, a);
}

// ================================================================ host side
static unsigned magic_of(int m) { return (unsigned)(((1ULL << 32) + m - 1) / m); }

// One work-group's LDS holds the map.
static bool fits_one(int method, int n, int m, int p)
{
    const int na = method == 1 ? 4 * n : n, s = method == 1 ? 1 : 2;
    return na <= kBN && p <= kBN && m <= kBM && s * m <= kBN;
}

// One work-group scans up to 512 blocks; more go in groups of 16 (or as many
// as leave 512 groups).
static int group_log(long nb)
{
    if (nb <= 512) return 0;
    int lg = 4;
    while (((nb + (1L << lg) - 1) >> lg) > 512) ++lg;
    return lg;
}
// Row tiles of the scan's one work-group: 128, 64, 64 and 32 rows at up to 16, 32, 48
// and 64 states, on 8 waves (12 at 48).  16 waves halve the dependent steps, but all
// products share one compute unit and each step then takes more than two did (us a
// solve with 8 and 16: n = 8, 4096 points 34.0, 38.3; n = 24, 9000 points 52.2, 57.5;
// n = 64, 4000 points 98.3, 114.3).
static int scan_row_tiles(int na) { return na <= 16 ? 8 : na <= 48 ? 4 : 2; }
// The rule: which systems run as block responses, and with how many steps per
// block: the fastest by the model below.  Covered: inputs and outputs present,
// horizons from 64 points, n up to 1024.  The general path was nowhere faster on
// either side's edges (us, general against blocks: RK4 n = 65, 64 points 172, 65;
// n = 1000, 100 points 789, 571; n = 100, 100 inputs and outputs, 5000 points 246,
// 241; ABM n = 256, 80 points 695, 370; n = 600, 100 points 10531, 10638, the
// start-up's; n = 17, 2^20 points 660, 261).  More steps per block make the scan
// shorter (2 n_a^2 products a block, and its chain of dependent steps), fewer make
// pass 2 (s m p T / 2 products a step) and the tables (2 n_a^2 (s m + p) T)
// cheaper.
int block_steps_log(int method, int n, int m, int p, bool useC, bool useD, long nScan, long nPad)
{
    const int na = method == 1 ? 4 * n : n, s = method == 1 ? 1 : 2;
    if (m < 1 || p < 1 || (!useC && useD) || nScan < 64) return 0;
    if (!useC) p = n;
    const bool one = fits_one(method, n, m, p);
    if (n > 1024 || (long)m * p > (1L << 20)) return 0;
    int best = 0;
    double bt = 0.0;
    const double N = (double)nScan, na2 = (double)na * na;
    for (int lb = 3; lb <= 8; ++lb) {
        const double T = 1 << lb, nb = N / T;
        if ((nPad >> lb) < 2) break;
        // (T m s < 2^16: the window index's multiply-high)
        if ((long)(s * T + 8) * m >= 65536) break;
        // microseconds: FP64 products at 40 TFLOP/s (25 over few tiles; pass 2 in
        // tiles of 16 or 32: 6), the scan's chain, the tables
        const double r1 = one ? 25e6 : 40e6, r2 = one && N * p < 64 * 4096 ? 6e6 : r1;
        const double pass1 = N * 2.0 * na * s * m / r1;
        const double pass = pass1 + N * (2.0 * p * na + 2.0 * s * m * p * (T / 2 + 32.0 / p + 2)) / r2;
        double scan, tab;
        if (one) {
            // k_blk_scan measured: 13 us + 2.4 for each 256 states at n_a = 8, 18 +
            // 3.1 for each 64 at 48; groups before it 5 + 0.95 a step and 6 + 1.6
            // (both ways).  (A fit: two of the launch's steps up to 32 states, one up
            // to 48; at 49 to 64 it is 2.4 us short for each 64 states.  The launch's
            // own steps and rows in its place: 160 of 702 shapes take another T, from
            // 9% faster to 14% slower, 0.3% faster on average.)
            const int lg = group_log((long)std::ceil(nb));
            const double rows = na <= 16 ? 256 : na <= 32 ? 128 : 64;
            const double Lg = std::exp2(std::max(0.0, std::ceil(std::log2(nb / (1 << lg) / rows))));
            scan = 12 + 0.13 * na + (2.3 + 0.017 * na) * Lg + (lg ? 6 + (0.85 + 0.016 * na) * (1 << lg) : 0);
            tab = lb * 1.2 + T * (s * m + p) / 64 * 0.05;
        } else {
            scan = 4 * na2 * nb / 40e6 + 2 * 5.0 * std::max(1.0, std::log2(nb));
            tab = 2 * na2 * (s * m + p) * T / 40e6 + 5.0 * lb;
        }
        // (what the squarings beside pass 1 take beyond it)
        const double sq = one ? std::max(0.0, std::log2(nb) * (0.8 + 0.018 * na) - 8 - pass1) : 0.0;
        const double t = pass + scan + tab + sq;
        if (!best || t < bt) {
            best = lb;
            bt = t;
        }
    }
    return best;
}

BlockShape block_shape(int method, int n, int m, int p, bool useC, bool useD, bool mirror, int lb,
                       int L)
{
    BlockShape s;
    s.method = method;
    s.n = n;
    s.m = m;
    s.p = useC ? p : n;
    s.na = method == 1 ? 4 * n : n;
    s.useC = useC;
    s.useD = useD;
    s.mirror = mirror;
    s.lb = lb;
    s.T = 1 << lb;
    s.L = L;
    s.s = method == 1 ? 1 : 2;
    s.taps = method == 1 ? 4 : 1;
    s.wide = !fits_one(method, n, m, s.p);
    return s;
}

size_t block_table_values(const BlockShape& s)
{
    return ((size_t)s.kb() + (size_t)s.T * s.p + (size_t)s.taps * s.m) * s.na +
           (size_t)s.kh() * s.p;
}

// The tree over a wide map's blocks.  Up, level k + 1 holds the responses of
// pairs of level k: a launch a level, beside which the next power's squaring
// runs.  Down, a step takes the start states from level k to the two levels
// below it at once (n_a <= 256: half the launches, whose products are shorter
// than a launch; a step's third power costs n_a^3 and its second products
// n_a^2, too much for wider maps) or to the one below.  A level's states are
// padded to whole nodes of four.
struct TreeLevel {
    long n;        // states of the level
    size_t s, e;   // responses and start states, in states from b.Z2 (level 0: b.Z, b.E)
};
static long tree_rows(long n) { return (n + 3) / 4 * 4; }
static bool structured_square(const BlockShape& s);
// The tree ends at few states, which are taken one after the other: a product of
// one row each in place of the levels above, and no squarings for those (which
// the up levels wait for): 8 states where a squaring is four dependent launches
// (ABM n = 203: 988 us a solve against 1075 with the whole tree, 1000 with 16), 4
// otherwise (n = 128: 399 against 401, 409 with 8; 512 systems together 44.7 ms
// against 46.5).
static long tree_top(const BlockShape& s) { return structured_square(s) ? 8 : 4; }
static std::vector<TreeLevel> tree_of(const BlockShape& s, long nb)
{
    std::vector<TreeLevel> t;
    size_t at = 0;
    for (long n = nb;; n = (n + 1) / 2) {
        const size_t rows = t.empty() ? 0 : (size_t)tree_rows(n);
        t.push_back(TreeLevel{n, at, at + rows});
        at += 2 * rows;
        if (n <= tree_top(s)) return t;
    }
}
// states from b.Z2 on that all levels take together (tree_of's last place: whole
// nodes at the top too, up to eight states)
static size_t tree_states(const std::vector<TreeLevel>& t)
{
    return t.size() == 1 ? 0 : t.back().e + (size_t)tree_rows(t.back().n);
}
static double* tree_s(const BlockShape& s, const BlockBufs& b, const std::vector<TreeLevel>& t, int k)
{
    return k == 0 ? b.Z : b.Z2 + t[k].s * s.na;
}
static double* tree_e(const BlockShape& s, const BlockBufs& b, const std::vector<TreeLevel>& t, int k)
{
    return k == 0 ? b.E : b.Z2 + t[k].e * s.na;
}
int block_tree_up_levels(const BlockShape& s, long nb) { return (int)tree_of(s, nb).size() - 1; }
// the levels that the down steps go to, from the top
static std::vector<int> tree_steps(const BlockShape& s, int top)
{
    std::vector<int> to;
    // pairs of levels lie at even distances from level 0 (their powers' stacks)
    for (int k = top; k > 0;) {
        k -= s.radix4() && k % 2 == 0 ? 2 : 1;
        to.push_back(k);
    }
    return to;
}
int block_tree_down_steps(const BlockShape& s, long nb)
{
    return (int)tree_steps(s, block_tree_up_levels(s, nb)).size();
}

// Z (and E): whole nodes and one state more; then Z2
static size_t state_rows0(const BlockShape& s, long nb)
{
    return s.wide ? (size_t)tree_rows(nb) : (size_t)nb + 1;
}
size_t block_state_values(const BlockShape& s, long nb)
{
    if (!s.wide) return (state_rows0(s, nb) + block_groups(nb) + 1) * s.na;
    return (2 * state_rows0(s, nb) + tree_states(tree_of(s, nb))) * s.na;
}

size_t block_scratch_values(const BlockShape& s)
{
    if (!s.wide) return 0;
    const size_t n = s.n, m = s.m, p = s.p;
    return 4 * n * n + 4 * n * m + n * p + m * p + 9 * m * n;
}

BlockBufs block_carve(const BlockShape& s, double* PT, double* tab, double* z, long nb, double* w)
{
    BlockBufs b;
    b.PT = PT;
    b.QT = tab;
    b.OT = b.QT + (size_t)s.kb() * s.na;
    b.Ht = b.OT + (size_t)s.T * s.p * s.na;
    b.DL = b.Ht + (size_t)s.kh() * s.p;
    b.Z = z;
    b.E = s.wide ? z + state_rows0(s, nb) * s.na : z;
    b.Z2 = b.E + state_rows0(s, nb) * s.na;
    b.W = w;
    return b;
}

void block_elem(hipStream_t st, const BlkElem& e)
{
    if (e.count <= 0) return;
    hipLaunchKernelGGL(k_blk_elem, dim3((unsigned)e.gx), dim3(256), 0, st, e);
    check_launch("block elem");
}

// Whether an ABM map's squarings take block column 0 by a product and the
// others by the companion's recurrence (56 n^3 flop in four dependent launches)
// rather than the whole square (128 n^3 in one): from n = 128, where the
// products' time exceeds the launches'.
static bool structured_square(const BlockShape& s) { return s.method == 1 && s.n > 128; }

int block_emit(const BlockShape& s, const BlockBufs& b, double h, const float* A, const float* B,
               const float* C, const float* D, const float* x0, double* seed, int last,
               BlockSink& sink, std::vector<int>* readyAt)
{
    const int n = s.n, m = s.m, p = s.p, na = s.na, sm = s.s * m, T = s.T;
    const size_t nn = (size_t)n * n, nm = (size_t)n * m;
    const size_t na2 = (size_t)na * na;
    BlkElem e{};
    e.s = s;
    e.h = h;
    e.rk = rk4_coefficients(h);
    e.ab = abm_coefficients(h);
    e.A = A;
    e.B = B;
    e.C = C;
    e.D = D;
    e.x0 = x0;
    e.PT = b.PT;
    e.QT = b.QT;
    e.OT = b.OT;
    e.DL = b.DL;
    e.seed = seed;
    e.A64 = b.W;
    e.A2 = e.A64 + nn;
    e.A3 = e.A2 + nn;
    e.A4 = e.A3 + nn;
    e.B64 = e.A4 + nn;
    e.AB = e.B64 + nm;
    e.A2B = e.AB + nm;
    e.A3B = e.A2B + nm;
    e.CT = e.A3B + nm;
    e.DT = e.CT + (size_t)n * p;
    e.B1 = e.DT + (size_t)m * p;
    e.VT = e.B1 + 4 * nm;
    auto elem = [&](int phase, int stage, long count) {
        e.stage = stage;
        e.count = count;
        e.gx = std::min<long>((count + 255) / 256, 1024);
        sink.elem(phase, e);
    };
    const bool rk4 = s.method == 0;
    elem(0, BlkElem::kPrep, (long)(nn + nm) + (long)m * p + (long)na * p + (rk4 && x0 ? n : 0));
    int base;
    if (s.mirror) {
        auto f = [](double* v) { return reinterpret_cast<float*>(v); };
        sink.seq(1, SeqOp{n, n, n, A, A, f(e.A2)});
        sink.seq(1, SeqOp{n, n, m, A, B, f(e.AB)});
        if (rk4) {
            sink.seq(2, SeqOp{n, n, n, f(e.A2), A, f(e.A3)});
            sink.seq(2, SeqOp{n, n, m, f(e.A2), B, f(e.A2B)});
            sink.seq(3, SeqOp{n, n, n, A, f(e.A3), f(e.A4)});
            sink.seq(3, SeqOp{n, n, m, f(e.A3), B, f(e.A3B)});
        }
        base = rk4 ? 4 : 2;
    } else {
        auto mul = [&](int phase, int c, const double* X, const double* Y, double* Z) {
            sink.gemm(phase, GemmOp{n, n, c, X, Y, Z, gemm_ld(n, c)});
        };
        mul(1, n, e.A64, e.A64, e.A2);
        mul(1, m, e.A64, e.B64, e.AB);
        if (rk4) {
            mul(2, n, e.A2, e.A64, e.A3);
            mul(2, n, e.A2, e.A2, e.A4);
            mul(2, m, e.A2, e.B64, e.A2B);
            mul(2, m, e.A2, e.AB, e.A3B);
        }
        base = rk4 ? 3 : 2;
    }
    elem(base, BlkElem::kComb, (long)na2 + (long)nm);
    double* GT = b.QT + (size_t)sm * (T - 1) * na;
    double* F = b.Ht + (size_t)s.s * (T - 1) * m * p;
    const long cols = (long)T * p;
    int ready;                       // the phase at which G can be read
    const double* G = GT;
    int ldg = na;
    if (rk4) {
        // G's first half: B1 + M B3 (transposed); F = D + C B3
        GemmLd ld{n, n, n};
        ld.add = e.B1;
        ld.lda = n;
        sink.gemm(base + 1, GemmOp{m, n, n, b.DL, b.PT, GT, ld});
        GemmLd lf{n, p, p};
        lf.add = e.DT;
        lf.lda = p;
        sink.gemm(base + 1, GemmOp{m, n, p, b.DL, e.CT, F, lf});
        ready = base + 2;
    } else {
        // V_t^T = B_{4-t}^T + [V_0 .. V_{t-1}]^T [M_{4-t} .. M_3]^T
        for (int t = 1; t < 5; ++t) {
            GemmLd ld{5 * n, na, 5 * n};
            ld.add = e.B1 + (size_t)(4 - t) * nm;
            ld.lda = n;
            sink.gemm(base + t, GemmOp{m, t * n, n, e.VT,
                                       b.PT + (size_t)(4 - t) * n * na + 3 * n, e.VT + t * n, ld});
        }
        ready = base + 5;
        elem(ready, BlkElem::kAsm, (long)m * na + 4L * m * na);
        for (int r = 0; r < 4; ++r) {
            GemmLd lf{5 * n, p, p};
            if (r == 3) {
                lf.add = e.DT;
                lf.lda = p;
            }
            sink.gemm(ready, GemmOp{m, n, p, e.VT + (3 - r) * n, e.CT, F + (size_t)r * m * p, lf});
        }
        G = e.VT + n;                // (GT itself is copied in phase `ready`)
        ldg = 5 * n;
    }
    // powers, and the tables by doubling
    const bool st = structured_square(s);
    const int spp = st ? 4 : 1;
    int q = ready - 1;
    for (int l = 0; l <= last || l < s.lb; ++l) {
        const int ph = base + 1 + spp * l;   // P_l can be read
        if (readyAt) readyAt->push_back(ph);
        const double* P = b.PT + s.slot(l) * na2;
        if (l < last) {
            double* P2 = b.PT + s.slot(l + 1) * na2;
            if (!st) {
                sink.gemm(ph, GemmOp{na, na, na, P, P, P2, gemm_ld(na, na)});
            } else {
                sink.gemm(ph, GemmOp{na, na, n, P, P, P2, GemmLd{na, na, na}});
                for (int c = 1; c < 4; ++c) {
                    GemmLd ld{na, na, na};
                    ld.add = P2 + (c - 1) * n;
                    ld.lda = na;
                    ld.shift = n;
                    sink.gemm(ph + c, GemmOp{na, n, n, b.PT + 3 * n,
                                             P2 + 3L * n * na + (c - 1) * n, P2 + c * n, ld});
                }
            }
        }
        // the third power of a radix-4 level
        if (s.radix4() && l > s.lb && l < last && ((l - s.lb) & 1))
            sink.gemm(ph, GemmOp{na, na, na, P, b.PT + s.slot(l - 1) * na2,
                                 b.PT + (s.slot(l - 1) - 2) * na2, gemm_ld(na, na)});
        if (l >= s.lb) continue;
        const int k = 1 << l;
        sink.gemm(ph, GemmOp{na, na, k * p, P, b.OT, b.OT + (long)k * p,
                             GemmLd{na, (int)cols, (int)cols}});
        q = std::max(q + 1, ph);
        sink.gemm(q, GemmOp{k * sm, na, na, l == 0 ? G : b.QT + (size_t)(T - k) * sm * na, P,
                            b.QT + (size_t)(T - 2 * k) * sm * na,
                            GemmLd{l == 0 ? ldg : na, na, na}});
    }
    GemmLd lh{ldg, (int)cols, p};
    lh.zp = p;
    lh.zs = -(long)sm * p;
    sink.gemm(std::max(ready, base + 2 + spp * (s.lb - 1)),
              GemmOp{sm, na, (T - 1) * p, G, b.OT, b.Ht + (size_t)(T - 2) * sm * p, lh});
    return q + 1;
}

// S'[i] = S[2i] P + S[2i + 1] (a last state without a pair is no other's left
// neighbour: not formed)
GemmOp block_tree_up(const BlockShape& s, const BlockBufs& b, long nb, int k)
{
    const std::vector<TreeLevel> t = tree_of(s, nb);
    const int na = s.na;
    double* S = tree_s(s, b, t, k);
    GemmLd ld{2 * na, na, na};
    ld.add = S + na;
    ld.lda = 2 * na;
    return GemmOp{(int)(t[k].n / 2), na, na, S, b.PT + (size_t)s.slot(s.lb + k) * na * na,
                  tree_s(s, b, t, k + 1), ld};
}
// E[i + 1] = E[i] P + S[i] at the tree's top
int block_tree_top_steps(const BlockShape& s, long nb) { return (int)tree_of(s, nb).back().n - 1; }
GemmOp block_tree_top(const BlockShape& s, const BlockBufs& b, long nb, int i)
{
    const std::vector<TreeLevel> t = tree_of(s, nb);
    const int na = s.na, top = (int)t.size() - 1;
    double* E = tree_e(s, b, t, top) + (size_t)i * na;
    GemmLd ld{na, na, na};
    ld.add = tree_s(s, b, t, top) + (size_t)i * na;
    ld.lda = na;
    return GemmOp{1, na, na, E, b.PT + (size_t)s.slot(s.lb + top) * na * na, E + na, ld};
}
// E[R i] = E'[i], E[R i + j] = E'[i] P^j + sum_{q < j} S[R i + q] P^(j-1-q), R = 2 or 4
std::vector<GemmOp> block_tree_down(const BlockShape& s, const BlockBufs& b, long nb, int j0)
{
    const std::vector<TreeLevel> t = tree_of(s, nb);
    const int na = s.na, top = (int)t.size() - 1;
    const std::vector<int> to = tree_steps(s, top);
    const int from = j0 == 0 ? top : to[j0 - 1], k = to[j0], R = 1 << (from - k);
    const double* S = tree_s(s, b, t, k);
    double* E = tree_e(s, b, t, k);
    std::vector<GemmOp> ops;
    for (int j = 1; j < R; ++j) {
        GemmLd ld{na, na, R * na};
        ld.add = S + (j - 1) * na;
        ld.lda = R * na;
        if (j == 1) {
            ld.cp = E;
        } else {
            ld.X2 = S;
            ld.ldx2 = R * na;
            ld.k1 = na;
        }
        ops.push_back(GemmOp{(int)t[from].n, j * na, na, tree_e(s, b, t, from),
                             b.PT + (size_t)(s.slot(s.lb + k) - (j - 1)) * na * na, E + j * na, ld});
    }
    return ops;
}

long block_groups(long nb)
{
    const int lg = group_log(nb);
    return lg ? (nb + (1L << lg) - 1) >> lg : 0;
}

void block_start_outputs(hipStream_t st, const BlockShape& s, const float* C, const float* D,
                         const double* X0, const void* U, bool uDouble, float* Y)
{
    if (uDouble)
        hipLaunchKernelGGL(k_blk_start_outputs<double>, dim3(1), dim3(1024), 0, st, s, C, D, X0,
                           (const double*)U, Y);
    else
        hipLaunchKernelGGL(k_blk_start_outputs<float>, dim3(1), dim3(1024), 0, st, s, C, D, X0,
                           (const float*)U, Y);
    check_launch("block start outputs");
}

// steps of a slice: the largest power of two of at most `rows` rows (at least one
// step: per rows, which fit the LDS)
static int slice_steps(int T, int per, int rows)
{
    int k = 1;
    while (2 * k <= T && 2 * k * per <= rows) k *= 2;
    return k;
}

static BlkTables table_args(const BlockShape& s, const BlockBufs& b, double h, const float* A,
                            const float* B, const float* C, const float* D, const float* x0,
                            const void* U, double* seed, float* Y, bool grouped)
{
    BlkTables a{s, h, rk4_coefficients(h), abm_coefficients(h), A, B, C, D, x0, U, b.PT, b.QT,
                b.OT, b.Ht, b.DL, seed, Y, 0, 0, 0};
    // Short slices while each has its compute unit: a level's time is that of its
    // products on one (n_a = 48: 20 us for six levels with 64 rows, 15.5 with 16).
    // Together with other systems the longest, since each slice squares for itself.
    for (int rows = grouped ? kBN : 16; rows <= kBN; rows *= 2) {
        a.ni = slice_steps(s.T, s.p, rows);
        a.nq = slice_steps(s.T, s.s * s.m, rows);
        a.gx = 1 + s.T / a.ni + s.T / a.nq;
        if (a.gx <= 255) break;
    }
    if (x0) ++a.gx;
    return a;
}

void block_tables(hipStream_t st, const BlockShape& s, const BlockBufs& b, double h, const float* A,
                  const float* B, const float* C, const float* D, const float* x0, const void* U,
                  bool uDouble, double* seed, float* Y)
{
    const BlkTables a = table_args(s, b, h, A, B, C, D, x0, U, seed, Y, false);
    if (uDouble)
        hipLaunchKernelGGL(k_blk_tables<double>, dim3((unsigned)a.gx), dim3(1024), 0, st, a);
    else
        hipLaunchKernelGGL(k_blk_tables<float>, dim3((unsigned)a.gx), dim3(1024), 0, st, a);
    check_launch("block_tables");
}

static BlkPass pass_args(const BlockShape& s, const BlockBufs& b, const BlockInput& in, long nb)
{
    BlkPass a{};
    a.na = s.na;
    a.m = s.m;
    a.p = s.p;
    a.s = s.s;
    a.T = s.T;
    a.taps = s.taps;
    a.nb = nb;
    a.U = in.U;
    a.blockU = s.T * in.sL * s.m;
    a.gm = (int)(in.sL / s.s - 1) * s.m;
    a.magic = magic_of(s.m);
    a.last = in.last;
    a.PT = b.PT;
    a.lb = s.lb;
    a.L = s.L;
    return a;
}

// The tiling of a pass, alone or in a grouped launch: 64 x 64 tiles from 64 of
// them (n_a = 48, 2^18 points: 208 us a solve against 262 from 192; n_a = 37,
// 50 001 points: 135 against 169 from 16), 16 x 16 while those are at most one
// for each compute unit, K over 16 waves where it is long (or where a work-group
// of pass 1 squares powers: 6 squarings of 48 x 48 take 10 us with 16 waves, 34
// with 4), 32 x 32 between.  Systems launched together fill the GPU between them:
// the wider tiles from fewer (64 small systems: 785 us from 32 and 64, 897 from 64
// and 256; 512 systems 43.3 ms against 48), whatever the group, so that a
// system's results do not depend on it.
static int pass_tiling(const BlkPass& a, bool out, bool grouped)
{
    const long tx = (a.cols + kPT - 1) / kPT, ty = (a.nb + kPT - 1) / kPT;
    const long sx = (a.cols + 15) / 16, sy = (a.nb + 15) / 16;
    if (tx * ty >= (grouped ? 32 : 64)) return kBlockTile;
    if (sx * sy > (grouped ? 64 : 256)) return kBlockMid;
    return (!out && a.na > 16) || ((out ? a.kz : 0) + a.ku) / 4 >= 64 ? kBlockSplit16 : kBlockSplit4;
}
static void pass_grid(BlkPass& a, int tiling)
{
    const int t = tiling == kBlockTile ? kPT : tiling == kBlockMid ? 32 : 16;
    a.gx = (a.cols + t - 1) / t;
    a.gy = (a.nb + t - 1) / t;
    if (a.gx * a.gy >= 0x7fffffffL) throw std::length_error("block pass: too many tiles");
}

// The groups of waves over K that a wide tile has: four while the tiles leave every
// compute unit at most two (abm n = 203, 195 tiles: 994 us a solve, 1015 with two),
// two up to three (rk4 n = 128, 512 tiles in pass 1: 375 against 378 with one), one
// above (1024 tiles in pass 2: 375, with two 385).
template <bool OUT>
static void launch_pass(hipStream_t st, BlkPass a, bool uDouble, bool powers, int tiling)
{
    if (!tiling) tiling = pass_tiling(a, OUT, false);
    pass_grid(a, tiling);
    const dim3 grid((unsigned)(a.gx * a.gy + (powers ? 1 : 0)));
    const long tiles = a.gx * a.gy;
#define PARODE_PASS(TU)                                                                     \
    do {                                                                                    \
        if (tiling == kBlockTile && tiles <= 384)                                          \
            hipLaunchKernelGGL((k_blk_tile<TU, OUT, 4>), grid, dim3(1024), 0, st, a);       \
        else if (tiling == kBlockTile && tiles <= 768)                                     \
            hipLaunchKernelGGL((k_blk_tile<TU, OUT, 2>), grid, dim3(512), 0, st, a);        \
        else if (tiling == kBlockTile)                                                      \
            hipLaunchKernelGGL((k_blk_tile<TU, OUT, 1>), grid, dim3(256), 0, st, a);        \
        else if (tiling == kBlockMid && tiles <= 256)                                       \
            hipLaunchKernelGGL((k_blk_split<TU, OUT, 16, 2>), grid, dim3(1024), 0, st, a);  \
        else if (tiling == kBlockMid && tiles <= 512)                                       \
            hipLaunchKernelGGL((k_blk_split<TU, OUT, 8, 2>), grid, dim3(512), 0, st, a);    \
        else if (tiling == kBlockMid)                                                       \
            hipLaunchKernelGGL((k_blk_split<TU, OUT, 4, 2>), grid, dim3(256), 0, st, a);    \
        else if (tiling == kBlockSplit16)                                                   \
            hipLaunchKernelGGL((k_blk_split<TU, OUT, 16, 1>), grid, dim3(1024), 0, st, a);  \
        else                                                                                \
            hipLaunchKernelGGL((k_blk_split<TU, OUT, 4, 1>), grid, dim3(256), 0, st, a);    \
    } while (0)
    if (uDouble)
        PARODE_PASS(double);
    else
        PARODE_PASS(float);
#undef PARODE_PASS
    check_launch("block pass");
}

static BlkPass pass1_args(const BlockShape& s, const BlockBufs& b, const BlockInput& in, long nb)
{
    BlkPass a = pass_args(s, b, in, nb);
    a.cols = s.na;
    a.kz = 0;
    a.ku = s.kb();
    a.BU = b.QT;
    a.S = b.Z;
    return a;
}
static BlkPass pass2_args(const BlockShape& s, const BlockBufs& b, const BlockInput& in, long nb,
                          long nReal, const double* seed, const float* D, float* Y)
{
    BlkPass a = pass_args(s, b, in, nb);
    a.cols = s.T * s.p;
    a.kz = s.na;
    a.ku = s.kh();
    a.nReal = nReal;
    a.Z = b.E;
    a.OT = b.OT;
    a.BU = b.Ht;
    a.Y = Y;
    a.seed = seed;
    a.D = s.useD ? D : nullptr;
    return a;
}

void block_pass1(hipStream_t st, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                 long nb, bool powers, int tiling)
{
    launch_pass<false>(st, pass1_args(s, b, in, nb), in.isDouble, powers, tiling);
}

void block_pass2(hipStream_t st, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                 long nb, long nReal, const double* seed, const float* D, float* Y, int tiling)
{
    launch_pass<true>(st, pass2_args(s, b, in, nb, nReal, seed, D, Y), in.isDouble, false, tiling);
}

static BlkScan scan_args(const BlockShape& s, const BlockBufs& b, const BlockInput& in, long nb,
                         const double* seed)
{
    BlkScan a{};
    a.na = s.na;
    a.l0 = s.lb;
    a.L = s.L;
    a.nb = nb;
    a.PT = b.PT;
    a.E = b.Z;
    a.Zg = b.Z2;
    a.seed = seed;
    a.DL = b.DL;
    a.U = in.U;
    a.uDouble = in.isDouble;
    a.km = s.taps * s.m;
    a.m = s.m;
    a.gm = (int)(in.sL / s.s - 1) * s.m;
    a.magic = magic_of(s.m);
    a.last = in.last;
    return a;
}

static size_t scan_lds_bytes(const BlkScan& a)
{
    return (size_t)2 * 16 * a.R * ((a.na + 15) / 16 * 16 + 1) * sizeof(double);
}

// The scan's launches: u and d when the blocks go in groups (returns true), a
// over the blocks or the groups.
static bool scan_plan(BlkScan a0, const BlockBufs& b, BlkScan& u, BlkScan& a, BlkScan& d)
{
    const int lg = group_log(a0.nb);
    a = a0;
    a.R = 1;
    if (lg) {
        u = a0;
        u.lg = lg;
        u.R = 1;
        const long groups = block_groups(a0.nb);
        u.gx = (groups + 15) / 16;
        d = u;
        a.nb = groups;
        a.E = b.Z2;
        a.l0 = a0.l0 + lg;
    }
    // no more row tiles than the blocks need
    while (a.R < scan_row_tiles(a.na) && 16L * a.R < a.nb) a.R *= 2;
    a.lg = 0;
    while ((16L * a.R << a.lg) < a.nb) ++a.lg;
    a.gx = 1;
    return lg > 0;
}

void block_tree_finish(hipStream_t st, const BlockShape& s, const BlockBufs& b,
                       const BlockInput& in, long nb, const double* seed)
{
    const std::vector<TreeLevel> t = tree_of(s, nb);
    hipLaunchKernelGGL(k_blk_root, dim3((unsigned)((s.na + 15) / 16)), dim3(256), 0, st,
                       scan_args(s, b, in, nb, seed), tree_e(s, b, t, (int)t.size() - 1));
    check_launch("block root");
    for (int i = 0; i < block_tree_top_steps(s, nb); ++i) {
        const GemmOp op = block_tree_top(s, b, nb, i);
        gemm_multi(st, &op, 1);
    }
    for (int j = 0; j < block_tree_down_steps(s, nb); ++j) {
        const std::vector<GemmOp> ops = block_tree_down(s, b, nb, j);
        gemm_multi(st, ops.data(), (int)ops.size());
    }
}

template <int MODE>
static void launch_scan(hipStream_t st, const BlkScan& a)
{
    const int nct = (a.na + 15) / 16;
    const dim3 grid((unsigned)a.gx), wg((unsigned)(64 * nct * a.R));
    const size_t lds = scan_lds_bytes(a);
    if (nct == 1)
        hipLaunchKernelGGL((k_blk_scan<MODE, 4>), grid, wg, lds, st, a);
    else if (nct == 2)
        hipLaunchKernelGGL((k_blk_scan<MODE, 8>), grid, wg, lds, st, a);
    else if (nct == 3)
        hipLaunchKernelGGL((k_blk_scan<MODE, 12>), grid, wg, lds, st, a);
    else
        hipLaunchKernelGGL((k_blk_scan<MODE, 16>), grid, wg, lds, st, a);
    check_launch("block scan");
}

void block_scan(hipStream_t st, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                long nb, const double* seed)
{
    if (s.wide) {
        for (int k = 0; k < block_tree_up_levels(s, nb); ++k) {
            const GemmOp op = block_tree_up(s, b, nb, k);
            gemm_multi(st, &op, 1);
        }
        block_tree_finish(st, s, b, in, nb, seed);
        return;
    }
    BlkScan u, a, d;
    const bool groups = scan_plan(scan_args(s, b, in, nb, seed), b, u, a, d);
    if (groups) launch_scan<kScanUp>(st, u);
    launch_scan<kScanAll>(st, a);
    if (groups) launch_scan<kScanDown>(st, d);
}

void block_carry(hipStream_t st, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                 long nb, const double* seed, double* seedOut)
{
    const BlkScan a = scan_args(s, b, in, nb, seed);
    if (s.wide) {   // (nb is a power of two here)
        const std::vector<TreeLevel> t = tree_of(s, nb);
        const int top = (int)t.size() - 1;
        const size_t at = (size_t)(t[top].n - 1) * s.na;
        hipLaunchKernelGGL(k_blk_carry_wide, dim3((s.na + 255) / 256), dim3(256),
                           s.na * sizeof(double), st, a,
                           b.PT + (size_t)s.slot(s.lb + top) * s.na * s.na,
                           tree_e(s, b, t, top) + at, tree_s(s, b, t, top) + at,
                           nb * s.s * s.T, nb * s.T * in.sL * s.m, seedOut);
        check_launch("block carry");
        return;
    }
    hipLaunchKernelGGL(k_blk_carry, dim3(1), dim3(256), 0, st, a, nb * s.s * s.T,
                       nb * s.T * in.sL * s.m, seedOut);
    check_launch("block carry");
}

// ---------------------------------------------------------- grouped launches
namespace g {

namespace {

struct StartOutB {
    BlockShape s;
    const float *C, *D;
    const double *X0, *U;
    float* Y;
    long gx;
};
struct RootB {
    BlkScan a;
    double* E;
    long gx;
};

__global__ __launch_bounds__(1024) void kg_blk_tables(const BlkTables* __restrict__ args,
                                                      const unsigned* __restrict__ st, int ns)
{
    PARODE_GROUP(BlkTables);
    __shared__ double lds[kTabLds];
    d_blk_tables<double>(vb, a, lds);
}
__global__ __launch_bounds__(256) void kg_blk_elem(const BlkElem* __restrict__ args,
                                                   const unsigned* __restrict__ st, int ns)
{
    PARODE_GROUP(BlkElem);
    d_blk_elem(vb, a);
}
__global__ __launch_bounds__(256) void kg_blk_start_outputs(const StartOutB* __restrict__ args,
                                                            const unsigned* __restrict__ st, int ns)
{
    PARODE_GROUP(StartOutB);
    (void)vb;
    d_start_outputs<double>(a.s, a.C, a.D, a.X0, a.U, a.Y);
}
// (a system's last work-group of pass 1 squares the rest of its powers, if any)
template <bool OUT, int NW, int R>
__global__ __launch_bounds__(NW * 64) void kg_blk_split(const BlkPass* __restrict__ args,
                                                        const unsigned* __restrict__ st, int ns)
{
    constexpr int kPart = R > 1 ? NW * 256 * R * R : (NW - 1) * 256;
    constexpr int kLds = OUT || kPart > kBN * kBP ? kPart : kBN * kBP;
    __shared__ double lds[kLds];
    __shared__ int bad;
    const int sys = system_of(st, ns);
    const BlkPass& a = args[sys];
    const long idx = (long)blockIdx.x - (long)st[sys];
    if (!OUT && idx == a.gx * a.gy) {
        d_blk_powers<NW>(a.na, a.lb, a.L, a.PT, lds);
        return;
    }
    d_blk_split<double, OUT, NW, R>(blk_place(idx, a.gx, a.gy), a, lds, &bad);
}
template <bool OUT>
__global__ __launch_bounds__(256, 4) void kg_blk_tile(const BlkPass* __restrict__ args,
                                                      const unsigned* __restrict__ st, int ns)
{
    __shared__ BlkTileLds<1> L;
    const int sys = system_of(st, ns);
    const BlkPass& a = args[sys];
    const long idx = (long)blockIdx.x - (long)st[sys];
    if (!OUT && idx == a.gx * a.gy) {
        d_blk_powers<4>(a.na, a.lb, a.L, a.PT, &L.stage[0].A[0][0][0]);
        return;
    }
    d_blk_tile<double, OUT, 1>(blk_place(idx, a.gx, a.gy), a, L);
}
template <int MODE>
__global__ __launch_bounds__(MODE == kScanAll ? 1024 : 256) void kg_blk_scan(
    const BlkScan* __restrict__ args, const unsigned* __restrict__ st, int ns)
{
    extern __shared__ double scan_lds[];
    PARODE_GROUP(BlkScan);
    d_blk_scan<MODE>(vb, a, scan_lds);
}
__global__ __launch_bounds__(256) void kg_blk_root(const RootB* __restrict__ args,
                                                   const unsigned* __restrict__ st, int ns)
{
    PARODE_GROUP(RootB);
    d_blk_root(vb, a.a, a.E);
}

void add_pass(Phase& ph, BlkPass a, bool out, bool powers)
{
    const int t = pass_tiling(a, out, true);
    pass_grid(a, t);
    const float cost = (float)((out ? a.kz : 0) + a.ku);
    append(ph,
           t == kBlockTile      ? kBlkTile
           : t == kBlockMid     ? kBlkMid
           : t == kBlockSplit16 ? kBlkSplit16
                                : kBlkSplit4,
           out, a,
           a.gx * a.gy + (powers ? 1 : 0), 0, cost);
}

}  // namespace

void add_block_tables(Phase& ph, const BlockShape& s, const BlockBufs& b, double h, const float* A,
                      const float* B, const float* C, const float* D, const float* x0, double* seed)
{
    // (an ABM start-up reads the input samples: it has a launch of its own)
    const BlkTables a = table_args(s, b, h, A, B, C, D, s.method == 0 ? x0 : nullptr, nullptr, seed,
                                   nullptr, true);
    append(ph, kBlkTables, false, a, a.gx, 0, (float)s.na * s.lb);
}
void add_block_elem(Phase& ph, const BlkElem& e)
{
    if (e.count <= 0) return;
    append(ph, kBlkElem, false, e, e.gx);
}
void add_block_start_outputs(Phase& ph, const BlockShape& s, const float* C, const float* D,
                             const double* X0, const double* U, float* Y)
{
    append(ph, kBlkStartOut, false, StartOutB{s, C, D, X0, U, Y, 1}, 1);
}
void add_block_pass1(Phase& ph, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                     long nb)
{
    add_pass(ph, pass1_args(s, b, in, nb), false, !s.wide);
}
void add_block_pass2(Phase& ph, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                     long nb, long nReal, const double* seed, const float* D, float* Y)
{
    add_pass(ph, pass2_args(s, b, in, nb, nReal, seed, D, Y), true, false);
}
void add_block_scan(Phase& up, Phase& all, Phase& down, const BlockShape& s, const BlockBufs& b,
                    const BlockInput& in, long nb, const double* seed)
{
    BlkScan u, a, d;
    if (scan_plan(scan_args(s, b, in, nb, seed), b, u, a, d)) {
        append(up, kBlkScanUp, false, u, u.gx, scan_lds_bytes(u), (float)(s.na << u.lg));
        append(down, kBlkScanDown, false, d, d.gx, scan_lds_bytes(d), (float)(s.na << d.lg));
    }
    append(all, kBlkScanAll, false, a, 1, scan_lds_bytes(a), (float)(s.na << a.lg));
}
void add_block_root(Phase& ph, const BlockShape& s, const BlockBufs& b, const BlockInput& in,
                    long nb, const double* seed)
{
    const std::vector<TreeLevel> t = tree_of(s, nb);
    const int top = (int)t.size() - 1;
    const long gx = (s.na + 15) / 16;
    append(ph, kBlkRoot, false, RootB{scan_args(s, b, in, nb, seed), tree_e(s, b, t, top), gx}, gx, 0,
           (float)(s.taps * s.m));
}

bool run_blocks(hipStream_t s, const Launch& L, const void* dArgs, const unsigned* dStart)
{
    const int ns = L.nsys();
    const dim3 grid(L.blocks());
    const size_t lds = L.lds;
#define PARODE_RUN(KERNEL, T, THREADS)                                                        \
    hipLaunchKernelGGL((KERNEL), grid, dim3(THREADS), lds, s, static_cast<const T*>(dArgs),   \
                       dStart, ns)
    switch (L.kind) {
    case kBlkTables: PARODE_RUN(kg_blk_tables, BlkTables, 1024); break;
    case kBlkElem: PARODE_RUN(kg_blk_elem, BlkElem, 256); break;
    case kBlkStartOut: PARODE_RUN(kg_blk_start_outputs, StartOutB, 256); break;
    case kBlkTile:
        if (L.flag)
            PARODE_RUN(kg_blk_tile<true>, BlkPass, 256);
        else
            PARODE_RUN(kg_blk_tile<false>, BlkPass, 256);
        break;
    case kBlkSplit4:
        if (L.flag)
            PARODE_RUN((kg_blk_split<true, 4, 1>), BlkPass, 256);
        else
            PARODE_RUN((kg_blk_split<false, 4, 1>), BlkPass, 256);
        break;
    case kBlkMid:
        if (L.flag)
            PARODE_RUN((kg_blk_split<true, 8, 2>), BlkPass, 512);
        else
            PARODE_RUN((kg_blk_split<false, 8, 2>), BlkPass, 512);
        break;
    case kBlkSplit16:
        if (L.flag)
            PARODE_RUN((kg_blk_split<true, 16, 1>), BlkPass, 1024);
        else
            PARODE_RUN((kg_blk_split<false, 16, 1>), BlkPass, 1024);
        break;
    case kBlkScanUp: PARODE_RUN(kg_blk_scan<kScanUp>, BlkScan, 256); break;
    case kBlkScanAll: PARODE_RUN(kg_blk_scan<kScanAll>, BlkScan, 1024); break;
    case kBlkScanDown: PARODE_RUN(kg_blk_scan<kScanDown>, BlkScan, 256); break;
    case kBlkRoot: PARODE_RUN(kg_blk_root, RootB, 256); break;
    default: return false;
    }
#undef PARODE_RUN
    return true;
}

}  // namespace g

}  // namespace k
}  // namespace parode
