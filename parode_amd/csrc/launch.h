// What the kernel files share: the place of a work-group in its system's grid,
// launch checks, the records of grouped launches, and the ABM start-up body.
#pragma once
#include "kernels.h"

#include <algorithm>
#include <cstring>
#include <stdexcept>
#include <string>

namespace parode {
namespace k {

typedef double doublex4 __attribute__((ext_vector_type(4)));
// two doubles at any 8-byte address (one 16-byte load: the hardware takes it)
typedef double double2u __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ void load4(const double* p, double (&r)[4])
{
    const double2u a = *reinterpret_cast<const double2u*>(p);
    const double2u b = *reinterpret_cast<const double2u*>(p + 2);
    r[0] = a.x;
    r[1] = a.y;
    r[2] = b.x;
    r[3] = b.y;
}
// four floats at any 4-byte address
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void load4(const float* p, double (&r)[4])
{
    const float4u a = *reinterpret_cast<const float4u*>(p);
    r[0] = a.x;
    r[1] = a.y;
    r[2] = a.z;
    r[3] = a.w;
}

// The block a kernel body works on: (x, y) and the grid's width in x.  A
// single-system launch passes its own blockIdx and gridDim; a grouped launch
// (many systems in one grid) passes the block's place in its system's grid.
struct VBlock {
    long x, y, gx;
};

inline void check_launch(const char* what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        throw std::runtime_error(std::string("kernel launch failed: ") + what + ": " +
                                 hipGetErrorString(e));
}

inline unsigned blocks_for(long work, int block, long cap = 1L << 20)
{
    long b = (work + block - 1) / block;
    if (b < 1) b = 1;
    return (unsigned)std::min(b, cap);
}

// ------------------------------------------------------------ ABM start-up
// Three classic RK4 steps (AdamsMoulton.cpp:96-103).  mirror: float state and
// float derivative sums (AdamsMoulton.cpp:15-27), stage combinations formed
// in double and stored to float (odeint runge_kutta4<vector<float>>).
// When A fits (pitch n + 1, no bank conflicts), it is staged in LDS once: the
// twelve derivative evaluations are chains of n dependent products per row,
// which from global memory wait on a load each.
template <typename TU>
__device__ __forceinline__ void d_abm_startup(const VBlock vb, bool mirror, int n, int m, double h, bool ldsA,
                              const float* __restrict__ A, const float* __restrict__ B,
                              const float* __restrict__ x0, const TU* __restrict__ Uh,
                              double* __restrict__ X0)
{
#pragma clang fp contract(off)
    extern __shared__ double sh[];
    double* x = sh;            // n
    double* xt = sh + n;       // n
    double* kb = sh + 2 * n;   // 4n: k1..k4
    float* As = reinterpret_cast<float*>(sh + 6 * n);   // n x (n + 1) when ldsA
    const double dh = h / 2.0, dt6 = h / 6.0, dt3 = h / 3.0;
    for (int r = threadIdx.x; r < n; r += blockDim.x) {
        x[r] = (double)x0[r];
        X0[r] = (double)x0[r];
    }
    if (ldsA)
        for (int t = threadIdx.x; t < n * n; t += blockDim.x) {
            const int r = t / n;
            As[t + r] = A[t];   // row r at r * (n + 1)
        }
    __syncthreads();
    const float* Ar = ldsA ? As : A;
    const long ap = ldsA ? n + 1 : n;
    auto deriv = [&](const double* xs, int urow, double* out) {
        for (int r = threadIdx.x; r < n; r += blockDim.x) {
            if (mirror) {
                float f = 0.0f;
                for (int c = 0; c < n; ++c) {
                    float pr = Ar[r * ap + c] * (float)xs[c];
                    f = f + pr;
                }
                for (int c = 0; c < m; ++c) {
                    float pr = B[(long)r * m + c] * (float)Uh[(long)urow * m + c];
                    f = f + pr;
                }
                out[r] = (double)f;
            } else {
                double f = 0.0;
                for (int c = 0; c < n; ++c) f = fma((double)Ar[r * ap + c], xs[c], f);
                for (int c = 0; c < m; ++c)
                    f = fma((double)B[(long)r * m + c], (double)Uh[(long)urow * m + c], f);
                out[r] = f;
            }
        }
        __syncthreads();
    };
    auto stage = [&](const double* kk, double coef) {
        for (int r = threadIdx.x; r < n; r += blockDim.x) {
            double v = 1.0 * x[r] + coef * kk[r];
            xt[r] = mirror ? (double)(float)v : v;
        }
        __syncthreads();
    };
    for (int s = 0; s < 3; ++s) {
        double* k1 = kb;
        double* k2 = kb + n;
        double* k3 = kb + 2 * n;
        double* k4 = kb + 3 * n;
        deriv(x, 2 * s, k1);
        stage(k1, dh);
        deriv(xt, 2 * s + 1, k2);
        stage(k2, dh);
        deriv(xt, 2 * s + 1, k3);
        stage(k3, h);
        deriv(xt, 2 * s + 2, k4);
        for (int r = threadIdx.x; r < n; r += blockDim.x) {
            double v;
            if (mirror)
                v = (double)(float)((((1.0 * x[r] + dt6 * k1[r]) + dt3 * k2[r]) + dt3 * k3[r]) +
                                    dt6 * k4[r]);
            else
                v = x[r] + (h / 6.0) * (k1[r] + 2.0 * k2[r] + 2.0 * k3[r] + k4[r]);
            x[r] = v;
            X0[(long)(s + 1) * n + r] = v;
        }
        __syncthreads();
    }
}

// The same steps for n, m <= 256 with 1024 threads: four lanes a row, each
// with NC of the row's columns in registers, so that a derivative is NC
// products from registers and LDS instead of a chain of n loads (us, one lane a
// row and four: n = 203 286 and 45, n = 64 48 and 13, n = 16 15 and 8, n = 1 6 and
// 8).  mirror: the row's float sum runs through the four lanes in column order, a
// chain of n products again (n = 203 286 and 138, n = 64 51 and 43, n = 16 15.7 and
// 15.6).
template <typename TU, int NC>
__device__ __forceinline__ void startup_rows(bool mirror, int n, int m, double h,
                                             const float* __restrict__ A,
                                             const float* __restrict__ B,
                                             const float* __restrict__ x0,
                                             const TU* __restrict__ Uh, double* __restrict__ X0)
{
#pragma clang fp contract(off)
    __shared__ double xs[4 * (NC + 2)], us[7 * 256];
    const int r = threadIdx.x >> 2, q = threadIdx.x & 3, lane = threadIdx.x & 63;
    const bool row = r < n;
    const int mq = (m + 3) / 4, mb = q * mq, me = mb + mq < m ? mb + mq : m;
    float a[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int k = q * NC + c;
        a[c] = (row && k < n) ? A[(long)r * n + k] : 0.0f;
    }
    for (int t = threadIdx.x; t < 7 * m; t += 1024) us[t / m * 256 + t % m] = (double)Uh[t];
    double x = row ? (double)x0[r] : 0.0;
    if (row && q == 0) X0[r] = x;
    const int slot = r / NC * (NC + 2) + r % NC;   // row r's place in xs
    if (q == 0 && r < 4 * NC) xs[slot] = x;
    __syncthreads();
    const float* Br = B + (long)(row ? r : 0) * m;
    auto deriv = [&](int urow) {
        const double* u = us + urow * 256;
        const double* xq = xs + q * (NC + 2);
        double y;
        if (mirror) {
            float f = 0.0f;
            // (segments past the last column or input add nothing)
#pragma unroll
            for (int seg = 0; seg < 4; ++seg) {
                if (seg * NC >= n) break;
                if (q == seg)
#pragma unroll
                    for (int c = 0; c < NC; ++c) {
                        const float pr = a[c] * (float)xq[c];
                        if (q * NC + c < n) f = f + pr;
                    }
                f = __shfl(f, (lane & ~3) + seg);
            }
            for (int seg = 0; seg < 4 && seg * mq < m; ++seg) {
                if (q == seg)
                    for (int c = mb; c < me; ++c) {
                        const float pr = Br[c] * (float)u[c];
                        f = f + pr;
                    }
                f = __shfl(f, (lane & ~3) + seg);
            }
            y = (double)f;
        } else {
            double f = 0.0;
#pragma unroll
            for (int c = 0; c < NC; ++c) f = fma((double)a[c], xq[c], f);
            for (int c = mb; c < me; ++c) f = fma((double)Br[c], u[c], f);
            f += __shfl_xor(f, 1);
            f += __shfl_xor(f, 2);
            y = f;
        }
        return y;
    };
    auto put = [&](double v) {
        __syncthreads();   // every derivative has read xs
        if (q == 0 && r < 4 * NC) xs[slot] = row ? v : 0.0;
        __syncthreads();
    };
    auto stage = [&](double k, double coef) {
        const double v = 1.0 * x + coef * k;
        put(mirror ? (double)(float)v : v);
    };
    const double dh = h / 2.0, dt6 = h / 6.0, dt3 = h / 3.0;
    for (int s = 0; s < 3; ++s) {
        const double k1 = deriv(2 * s);
        stage(k1, dh);
        const double k2 = deriv(2 * s + 1);
        stage(k2, dh);
        const double k3 = deriv(2 * s + 1);
        stage(k3, h);
        const double k4 = deriv(2 * s + 2);
        if (mirror)
            x = (double)(float)((((1.0 * x + dt6 * k1) + dt3 * k2) + dt3 * k3) + dt6 * k4);
        else
            x = x + (h / 6.0) * (k1 + 2.0 * k2 + 2.0 * k3 + k4);
        if (row && q == 0) X0[(long)(s + 1) * n + r] = x;
        put(x);
    }
}

inline bool startup_rows_fit(int n, int m) { return n <= 256 && m <= 256; }
template <typename TU>
__device__ __forceinline__ void d_startup_rows(bool mirror, int n, int m, double h, const float* A,
                                               const float* B, const float* x0, const TU* Uh,
                                               double* X0)
{
    if (n <= 16)
        startup_rows<TU, 4>(mirror, n, m, h, A, B, x0, Uh, X0);
    else if (n <= 64)
        startup_rows<TU, 16>(mirror, n, m, h, A, B, x0, Uh, X0);
    else if (n <= 128)
        startup_rows<TU, 32>(mirror, n, m, h, A, B, x0, Uh, X0);
    else
        startup_rows<TU, 64>(mirror, n, m, h, A, B, x0, Uh, X0);
}

// ---------------------------------------------------------- grouped launches
namespace g {

__device__ __forceinline__ int system_of(const unsigned* __restrict__ start, int nsys)
{
    const unsigned b = blockIdx.x;
    int lo = 0, hi = nsys - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (start[mid] <= b)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ VBlock block_of(const unsigned* __restrict__ start, int s, long gx)
{
    const long lb = (long)blockIdx.x - (long)start[s];
    return VBlock{lb % gx, lb / gx, gx};
}

#define PARODE_GROUP(T)                          \
    const int sys_ = system_of(st, ns);          \
    const T& a = args[sys_];                     \
    const VBlock vb = block_of(st, sys_, a.gx)

// The record of the launch (kind, flag) in phase ph, created on first use.
template <typename A>
inline Launch& slot(Phase& ph, int kind, bool flag, int cls)
{
    Launch& L = ph[{kind, (flag ? 1 : 0) + 2 * cls}];
    if (L.kind < 0) {
        L.kind = kind;
        L.flag = flag;
        L.argSize = sizeof(A);
    }
    if (L.argSize != sizeof(A)) throw std::logic_error("grouped launch: argument type mismatch");
    return L;
}

// Systems whose dynamic LDS differs go to separate launches by size class
// (up to 8, 16, 32, 48, 64 KiB ...): a launch reserves its largest system's
// LDS for every work-group, which would cap the occupancy of the others.
inline int lds_class(size_t lds)
{
    if (lds == 0) return 0;
    const size_t kib = (lds + 1023) / 1024;
    return kib <= 8 ? 1 : kib <= 16 ? 2 : kib <= 32 ? 3 : kib <= 48 ? 4 : 5 + (int)((kib - 49) / 16);
}

template <typename A>
inline void append(Phase& ph, int kind, bool flag, const A& a, long blocks, size_t lds = 0,
            float cost = 0.0f)
{
    if (blocks < 1) return;
    // (the top of the tree runs one 1024-thread work-group per system, one per
    // CU whatever its LDS: its systems share one launch)
    const bool oneClass = kind == kTopMfma || kind == kTopSimt;
    Launch& L = slot<A>(ph, kind, flag, oneClass ? 0 : lds_class(lds));
    const size_t o = L.args.size();
    L.args.resize(o + sizeof(A));
    std::memcpy(L.args.data() + o, &a, sizeof(A));
    const unsigned long next = (unsigned long)L.start.back() + (unsigned long)blocks;
    if (next > 0x7fffffffUL) throw std::length_error("grouped launch: too many blocks");
    L.start.push_back((unsigned)next);
    L.cost.push_back(cost);
    L.lds = std::max(L.lds, lds);
}

}  // namespace g
}  // namespace k
}  // namespace parode
