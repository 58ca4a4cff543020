#pragma once
// Vector kernels of the GMRES solvers (krylov.hip), for FP32 and FP64 bases: the dot products of an Arnoldi step in one
// pass over the basis, its update in another, and the hand-over of the step's coefficients to the host, which runs the
// Hessenberg least squares.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

namespace mhdg
{
constexpr int kDotChunk = 16;       // basis vectors per dot-product pass
constexpr int kOrthoBlocks = 1024;  // largest grid of the vector kernels (512 and 2048 measured no better)
constexpr int kOrthoThreads = 256;
// Up to this many blocks of a dot-product pass the update's blocks sum the partials themselves (1 KB a column from the L2: 17
// columns for 16 vectors, 121 with the Gram columns of 60) and the launch that sums them, 4 us and its gap on a step of 40 us, goes; with 1024 blocks of partials
// that would read 280 MB.
constexpr int kFoldBlocks = 128;
constexpr int kMaxRestart = 60;     // vectors of a cycle: their coefficients, the norm, then slots 62 (re-projection) and 63 (<w, w>)
// Columns of partial sums: <V_i, w> at i, <w, w> at kColWW, <V_i, V_j> at kColGram + i
constexpr int kColWW = 63, kColGram = 64, kCols = 128;
static_assert(kMaxRestart + 1 < 62 && kMaxRestart <= kCols - kColGram, "the coefficients and the norm end before slot 62");

// What a kernel hands to the host (pinned host memory): written, then the ticket.
struct HostBox
{
    double v[64];
    uint64_t ticket;
};

// values to the host: every thread's store, then the ticket after a system-scope release (called by a whole block)
__device__ __forceinline__ void publish(HostBox *box, uint64_t ticket, const double *v, int32_t n)
{
    if (int32_t(threadIdx.x) < n) __hip_atomic_store(&box->v[threadIdx.x], v[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(&box->ticket, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

inline int ortho_blocks(int32_t n, int vec)
{
    const int64_t b = (int64_t(n) / vec + kOrthoThreads) / kOrthoThreads;
    return static_cast<int>(b < kOrthoBlocks ? b : kOrthoBlocks);
}

// Orthogonalisation of w against V_0 .. V_{nv-1}
template <class T> struct Ortho
{
    const T *const *V;   // basis pointers
    int32_t nv, n;
    T *w, *vnext;        // the vector, and V_nv
    const T *vj;         // V_{nv-1}, the newest basis vector
    const T *invdiag;    // FP32: pv = dir ? 0 : V_nv invdiag is written too
    const int8_t *dir;
    T *pv;
    double *part;        // kCols columns of kOrthoBlocks partials
    double *cols;        // kCols sums
    double *h;           // 64: the coefficients of kPlain and kMgs, for ortho_scale
    double *gram;        // 64 x 64: <V_i, V_k>, k < i (modified Gram-Schmidt)
    double *norms;       // kOrthoBlocks partials of |w'|^2
    HostBox *box;
    uint64_t ticket;
};
// coefficients of the solution update, by value (no copy to the device per cycle)
struct Coefs
{
    double v[64];
};

// Hessenberg least squares of restarted GMRES with Givens rotations (ImplicitInduction.cpp:326-377)
struct Hessenberg
{
    std::vector<std::vector<double>> H;
    std::vector<double> cs, sn, g;
    explicit Hessenberg(int m) : H(m + 1, std::vector<double>(m, 0.0)), cs(m), sn(m), g(m + 1) {}
    void start(double beta)
    {
        std::fill(g.begin(), g.end(), 0.0);
        g[0] = beta;
    }
    // column j: h_0 .. h_j (plus `shift` on the diagonal), h_{j+1,j} = hn; returns the residual estimate |g_{j+1}|
    double add(int j, const double *h, double shift, double hn)
    {
        for (int i = 0; i <= j; ++i) H[i][j] = h[i];
        H[j][j] += shift;
        H[j + 1][j] = hn;
        for (int i = 0; i < j; ++i)
        {
            const double tt = cs[i] * H[i][j] + sn[i] * H[i + 1][j];
            H[i + 1][j] = -sn[i] * H[i][j] + cs[i] * H[i + 1][j];
            H[i][j] = tt;
        }
        const double den = std::hypot(H[j][j], H[j + 1][j]);
        cs[j] = den > 0 ? H[j][j] / den : 1.0;
        sn[j] = den > 0 ? H[j + 1][j] / den : 0.0;
        H[j][j] = den;
        H[j + 1][j] = 0.0;
        g[j + 1] = -sn[j] * g[j];
        g[j] = cs[j] * g[j];
        return std::abs(g[j + 1]);
    }
    Coefs solve(int j) const
    {
        Coefs y{};
        for (int i = j - 1; i >= 0; --i)
        {
            double s = g[i];
            for (int k = i + 1; k < j; ++k) s -= H[i][k] * y.v[k];
            y.v[i] = s / H[i][i];
        }
        return y;
    }
};
enum : int { kCgs = 0, kPlain = 1, kMgs = 2 };

// all dot products of the step in one pass over V and w (two for more than kDotChunk vectors)
template <class T> void ortho_dots(const Ortho<T> &o, bool gram, hipStream_t s);
// mode kCgs: w' = w - sum h_i V_i with h_i = <V_i, w>, V_nv = w' / hn with hn^2 = <w, w> - sum h_i^2, when that keeps at
//   least dgks of |w|; else w' goes to w for a second projection (box v[62] = 1).  Box: h_0 .. h_{nv-1}, hn at nv.
// mode kPlain: V_nv = w' unscaled (the second projection); mode kMgs: the same with modified Gram-Schmidt's coefficients.
template <class T> void ortho_update(const Ortho<T> &o, int mode, double dgks, hipStream_t s);
// V_nv = w' / |w'| after kPlain or kMgs.  Box: the coefficients and |w'| at nv.
template <class T> void ortho_scale(const Ortho<T> &o, hipStream_t s);
// delta += dir ? 0 : invdiag sum_{i < j} y_i V_i, x = x0 + delta (the Krylov solution, right Jacobi preconditioner)
template <class T>
void solution_update(const T *const *V, const Coefs &y, int32_t j, const T *invdiag, const int8_t *dir, int32_t n, const double *x0,
                     double *delta, double *x, hipStream_t s);
// box v[0] = <a, a>, v[1] = <b, b> (b nullable) and their square roots on the device in out[0], out[1]
void norms2(const double *a, const double *b, int32_t n, double *part, double *out, HostBox *box, uint64_t ticket, hipStream_t s);
} // namespace mhdg
