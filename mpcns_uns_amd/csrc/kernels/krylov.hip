// Vector kernels of the GMRES solvers (krylov.h).  Every reduction has a fixed grid for its length, a fixed tree per block
// and a fixed order over the blocks, so reruns are bit-identical.
//
// All of them stream: their time is their bytes over the copy rate (6.1 TB/s here) on large meshes, and launches plus one
// round trip through memory on small ones.  So an Arnoldi step reads the basis twice and no more (modified Gram-Schmidt,
// whose coefficients depend on each other, read w and two vectors and wrote w for each of them: 2 (j + 2) launches), its
// coefficients reach the host through pinned memory that the kernel writes (a copy, an event wait and their gaps cost
// 12 us a step), and the update walks its range backwards: the end of what the dot products read last is still in the
// 256 MB cache behind the L2s (3 % of the update on the 8M shell).
//
// Measured on one MI355X, with the high-valence edges in the operator's own launch: the FP64 Hall step with modified
// Gram-Schmidt 1.95M tetrahedra 12.3 -> 9.7 ms (18 iterations; its orthogonalisation 3.95 -> 1.4 ms), 9.5k tetrahedra 490
// -> 235 us (4 and 3 iterations); the mixed step, 60k tetrahedra 590 -> 350 us (6 and 5 iterations), 7.83M 42.5 -> 40.2 ms.
#include "krylov.h"

#include <array>
#include <utility>

namespace mhdg
{
namespace
{
template <class T> struct Pack;
template <> struct Pack<float>
{
    static constexpr int N = 4;
    typedef float Raw __attribute__((ext_vector_type(4)));
};
template <> struct Pack<double>
{
    static constexpr int N = 2;
    typedef double Raw __attribute__((ext_vector_type(2)));
};
// 16-byte loads through a pointer known to be global memory (a pointer read from LDS or an array is generic, and its
// loads become flat loads that also count against the LDS wait counter)
template <class T> __device__ __forceinline__ typename Pack<T>::Raw ldg(const T *p, int32_t q)
{
    typedef const __attribute__((address_space(1))) typename Pack<T>::Raw *G;
    return ((G)p)[q];
}
template <class T> __device__ __forceinline__ double dot_pack(const typename Pack<T>::Raw &a, const typename Pack<T>::Raw &b)
{
    if constexpr (sizeof(T) == 4) return (double(a.x) * b.x + double(a.y) * b.y) + (double(a.z) * b.z + double(a.w) * b.w);
    else return a.x * b.x + a.y * b.y;
}
__device__ __forceinline__ double wave_sum(double v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}
// sum over the block in thread 0 (sh: one slot per wave)
__device__ __forceinline__ double block_total(double v, double *sh)
{
    const double s = wave_sum(v);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    const double r = ((sh[0] + sh[1]) + sh[2]) + sh[3];
    __syncthreads();
    return r;
}
// Per-block partials of <V_{i0+k}, w>, k < NV, of <w, w> (ww) and of <V_{i0+k}, V_j> (GRAM, vj).  NV is a template argument
// so that the NV loads of an iteration are issued together (a run-time count guarded each load by a branch and kept one
// load in flight per thread).
template <class T, int NV, bool GRAM>
__global__ void __launch_bounds__(kOrthoThreads) k_dots(const T *const *V, int32_t i0, const T *w, const T *vj, int32_t n, int32_t ww,
                                                        double *part)
{
    constexpr int P = Pack<T>::N, NC = NV + 1 + (GRAM ? NV : 0);
    __shared__ double sh[4][NC];
    double acc[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) acc[k] = 0.0;
    const T *Vk[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) Vk[k] = V[i0 + k];
    const int32_t np = n / P;
    for (int32_t q = blockIdx.x * kOrthoThreads + threadIdx.x; q < np; q += gridDim.x * kOrthoThreads)
    {
        const auto a = ldg<T>(w, q);
        typename Pack<T>::Raw g = a;
        if (GRAM) g = ldg<T>(vj, q);
        typename Pack<T>::Raw b[NV];
#pragma unroll
        for (int k = 0; k < NV; ++k) b[k] = ldg<T>(Vk[k], q);
#pragma unroll
        for (int k = 0; k < NV; ++k) acc[k] += dot_pack<T>(a, b[k]);
        acc[NV] += dot_pack<T>(a, a);
        if (GRAM)
#pragma unroll
            for (int k = 0; k < NV; ++k) acc[NV + 1 + k] += dot_pack<T>(g, b[k]);
    }
    if (blockIdx.x == 0 && int32_t(threadIdx.x) < n - P * np)
    {
        const int32_t e = P * np + threadIdx.x;
        const double a = w[e];
#pragma unroll
        for (int k = 0; k < NV; ++k)
        {
            acc[k] += a * Vk[k][e];
            if (GRAM) acc[NV + 1 + k] += double(vj[e]) * Vk[k][e];
        }
        acc[NV] += a * a;
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NC; ++k)
    {
        const double s = wave_sum(acc[k]);
        if (lane == 0) sh[wv][k] = s;
    }
    __syncthreads();
    const int k = threadIdx.x;
    if (k < NC && (k != NV || ww))
    {
        const int col = k < NV ? i0 + k : k == NV ? kColWW : kColGram + i0 + (k - NV - 1);
        part[size_t(col) * kOrthoBlocks + blockIdx.x] = ((sh[0][k] + sh[1][k]) + sh[2][k]) + sh[3][k];
    }
}
// one column's sum per block: columns 0 .. nv-1, <w, w>, and with `gram` <V_i, V_j> for i < nv
__global__ void __launch_bounds__(kOrthoThreads) k_cols_final(const double *part, int32_t nblocks, int32_t nv, double *cols)
{
    __shared__ double sh[4];
    const int b = blockIdx.x, col = b < nv ? b : b == nv ? kColWW : kColGram + (b - nv - 1);
    double t = 0.0;
    for (int32_t i = threadIdx.x; i < nblocks; i += kOrthoThreads) t += part[size_t(col) * kOrthoBlocks + i];
    t = block_total(t, sh);
    if (threadIdx.x == 0) cols[col] = t;
}

// The step's sums in LDS: c[i] = <V_i, w>, c[63] = <w, w>, and with GRAM g[i] = <V_i, V_j>; from `cols`, or (fold blocks of
// partials) summed here, four threads to a column
template <bool GRAM> __device__ __forceinline__ void load_cols(const double *part, const double *cols, int32_t fold, int32_t nv, double *c, double *g)
{
    const int32_t nc = nv + 1 + (GRAM ? nv : 0);
    for (int32_t k0 = 0; k0 < nc; k0 += kOrthoThreads / 4)
    {
        const int32_t k = k0 + int32_t(threadIdx.x >> 2), q = threadIdx.x & 3;
        const int32_t col = k < nv ? k : k == nv ? kColWW : kColGram + (k - nv - 1);
        double t = 0.0;
        if (k < nc)
        {
            if (fold)
                for (int32_t i = q; i < fold; i += 4) t += part[size_t(col) * kOrthoBlocks + i];
            else if (q == 0) t = cols[col];
        }
        const double t1 = __shfl_down(t, 1, 4), t2 = __shfl_down(t, 2, 4), t3 = __shfl_down(t, 3, 4);
        if (k < nc && q == 0)
        {
            if (fold) t = ((t + t1) + t2) + t3;
            if (k <= nv) c[k < nv ? k : kColWW] = t;
            else g[k - nv - 1] = t;
        }
    }
    __syncthreads();
}

// x -= h_i V_i for the G vectors from i0 on, in order (their G loads issued together)
template <class T, int G>
__device__ __forceinline__ void axpy_group(const T *const *vp, const double *hs, int32_t i0, int32_t q, double (&x)[Pack<T>::N])
{
    typename Pack<T>::Raw b[G];
#pragma unroll
    for (int k = 0; k < G; ++k) b[k] = ldg<T>(vp[i0 + k], q);
#pragma unroll
    for (int k = 0; k < G; ++k)
    {
        const double hi = hs[i0 + k];
#pragma unroll
        for (int m = 0; m < Pack<T>::N; ++m) x[m] -= hi * b[k][m];
    }
}
constexpr int kAxpyGroup = 8;
// x -= sum_{i < nv} h_i V_i in order of i: groups of kAxpyGroup loads, then the remainder's loads together
template <class T> __device__ __forceinline__ void axpy_all(const T *const *vp, const double *hs, int32_t nv, int32_t q, double (&x)[Pack<T>::N])
{
    int32_t i = 0;
    for (; i + kAxpyGroup <= nv; i += kAxpyGroup) axpy_group<T, kAxpyGroup>(vp, hs, i, q, x);
    switch (nv - i)
    {
    case 7: axpy_group<T, 7>(vp, hs, i, q, x); break;
    case 6: axpy_group<T, 6>(vp, hs, i, q, x); break;
    case 5: axpy_group<T, 5>(vp, hs, i, q, x); break;
    case 4: axpy_group<T, 4>(vp, hs, i, q, x); break;
    case 3: axpy_group<T, 3>(vp, hs, i, q, x); break;
    case 2: axpy_group<T, 2>(vp, hs, i, q, x); break;
    case 1: axpy_group<T, 1>(vp, hs, i, q, x); break;
    default: break;
    }
}

// Modified Gram-Schmidt's coefficients from one pass of dot products: h_i = <V_i, w - sum_{k<i} h_k V_k> is the forward
// substitution (I + L) h = s with L_ik = <V_i, V_k>, k < i (the inverse compact form of Swirydowicz, Langou, Ananthan, Yang
// and Thomas, Low synchronization Gram-Schmidt and GMRES algorithms, 2021), so the products with the newest vector are
// formed in the same pass.  One wave, lane i the unknown h_i; block 0 keeps the new row of L.
__device__ __forceinline__ void mgs_coefficients(double *gram, const double *g, int32_t nv, double *c, double *L)
{
    const int32_t j = nv - 1, t = threadIdx.x;
    for (int32_t q = t; q < 64 * j; q += kOrthoThreads)
    {
        const int32_t i = q >> 6, k = q & 63;
        if (k < i) L[65 * i + k] = gram[64 * i + k];
    }
    if (t < j)
    {
        L[65 * j + t] = g[t];
        if (blockIdx.x == 0) gram[64 * j + t] = g[t];
    }
    __syncthreads();
    if (t < 64)
    {
        double s = t < nv ? c[t] : 0.0;
        for (int32_t k = 0; k < j; ++k)
        {
            const double hk = __shfl(s, k, 64);
            if (t > k && t < nv) s -= L[65 * t + k] * hk;
        }
        if (t < nv) c[t] = s;
    }
    __syncthreads();
}

template <class T, int MODE>
__global__ void __launch_bounds__(kOrthoThreads) k_update(Ortho<T> o, int32_t fold, double dgks)
{
    constexpr int P = Pack<T>::N;
    __shared__ double c[64], sh[4];
    __shared__ double g[MODE == kMgs ? 64 : 1], L[MODE == kMgs ? 64 * 65 : 1];
    __shared__ const T *vp[64];
    const int32_t nv = o.nv, t = threadIdx.x;
    if (t < nv) vp[t] = o.V[t];
    load_cols<MODE == kMgs>(o.part, o.cols, fold, nv, c, g);
    if (MODE == kMgs) mgs_coefficients(o.gram, g, nv, c, L);
    bool direct = false;
    double inv = 1.0;
    if (MODE == kCgs)
    {
        double ss = 0.0;
        for (int32_t i = 0; i < nv; ++i) ss += c[i] * c[i];
        const double ww = c[kColWW], hn2 = ww - ss, hp = hn2 > 0 ? sqrt(hn2) : 0.0;
        direct = hp >= dgks * sqrt(ww > 0 ? ww : 0.0) && hp > 1e-300;
        if (direct) inv = 1.0 / hp;
        if (blockIdx.x == gridDim.x - 1)
        {
            // a block of its own: the host has the step's coefficients while the vectors are still being written
            __syncthreads();
            if (t == 0) { c[nv] = hp; c[62] = direct ? 0.0 : 1.0; }
            __syncthreads();
            publish(o.box, o.ticket, c, 64);
            return;
        }
    }
    else if (blockIdx.x == 0 && t < nv) o.h[t] = c[t]; // for ortho_scale (cols is still being read by other blocks)
    double acc = 0.0;
    const int32_t np = o.n / P;
    // backwards: the dot products' last reads first
    const int32_t nb = int32_t(gridDim.x) - (MODE == kCgs ? 1 : 0), stride = nb * kOrthoThreads, first = int32_t(blockIdx.x) * kOrthoThreads + t;
    for (int32_t p = first; p < np; p += stride)
    {
        const int32_t q = np - 1 - p;
        const auto a = ldg<T>(o.w, q);
        double x[P];
#pragma unroll
        for (int m = 0; m < P; ++m) x[m] = a[m];
        axpy_all<T>(vp, c, nv, q, x);
        typename Pack<T>::Raw r;
        if (MODE == kCgs && direct)
        {
#pragma unroll
            for (int m = 0; m < P; ++m) r[m] = T(x[m] * inv);
            reinterpret_cast<typename Pack<T>::Raw *>(o.vnext)[q] = r;
            if (o.pv)
            {
                const auto iv = ldg<T>(o.invdiag, q);
                typename Pack<T>::Raw z;
#pragma unroll
                for (int m = 0; m < P; ++m) z[m] = o.dir[P * q + m] ? T(0) : r[m] * iv[m];
                reinterpret_cast<typename Pack<T>::Raw *>(o.pv)[q] = z;
            }
        }
        else
        {
#pragma unroll
            for (int m = 0; m < P; ++m) { r[m] = T(x[m]); acc += double(r[m]) * double(r[m]); }
            reinterpret_cast<typename Pack<T>::Raw *>(MODE == kCgs ? o.w : o.vnext)[q] = r;
        }
    }
    if (blockIdx.x == 0 && t < o.n - P * np)
    {
        const int32_t e = P * np + t;
        double x = o.w[e];
        for (int32_t i = 0; i < nv; ++i) x -= c[i] * double(vp[i][e]);
        if (MODE == kCgs && direct)
        {
            const T v = T(x * inv);
            o.vnext[e] = v;
            if (o.pv) o.pv[e] = o.dir[e] ? T(0) : v * o.invdiag[e];
        }
        else
        {
            const T r = T(x);
            acc += double(r) * double(r);
            (MODE == kCgs ? o.w : o.vnext)[e] = r;
        }
    }
    if (MODE == kCgs) return;
    const double s = block_total(acc, sh);
    if (t == 0) o.norms[blockIdx.x] = s;
}

// Blocks of kScalePacks packs per thread, loaded ahead of the norm's reduction; the last block hands over
constexpr int kScalePacks = 4;
template <class T> __global__ void __launch_bounds__(kOrthoThreads) k_scale(Ortho<T> o, int32_t nblocks)
{
    constexpr int P = Pack<T>::N;
    __shared__ double sh[4], c[64];
    const int32_t t = threadIdx.x, np = o.n / P, q0 = int32_t(blockIdx.x) * kOrthoThreads * kScalePacks + t;
    const bool last = blockIdx.x == gridDim.x - 1;
    typename Pack<T>::Raw a[kScalePacks];
    if (!last)
#pragma unroll
        for (int u = 0; u < kScalePacks; ++u)
            if (q0 + u * kOrthoThreads < np) a[u] = ldg<T>(o.vnext, q0 + u * kOrthoThreads);
    double s = 0.0;
    for (int32_t i = t; i < nblocks; i += kOrthoThreads) s += o.norms[i];
    const double hn = sqrt(block_total(s, sh));
    auto put = [&](int32_t e, T v) {
        if (o.pv) o.pv[e] = o.dir[e] ? T(0) : v * o.invdiag[e];
        return v;
    };
    const bool keep = hn > 1e-300;
    if (last)
    {
        if (t < 64) c[t] = t < o.nv ? o.h[t] : t == o.nv ? hn : 0.0;
        __syncthreads();
        publish(o.box, o.ticket, c, 64);
        if (keep && t < o.n - P * np) o.vnext[P * np + t] = put(P * np + t, T(double(o.vnext[P * np + t]) / hn));
        return;
    }
    if (!keep) return;
#pragma unroll
    for (int u = 0; u < kScalePacks; ++u)
    {
        const int32_t q = q0 + u * kOrthoThreads;
        if (q >= np) break;
#pragma unroll
        for (int m = 0; m < P; ++m) a[u][m] = put(P * q + m, T(double(a[u][m]) / hn));
        reinterpret_cast<typename Pack<T>::Raw *>(o.vnext)[q] = a[u];
    }
}

// one pack of edges per thread (the grid covers n / N + 1 threads), the sum in order of i
template <class T>
__global__ void __launch_bounds__(kOrthoThreads) k_solution(const T *const *V, Coefs y, int32_t j, const T *invdiag, const int8_t *dir, int32_t n,
                                                            const double *x0, double *delta, double *x)
{
    constexpr int P = Pack<T>::N;
    __shared__ double ny[64];
    __shared__ const T *vp[64];
    if (int32_t(threadIdx.x) < j) { ny[threadIdx.x] = -y.v[threadIdx.x]; vp[threadIdx.x] = V[threadIdx.x]; }
    __syncthreads();
    const int32_t q = int32_t(blockIdx.x) * kOrthoThreads + int32_t(threadIdx.x), np = n / P;
    auto put = [&](int32_t e, double s, T iv) {
        double dl = delta[e];
        if (!dir[e])
        {
            dl += s * double(iv);
            delta[e] = dl;
        }
        x[e] = x0[e] + dl;
    };
    if (q < np)
    {
        double s[P] = {}; // s - (-y_i) v is s + y_i v exactly
        axpy_all<T>(vp, ny, j, q, s);
        const auto iv = ldg<T>(invdiag, q);
#pragma unroll
        for (int m = 0; m < P; ++m) put(P * q + m, s[m], iv[m]);
    }
    else if (q == np)
        for (int32_t e = P * np; e < n; ++e)
        {
            double s = 0.0;
            for (int32_t i = 0; i < j; ++i) s -= ny[i] * double(vp[i][e]);
            put(e, s, invdiag[e]);
        }
}

__global__ void __launch_bounds__(kOrthoThreads) k_norms2(const double *a, const double *b, int32_t n, double *part)
{
    __shared__ double sh[4];
    double sa = 0.0, sb = 0.0;
    const int32_t np = n / 2;
    for (int32_t q = int32_t(blockIdx.x) * kOrthoThreads + int32_t(threadIdx.x); q < np; q += int32_t(gridDim.x) * kOrthoThreads)
    {
        const auto x = ldg<double>(a, q);
        sa += dot_pack<double>(x, x);
        if (b)
        {
            const auto y = ldg<double>(b, q);
            sb += dot_pack<double>(y, y);
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && (n & 1))
    {
        sa += a[n - 1] * a[n - 1];
        if (b) sb += b[n - 1] * b[n - 1];
    }
    sa = block_total(sa, sh);
    sb = block_total(sb, sh);
    if (threadIdx.x == 0) { part[blockIdx.x] = sa; part[kOrthoBlocks + blockIdx.x] = sb; }
}
__global__ void __launch_bounds__(kOrthoThreads) k_norms2_final(const double *part, int32_t nblocks, double *out, HostBox *box, uint64_t ticket)
{
    __shared__ double sh[4], c[2];
    for (int k = 0; k < 2; ++k)
    {
        double s = 0.0;
        for (int32_t i = threadIdx.x; i < nblocks; i += kOrthoThreads) s += part[k * kOrthoBlocks + i];
        s = block_total(s, sh);
        if (threadIdx.x == 0) { c[k] = s; out[k] = sqrt(s); }
    }
    __syncthreads();
    publish(box, ticket, c, 2);
}

template <class T, bool GRAM> using DotsFn = void (*)(const T *const *, int32_t, const T *, const T *, int32_t, int32_t, double *);
template <class T, bool GRAM, int... I> constexpr std::array<DotsFn<T, GRAM>, sizeof...(I) + 1> dots_table(std::integer_sequence<int, I...>)
{
    return {nullptr, &k_dots<T, I + 1, GRAM>...};
}
// [nv]: the pass over nv basis vectors, 1 <= nv <= kDotChunk
template <class T, bool GRAM> const std::array<DotsFn<T, GRAM>, kDotChunk + 1> kDots = dots_table<T, GRAM>(std::make_integer_sequence<int, kDotChunk>{});
} // namespace

template <class T> void ortho_dots(const Ortho<T> &o, bool gram, hipStream_t s)
{
    const int nb = ortho_blocks(o.n, Pack<T>::N);
    for (int32_t i0 = 0; i0 < o.nv; i0 += kDotChunk)
    {
        const int nv = o.nv - i0 < kDotChunk ? o.nv - i0 : kDotChunk;
        auto f = kDots<T, false>[nv];
        if constexpr (sizeof(T) == 8)
            if (gram) f = kDots<T, true>[nv];
        hipLaunchKernelGGL(f, dim3(nb), dim3(kOrthoThreads), 0, s, o.V, i0, static_cast<const T *>(o.w), o.vj, o.n,
                           i0 == 0 ? 1 : 0, o.part);
    }
    if (nb > kFoldBlocks)
        hipLaunchKernelGGL(k_cols_final, dim3(o.nv + 1 + (gram ? o.nv : 0)), dim3(kOrthoThreads), 0, s, static_cast<const double *>(o.part), nb, o.nv,
                           o.cols);
}
template <class T> void ortho_update(const Ortho<T> &o, int mode, double dgks, hipStream_t s)
{
    const int nb = ortho_blocks(o.n, Pack<T>::N), fold = nb > kFoldBlocks ? 0 : nb;
    if (mode == kCgs) hipLaunchKernelGGL((k_update<T, kCgs>), dim3(nb + 1), dim3(kOrthoThreads), 0, s, o, fold, dgks);
    else if (mode == kPlain) hipLaunchKernelGGL((k_update<T, kPlain>), dim3(nb), dim3(kOrthoThreads), 0, s, o, fold, dgks);
    else if constexpr (sizeof(T) == 8) hipLaunchKernelGGL((k_update<T, kMgs>), dim3(nb), dim3(kOrthoThreads), 0, s, o, fold, dgks);
}
template <class T> void ortho_scale(const Ortho<T> &o, hipStream_t s)
{
    const int nb = ortho_blocks(o.n, Pack<T>::N);
    hipLaunchKernelGGL(k_scale<T>, dim3((o.n / Pack<T>::N + kOrthoThreads * kScalePacks - 1) / (kOrthoThreads * kScalePacks) + 1), dim3(kOrthoThreads), 0,
                       s, o, nb);
}
template void ortho_dots<float>(const Ortho<float> &, bool, hipStream_t);
template void ortho_dots<double>(const Ortho<double> &, bool, hipStream_t);
template void ortho_update<float>(const Ortho<float> &, int, double, hipStream_t);
template void ortho_update<double>(const Ortho<double> &, int, double, hipStream_t);
template void ortho_scale<float>(const Ortho<float> &, hipStream_t);
template void ortho_scale<double>(const Ortho<double> &, hipStream_t);

template <class T>
void solution_update(const T *const *V, const Coefs &y, int32_t j, const T *invdiag, const int8_t *dir, int32_t n, const double *x0,
                     double *delta, double *x, hipStream_t s)
{
    hipLaunchKernelGGL(k_solution<T>, dim3(n / Pack<T>::N / kOrthoThreads + 1), dim3(kOrthoThreads), 0, s, V, y, j, invdiag, dir, n, x0, delta, x);
}
template void solution_update<float>(const float *const *, const Coefs &, int32_t, const float *, const int8_t *, int32_t, const double *, double *,
                                     double *, hipStream_t);
template void solution_update<double>(const double *const *, const Coefs &, int32_t, const double *, const int8_t *, int32_t, const double *,
                                      double *, double *, hipStream_t);

void norms2(const double *a, const double *b, int32_t n, double *part, double *out, HostBox *box, uint64_t ticket, hipStream_t s)
{
    const int nb = ortho_blocks(n, 2);
    hipLaunchKernelGGL(k_norms2, dim3(nb), dim3(kOrthoThreads), 0, s, a, b, n, part);
    hipLaunchKernelGGL(k_norms2_final, dim3(1), dim3(kOrthoThreads), 0, s, static_cast<const double *>(part), nb, out, box, ticket);
}
} // namespace mhdg
