// One launch for the first two of the four of a product with the induction operator (ImplicitInduction.cpp:139-182).  Four
// lanes per cell stage the cell's edge values in LDS, each lane forms the fluxes of its faces from them (a face's two
// cells form it twice; one writes it for the edge kernel) and its part of the cell's field.
//
// It serves meshes whose tables stay in the caches (DevMesh::xcd_ranges: up to 457k tetrahedra with two ions), where a launch
// and its gap cost more than the faces' fluxes do, and the tables (40 bytes a tetrahedron) are not read from HBM.
//
// Hall steps, microseconds in FP64 / mixed precision, without and with it, forced either way: 9.5k tetrahedra 329 / 282 and
// 298 / 263, 60k 445 / 375 and 422 / 357, 150k 653 / 589 and 641 / 577, 290k 1066 / 911 and 1028 / 897, 435k 1552 / 1269 and 1502 /
// 1261; above the line 484k 1809 / 1422 and 1812 / 1411, 683k 2616 / 1919 and 2603 / 1934, 1.06M 4564 / 3272 and 4574 / 3354 (per
// product, FP64 at 1.95M 94 us both; FP32 at 7.83M 191 us against 245), so the tables are built below it only.
#include <stdexcept>
#include <string>

#include "ctx.h"
#include "flux_cell.h"

namespace mhdg
{
namespace
{
template <int DEG> struct Shape; // edges per face and per cell, and the LDS row of a cell (odd: no bank conflicts)
template <> struct Shape<4> { static constexpr int face = 3, cell = 6, row = 7; };
template <> struct Shape<6> { static constexpr int face = 4, cell = 12, row = 13; };
constexpr int kLanes = 4;

// The flux of (cell, face) entry code from the cell's staged edge values
template <int DEG, class T> __device__ __forceinline__ T face_flux(const T *x, uint32_t code)
{
    T s = 0;
#pragma unroll
    for (int q = 0; q < Shape<DEG>::face; ++q)
    {
        const T e = x[code >> (4 * q) & 15];
        s += (code >> (16 + q) & 1) ? -e : e;
    }
    return s;
}
} // namespace

template <int DEG> __global__ void __launch_bounds__(256) k_cell_edges(DevMesh d, int32_t *edge, uint32_t *face, int32_t *counts)
{
    const int32_t c = gid();
    if (c >= d.nc) return;
    constexpr int NE = Shape<DEG>::cell;
    int32_t id[NE], n = 0, owned = 0;
    for (int i = 0; i < DEG; ++i)
    {
        const int32_t k = DEG * c + i, f = pid(d.c2f[k]), l = d.fL[f], r = d.fR[f];
        uint32_t code = 0;
        for (int q = 0; q < Shape<DEG>::face; ++q)
        {
            const int32_t v = d.f2e[Shape<DEG>::face * f + q], e = pid(v);
            int32_t at = 0;
            while (at < n && id[at] != e) ++at;
            if (at == n)
            {
                if (n == NE)
                {
                    atomicAdd(counts, 1);
                    return;
                }
                id[n++] = e;
            }
            code |= uint32_t(at) << (4 * q) | (v < 0 ? 1u << (16 + q) : 0u);
        }
        bool own = c == (l >= 0 ? l : r);
        for (int j = 0; j < i; ++j) own = own && pid(d.c2f[DEG * c + j]) != f; // a face of the cell twice
        if (own) { code |= kOwnFace; ++owned; }
        face[k] = code;
    }
    for (int i = 0; i < NE; ++i) edge[NE * c + i] = id[i < n ? i : 0];
    atomicAdd(counts + 1, owned);
}

template <int DEG>
__global__ void __launch_bounds__(256) k_flux_cell(DevMesh d, CellEdges t, const double *v, const double *invdiag, const int8_t *dir, double *phi,
                                                   double *b)
{
    constexpr int NE = Shape<DEG>::cell, EL = (NE + kLanes - 1) / kLanes, FL = (DEG + kLanes - 1) / kLanes;
    __shared__ double xs[256 / kLanes * Shape<DEG>::row];
    const int32_t i = gid(d), c = i / kLanes, lane = i % kLanes;
    const bool ok = c < d.nc;
    double *x = xs + Shape<DEG>::row * (int32_t(threadIdx.x) / kLanes);
    uint32_t code[FL];
    int32_t f[FL];
    if (ok)
    {
        int32_t e[EL];
#pragma unroll
        for (int u = 0; u < EL; ++u)
            if (lane + kLanes * u < NE) e[u] = t.edge[NE * c + lane + kLanes * u];
#pragma unroll
        for (int u = 0; u < FL; ++u)
            if (lane + kLanes * u < DEG) { code[u] = t.face[DEG * c + lane + kLanes * u]; f[u] = pid(d.c2f[DEG * c + lane + kLanes * u]); }
#pragma unroll
        for (int u = 0; u < EL; ++u)
            if (lane + kLanes * u < NE)
            {
                double q = v[e[u]];
                if (invdiag)
                {
                    const double iv = invdiag[e[u]];
                    q = dir[e[u]] ? 0.0 : q * iv;
                }
                x[lane + kLanes * u] = q;
            }
    }
    __syncthreads();
    double bx = 0.0, by = 0.0, bz = 0.0;
#pragma unroll
    for (int u = 0; u < FL; ++u)
    {
        const int32_t n = lane + kLanes * u;
        double px = 0.0, py = 0.0, pz = 0.0;
        if (ok && n < DEG)
        {
            const double s = face_flux<DEG>(x, code[u]), *r = d.recon + 3 * (size_t(DEG) * size_t(c) + n);
            if (code[u] & kOwnFace) phi[f[u]] = s;
            px = r[0] * s; py = r[1] * s; pz = r[2] * s;
        }
#pragma unroll
        for (int q = 0; q < kLanes; ++q)
        {
            const double qx = __shfl(px, q, kLanes), qy = __shfl(py, q, kLanes), qz = __shfl(pz, q, kLanes);
            if (kLanes * u + q < DEG) { bx += qx; by += qy; bz += qz; }
        }
    }
    if (ok && lane == 0) { b[3 * size_t(c)] = bx; b[3 * size_t(c) + 1] = by; b[3 * size_t(c) + 2] = bz; }
}

template <int DEG>
__global__ void __launch_bounds__(256) k_flux_cell_f32(DevMesh d, CellEdges t, const float *recon, const float *pv, float *phi, float *b)
{
    constexpr int NE = Shape<DEG>::cell, EL = (NE + kLanes - 1) / kLanes, FL = (DEG + kLanes - 1) / kLanes;
    __shared__ float xs[256 / kLanes * Shape<DEG>::row];
    const int32_t i = gid(d), c = i / kLanes, lane = i % kLanes;
    const bool ok = c < d.nc;
    float *x = xs + Shape<DEG>::row * (int32_t(threadIdx.x) / kLanes);
    uint32_t code[FL];
    int32_t f[FL];
    if (ok)
    {
        int32_t e[EL];
#pragma unroll
        for (int u = 0; u < EL; ++u)
            if (lane + kLanes * u < NE) e[u] = t.edge[NE * c + lane + kLanes * u];
#pragma unroll
        for (int u = 0; u < FL; ++u)
            if (lane + kLanes * u < DEG) { code[u] = t.face[DEG * c + lane + kLanes * u]; f[u] = pid(d.c2f[DEG * c + lane + kLanes * u]); }
#pragma unroll
        for (int u = 0; u < EL; ++u)
            if (lane + kLanes * u < NE) x[lane + kLanes * u] = pv[e[u]];
    }
    __syncthreads();
    float bx = 0.0f, by = 0.0f, bz = 0.0f;
#pragma unroll
    for (int u = 0; u < FL; ++u)
    {
        const int32_t n = lane + kLanes * u;
        if (ok && n < DEG)
        {
            const float s = face_flux<DEG>(x, code[u]), *r = recon + 3 * (size_t(DEG) * size_t(c) + n);
            if (code[u] & kOwnFace) phi[f[u]] = s;
            bx += r[0] * s; by += r[1] * s; bz += r[2] * s;
        }
    }
    for (int o = kLanes / 2; o > 0; o >>= 1)
    {
        bx += __shfl_xor(bx, o, kLanes); by += __shfl_xor(by, o, kLanes); bz += __shfl_xor(bz, o, kLanes);
    }
    if (ok && lane == 0) { b[3 * size_t(c)] = bx; b[3 * size_t(c) + 1] = by; b[3 * size_t(c) + 2] = bz; }
}
} // namespace mhdg

using namespace mhdg;

namespace
{
inline int blocks(int64_t n) { return static_cast<int>((n + 255) / 256); }
} // namespace

#define LAUNCH(NAME, ...)                                                                                                    \
    do                                                                                                                       \
    {                                                                                                                        \
        prof_begin(NAME);                                                                                                    \
        hipLaunchKernelGGL(__VA_ARGS__);                                                                                     \
        prof_end();                                                                                                          \
    } while (0)

void mhdg_ctx::flux_cell_build()
{
    const bool tets = cdeg == 4 && fdeg == 3, hexes = cdeg == 6 && fdeg == 4;
    if (!(d.xcd_ranges && (tets || hexes) && (op_hall || ideal_cfg)) || nc == 0) return;
    int32_t *edge = static_cast<int32_t *>(alloc(sizeof(int32_t) * size_t(tets ? 6 : 12) * size_t(nc)));
    uint32_t *face = static_cast<uint32_t *>(alloc(sizeof(uint32_t) * c2f_nnz));
    int32_t *counts = static_cast<int32_t *>(alloc(2 * sizeof(int32_t)));
    if (hipMemsetAsync(counts, 0, 2 * sizeof(int32_t), stream) != hipSuccess) throw std::runtime_error("memset: cell edges");
    hipLaunchKernelGGL(tets ? k_cell_edges<4> : k_cell_edges<6>, dim3(blocks(nc)), dim3(256), 0, stream, d, edge, face, counts);
    check_launch("cell edges");
    int32_t h[2];
    d2h(h, counts, sizeof(h));
    // a cell with more edges than its shape has, or a face without a cell: the separate kernels
    if (h[0] == 0 && h[1] == nf) { ce.edge = edge; ce.face = face; }
}

bool mhdg_ctx::flux_cell(const double *v, const double *inv, const int8_t *dir, double *phi, double *b)
{
    if (!ce.edge) return false;
    LAUNCH("flux_cell", cdeg == 4 ? k_flux_cell<4> : k_flux_cell<6>, dim3(blocks(int64_t(kLanes) * nc)), dim3(256), 0, stream, d, ce, v, inv, dir,
           phi, b);
    return true;
}

bool mhdg_ctx::flux_cell(const float *pv, float *phi, float *b)
{
    if (!ce.edge) return false;
    LAUNCH("flux_cell_f32", cdeg == 4 ? k_flux_cell_f32<4> : k_flux_cell_f32<6>, dim3(blocks(int64_t(kLanes) * nc)), dim3(256), 0, stream, d, ce,
           mixed->s.recon, pv, phi, b);
    return true;
}
