#pragma once
// Device helpers of the resident step's cell and face rows, shared by its kernels and their transposes.
#include "explicit_step.h"
#include "fv.h"

namespace mhdg
{
namespace
{
__device__ __forceinline__ double2 ld2(const double *p) { return *reinterpret_cast<const double2 *>(p); }
__device__ __forceinline__ V3 geo_normal(const DevMesh &d, int32_t f, double &A)
{
    const double2 p = ld2(d.geo + 4 * size_t(f)), q = ld2(d.geo + 4 * size_t(f) + 2);
    A = q.y;
    return V3(p.x, p.y, q.x);
}
// row of cell c in a (cell, face) table: the fixed length DEG, or the row pointers (DEG 0)
template <int DEG> __device__ __forceinline__ void row_of(const DevMesh &d, int32_t c, int32_t &k0, int32_t &nk)
{
    if (DEG > 0) { k0 = c * DEG; nk = DEG; }
    else { k0 = d.c2f_ptr[c]; nk = d.c2f_ptr[c + 1] - k0; }
}
// the DEG entries of row k0 of a (cell, face) id table
template <int DEG> __device__ __forceinline__ void row_ids(const int32_t *tab, int32_t k0, int32_t (&v)[DEG])
{
    if constexpr (DEG == 4)
    {
        const int4 q = *reinterpret_cast<const int4 *>(tab + k0);
        v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    }
    else
    {
#pragma unroll
        for (int i = 0; i < DEG; i += 2)
        {
            const int2 q = *reinterpret_cast<const int2 *>(tab + k0 + i);
            v[i] = q.x; v[i + 1] = q.y;
        }
    }
}
// Right-hand side of ion s of cell c (record `row`, volume V): owner gather of the fluxes in ascending face order
// (FluxRHS.cpp:71-72), Lorentz and production sources (MercurySources.cpp:20-63)
template <int DEG>
__device__ __forceinline__ void cell_rhs(const DevMesh &d, const Params &P, const StepFields &F, int32_t c, int32_t s, int32_t ns,
                                         const double *row, double V, double dt, double (&rhs)[5])
{
    constexpr int N = DEG > 0 ? DEG : 1;
    for (int m = 0; m < 5; ++m) rhs[m] = 0;
    int32_t k0, nk;
    row_of<DEG>(d, c, k0, nk);
    auto add = [&](int32_t v, const double *fa) {
        if (v >= 0) for (int m = 0; m < 5; ++m) rhs[m] -= fa[m] / V;
        else for (int m = 0; m < 5; ++m) rhs[m] += fa[m] / V;
    };
    if constexpr (DEG > 0)
    {
        int32_t v[N];
        double fa[N][5];
        row_ids<DEG>(d.cfs, k0, v);
#pragma unroll
        for (int i = 0; i < DEG; ++i)
            for (int m = 0; m < 5; ++m) fa[i][m] = F.FA[5 * (size_t(pid(v[i])) * size_t(ns) + s) + m];
#pragma unroll
        for (int i = 0; i < DEG; ++i) add(v[i], fa[i]);
    }
    else
        for (int32_t k = k0; k < k0 + nk; ++k) add(d.cfs[k], F.FA + 5 * (size_t(pid(d.cfs[k])) * size_t(ns) + s));
    const double *W = row + 5 * s;
    double ne = ion_density(P, 0, row[0]);
    for (int q = 1; q < ns; ++q) ne = ne + ion_density(P, q, row[5 * q]);
    const double ws = ion_density(P, s, W[0]) / sqrt(ne * ne + P.ne_floor * P.ne_floor);
    const double rho = mx(W[0], 0.0);
    const V3 vel(W[1], W[2], W[3]);
    V3 S;
    if (P.lorentz) S += (P.inver_MA2 * ws) * cross(L3(F.J, c), L3(F.Btot, c));
    rhs[1] += S.x; rhs[2] += S.y; rhs[3] += S.z;
    rhs[4] += dot(vel, S) + (rho > 1e-30 ? 0.5 * dt * dot(S, S) / rho : 0.0);
    if (P.src_rate[s] != 0.0 && d.atm)
    {
        const double q = P.src_rate[s] * d.atm[c];
        rhs[0] += q;
        rhs[4] += q * P.src_T / (P.gamma - 1.0);
    }
}
} // namespace
} // namespace mhdg
