#pragma once
// Finite-volume device helpers shared by the explicit-stage kernels and their adjoints: cell vector
// reconstruction, CFL time step, face states, Rusanov flux, ghost states, the UCT edge quantities and the
// boundary EMF.  Templates on the real type R (double, or Dual for forward-mode derivatives).
#include "kernels.h"

namespace mhdg
{
namespace
{
constexpr int kGradFast = 4; // cells with up to this many faces keep their face rows in registers (tetrahedra)
// Only the double instantiations do: the Dual (forward-mode) ones would spill the rows to scratch memory
template <class R> constexpr bool kRowsInRegisters = sizeof(R) == sizeof(double);

// src/uns/geometry/Reconstruct.cpp:11-45 for one cell: the face term (c2f entry v, |A|, area vector, flux) and
// the 3x3 solve
template <class R> __device__ __forceinline__ void cell_vector_add(R (&M)[3][3], R (&r)[3], int32_t v, const R &A, const V3 &area, const R &flux)
{
    if (A <= 0) return;
    const V3T<R> n = (psg(v) / A) * area;
    const R nv[3] = {n.x, n.y, n.z};
    const R phi = psg(v) * flux;
    for (int i = 0; i < 3; ++i)
    {
        r[i] += nv[i] * phi;
        for (int j = 0; j < 3; ++j) M[i][j] += A * nv[i] * nv[j];
    }
}
template <class R> __device__ V3T<R> cell_vector_solve(const R (&M)[3][3], const R (&r)[3])
{
    const R det = M[0][0] * (M[1][1] * M[2][2] - M[1][2] * M[2][1]) - M[0][1] * (M[1][0] * M[2][2] - M[1][2] * M[2][0]) +
                       M[0][2] * (M[1][0] * M[2][1] - M[1][1] * M[2][0]);
    const R sc = mx(mx(mx(M[0][0], M[1][1]), M[2][2]), 1e-300);
    if (fabs(det) < 1e-12 * sc * sc * sc) return V3T<R>();
    R I[3][3];
    I[0][0] = (M[1][1] * M[2][2] - M[1][2] * M[2][1]) / det;
    I[0][1] = (M[0][2] * M[2][1] - M[0][1] * M[2][2]) / det;
    I[0][2] = (M[0][1] * M[1][2] - M[0][2] * M[1][1]) / det;
    I[1][0] = (M[1][2] * M[2][0] - M[1][0] * M[2][2]) / det;
    I[1][1] = (M[0][0] * M[2][2] - M[0][2] * M[2][0]) / det;
    I[1][2] = (M[0][2] * M[1][0] - M[0][0] * M[1][2]) / det;
    I[2][0] = (M[1][0] * M[2][1] - M[1][1] * M[2][0]) / det;
    I[2][1] = (M[0][1] * M[2][0] - M[0][0] * M[2][1]) / det;
    I[2][2] = (M[0][0] * M[1][1] - M[0][1] * M[1][0]) / det;
    return {I[0][0] * r[0] + I[0][1] * r[1] + I[0][2] * r[2], I[1][0] * r[0] + I[1][1] * r[1] + I[1][2] * r[2],
            I[2][0] * r[0] + I[2][1] * r[1] + I[2][2] * r[2]};
}
template <class R> __device__ V3T<R> cell_vector(const DevMesh &d, int32_t c, const R *flux)
{
    R M[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, r[3] = {0, 0, 0};
    for (int32_t k = d.c2f_ptr[c]; k < d.c2f_ptr[c + 1]; ++k)
    {
        const int32_t v = d.c2f[k], f = pid(v);
        cell_vector_add(M, r, v, R(d.famag[f]), L3(d.farea, f), flux[f]);
    }
    return cell_vector_solve(M, r);
}

// MercuryUns/fluid/MercurySources.cpp:104-145 for one fluid cell (+inf if no face restricts it)
// (every ion species; the total density of the fast speed summed in species order)
// (the species rows of cell c are read at row `row` of the species arrays Ws: c itself, or 0 for a one-cell copy)
template <class R> __device__ R cell_dt(const DevMesh &d, const Params &P, int32_t c, const R *const *Ws, const V3T<R> &b, size_t row)
{
    R dt = __builtin_inf();
    const R B2 = dot(b, b);
    R rho_sum = Ws[0][5 * row];
    for (int s = 1; s < P.ns; ++s) rho_sum = rho_sum + Ws[s][5 * row];
    const R rho_tot = mx(rho_sum, P.rho_floor_dt);
    const R vA2 = P.inver_MA2 * B2 / rho_tot; // the same for every face and species
    for (int s = 0; s < P.ns; ++s)
    {
        const R *w = Ws[s] + 5 * row;
        const R cs2 = P.gamma * w[4] / mx(w[0], 1e-30);
        R denom = 0;
        for (int32_t k = d.c2f_ptr[c]; k < d.c2f_ptr[c + 1]; ++k)
        {
            const int32_t f = pid(d.c2f[k]);
            const R A = d.famag[f];
            const V3T<R> n = (1.0 / A) * L3(d.farea, f);
            const R vAn2 = P.inver_MA2 * dot(b, n) * dot(b, n) / rho_tot;
            const R term = cs2 + vA2;
            const R cf = sqrt(0.5 * (term + sqrt(mx(0.0, term * term - 4 * cs2 * vAn2))));
            denom += (fabs(w[1] * n.x + w[2] * n.y + w[3] * n.z) + cf) * A;
        }
        if (denom > 0) dt = mn(dt, P.cfl * d.cvol[c] / denom);
    }
    return dt;
}

template <class R> __device__ __forceinline__ R block_min(R v, R *sh)
{
    const int t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1)
    {
        if (t < s) sh[t] = mn(sh[t], sh[t + s]);
        __syncthreads();
    }
    return sh[0];
}

// Common/fluid/FluxRHS.cpp:16-27
template <class R> __device__ __forceinline__ PrimT<R> face_state(const R *W, const R *grad, int32_t c, const V3T<R> &dx)
{
    const R *w = W + 5 * size_t(c);
    const R *g = grad + 15 * size_t(c);
    PrimT<R> r;
    r.rho = w[0] + g[0] * dx.x + g[1] * dx.y + g[2] * dx.z;
    r.u = w[1] + g[3] * dx.x + g[4] * dx.y + g[5] * dx.z;
    r.v = w[2] + g[6] * dx.x + g[7] * dx.y + g[8] * dx.z;
    r.w = w[3] + g[9] * dx.x + g[10] * dx.y + g[11] * dx.z;
    r.p = w[4] + g[12] * dx.x + g[13] * dx.y + g[14] * dx.z;
    if (r.rho > 0 && r.p > 0) return r;
    return PrimT<R>{w[0], w[1], w[2], w[3], w[4]};
}

// Common/physics/Euler.h:29-49
template <class R> __device__ void rusanov(const PrimT<R> &L, const PrimT<R> &Rt, const R n[3], double gamma, R *F)
{
    R UL[5], UR[5], FL[5], FR[5];
    to_cons(L, gamma, UL);
    to_cons(Rt, gamma, UR);
    const R unL = L.u * n[0] + L.v * n[1] + L.w * n[2];
    FL[0] = L.rho * unL; FL[1] = L.rho * unL * L.u + L.p * n[0]; FL[2] = L.rho * unL * L.v + L.p * n[1];
    FL[3] = L.rho * unL * L.w + L.p * n[2]; FL[4] = unL * (UL[4] + L.p);
    const R unR = Rt.u * n[0] + Rt.v * n[1] + Rt.w * n[2];
    FR[0] = Rt.rho * unR; FR[1] = Rt.rho * unR * Rt.u + Rt.p * n[0]; FR[2] = Rt.rho * unR * Rt.v + Rt.p * n[1];
    FR[3] = Rt.rho * unR * Rt.w + Rt.p * n[2]; FR[4] = unR * (UR[4] + Rt.p);
    const R sL = fabs(L.u * n[0] + L.v * n[1] + L.w * n[2]) + sqrt(gamma * L.p / L.rho);
    const R sR = fabs(Rt.u * n[0] + Rt.v * n[1] + Rt.w * n[2]) + sqrt(gamma * Rt.p / Rt.rho);
    const R s = mx(sL, sR);
    for (int m = 0; m < 5; ++m) F[m] = 0.5 * (FL[m] + FR[m]) - 0.5 * s * (UR[m] - UL[m]);
}

// Stencil neighbour state of a boundary entry (nb < 0, face f = -(nb + 1), c2f entry v): the ghost table row, or
// ghost_state (Common/fluid/Reconstruction.cpp:9-24) with the cell value wc inside.
template <class R>
__device__ __forceinline__ void stencil_ghost(const DevMesh &d, int32_t sp, const R *gh, const R *wc, const R *fs, int32_t v, int32_t nb,
                                              R *wn)
{
    const int32_t f = -(nb + 1);
    if (gh)
    {
        for (int m = 0; m < 5; ++m) wn[m] = gh[5 * size_t(f) + m];
        return;
    }
    const int8_t kind = d.kind[f];
    for (int m = 0; m < 5; ++m) wn[m] = wc[m];
    if (kind == kWall)
    {
        if (sp == 1) { wn[0] = 1e-12; wn[1] = 0; wn[2] = 0; wn[3] = 0; wn[4] = 1e-12; }
        else
        {
            const V3T<R> n = (psg(v) / d.famag[f]) * L3(d.farea, f);
            const R un = wc[1] * n.x + wc[2] * n.y + wc[3] * n.z;
            wn[1] -= 2 * un * n.x; wn[2] -= 2 * un * n.y; wn[3] -= 2 * un * n.z;
        }
    }
    else if (kind == kInflow)
        for (int m = 0; m < 5; ++m) wn[m] = fs[m];
}

// ghost_state (Common/fluid/Reconstruction.cpp:9-24)
template <class R> __device__ __forceinline__ PrimT<R> ghost_state(int8_t kind, int species, const PrimT<R> &in, const V3T<R> &n, const R *fs)
{
    if (kind == kWall)
    {
        if (species == 1) return PrimT<R>{1e-12, 0, 0, 0, 1e-12};
        const R un = in.u * n.x + in.v * n.y + in.w * n.z;
        PrimT<R> g = in;
        g.u -= 2 * un * n.x; g.v -= 2 * un * n.y; g.w -= 2 * un * n.z;
        return g;
    }
    if (kind == kInflow) return PrimT<R>{fs[0], fs[1], fs[2], fs[3], fs[4]};
    return in;
}

// The per-face quantities of the UCT edge sum (IdealEMF.cpp:79-88)
__device__ __forceinline__ void face_dirs(const DevMesh &d, int32_t f, int32_t e, const V3 &th, V3 &m, V3 &nrm)
{
    V3 v = L3(d.fcen, f) - L3(d.emid, e);
    v -= dot(v, th) * th;
    const double nv = norm(v);
    m = nv > 0 ? (1.0 / nv) * v : V3();
    const double *g = d.geo + 4 * size_t(f);
    nrm = V3(g[0], g[1], g[2]);
}
template <class R> __device__ __forceinline__ R edge_amax(const DevMesh &d, const R *u_cell, int32_t c0, int32_t c1, const V3T<R> &m)
{
    R a = 0.0;
    for (int32_t k = c0; k < c1; ++k) a = mx(a, fabs(dot(L3(u_cell, d.ec_cell[k]), m)));
    return a;
}
__device__ __forceinline__ void plane_basis(const V3 &t, V3 &e1, V3 &e2)
{
    const V3 a = fabs(t.x) < 0.9 ? V3(1, 0, 0) : V3(0, 1, 0);
    e1 = cross(t, a);
    e1 *= 1.0 / norm(e1);
    e2 = cross(t, e1);
}
// eps-regularised 2x2 solve of the omega correction (IdealEMF.cpp:110-118)
template <class R> __device__ __forceinline__ void uct_solve(R M11, R M12, R M22, R g1, R g2, R &l1, R &l2)
{
    const R tr = M11 + M22;
    const R eps = 1e-14 * tr;
    const R det = (M11 + eps) * (M22 + eps) - M12 * M12;
    l1 = 0;
    l2 = 0;
    if (tr > 0 && det > 0)
    {
        l1 = ((M22 + eps) * g1 - M12 * g2) / det;
        l2 = ((M11 + eps) * g2 - M12 * g1) / det;
    }
}
constexpr int kEmfFast = 6; // valence served from registers by k_edge_emf
// boundary EMF of Solver::rhs (MercuryUns/driver/Solver.cpp:162-167)
template <class R> __device__ __forceinline__ R edge_bc(const DevMesh &d, const Params &P, int32_t e, R v)
{
    const int8_t mode = d.emode[e];
    if (mode == 1) return 0.0;
    if (mode == 2)
        return dot(V3T<R>(seeded<R>(P.E_inf[0], P.dE_inf[0]), seeded<R>(P.E_inf[1], P.dE_inf[1]), seeded<R>(P.E_inf[2], P.dE_inf[2])),
                   L3(d.evec, e));
    return v;
}
} // namespace
namespace
{
template <class R> __device__ __forceinline__ V3T<R> emf_of(const R *Ef, int32_t f)
{
    const R *q = Ef + 4 * size_t(f);
    return V3T<R>(q[0], q[1], q[2]);
}

// One high-valence edge per block (pole axes of a lat-lon net): per-face terms in parallel, every sum sequential in the
// reference's order.  sh holds kEmfHeavyRows rows of hv values (hv the largest valence of the mesh).
template <class R>
__device__ __forceinline__ void edge_emf_heavy(const DevMesh &d, const Params &P, const R *Ef, const R *u_cell, double cuct, int32_t e,
                                               const R *E_in, R *E_out, int32_t apply_bc, R *sh, int32_t hv)
{
    constexpr int kHS = kHeavyShared<R>();
    R *s_w = sh, *s_ec = sh + hv, *s_qa = sh + 2 * hv, *s_qb = sh + 3 * hv, *s_sig = sh + 4 * hv, *s_aef = sh + 5 * hv;
    __shared__ R s_l[3];
    const int32_t f0 = d.e2f_ptr[e], f1 = d.e2f_ptr[e + 1], nf = f1 - f0;
    const int32_t c0 = d.ec_ptr[e], c1 = d.ec_ptr[e + 1];
    bool any_fluid = false;
    for (int32_t k = c0; k < c1 && !any_fluid; ++k) any_fluid = d.mat[d.ec_cell[k]] == 0;
    const bool active = nf > 0 && d.elen[e] > 0 && any_fluid;
    const V3 t = L3(d.evec, e);
    const double L = d.elen[e];
    const V3 th = (1.0 / L) * t;
    V3 e1, e2;
    plane_basis(th, e1, e2);
    // The edge's cell velocities are staged in LDS (in s_qa, s_qb, s_sig, before those take the per-face terms):
    // every face's max over the cells then reads LDS, where a dependent global gather per (face, cell) pair made
    // this kernel latency-bound (n_lon^2 pairs per pole-axis edge).  Same values, same order.
    const int32_t nc = c1 - c0;
    const bool staged = active && nc <= hv;
    if (staged)
        for (int32_t k = threadIdx.x; k < nc; k += blockDim.x)
        {
            const V3T<R> u = L3(u_cell, d.ec_cell[c0 + k]);
            s_qa[k] = u.x; s_qb[k] = u.y; s_sig[k] = u.z;
        }
    __syncthreads();
    constexpr int kPer = (kHS + 255) / 256; // faces per thread (nf <= kHS, 256 threads)
    R qa_r[kPer], qb_r[kPer], sig_r[kPer];
    if (active)
#pragma unroll
        for (int j = 0; j < kPer; ++j)
        {
            const int32_t i = int32_t(threadIdx.x) + j * int32_t(blockDim.x);
            if (i >= nf) break;
            const int32_t f = pid(d.e2f[f0 + i]);
            s_w[i] = d.efw[f0 + i];
            s_ec[i] = dot(emf_of(Ef, f), t);
            V3 m, nrm;
            face_dirs(d, f, e, th, m, nrm);
            R aef = 0.0;
            if (staged)
                for (int32_t k = 0; k < nc; ++k) aef = mx(aef, fabs(dot(V3T<R>(s_qa[k], s_qb[k], s_sig[k]), m)));
            else
                aef = edge_amax(d, u_cell, c0, c1, m);
            const R sig = dot(th, cross(m, nrm));
            const V3T<R> qv = (aef * sig) * nrm;
            qa_r[j] = dot(qv, e1);
            qb_r[j] = dot(qv, e2);
            sig_r[j] = sig;
            s_aef[i] = aef;
        }
    __syncthreads(); // every read of the staged velocities is done
    if (active)
#pragma unroll
        for (int j = 0; j < kPer; ++j)
        {
            const int32_t i = int32_t(threadIdx.x) + j * int32_t(blockDim.x);
            if (i >= nf) break;
            s_qa[i] = qa_r[j]; s_qb[i] = qb_r[j]; s_sig[i] = sig_r[j];
        }
    __syncthreads();
    // the sequential sums side by side: M11, M12, M22, g1, g2 and Ec on a wave each would be idle most of the time, so
    // the first lanes of one wave take one sum each
    __shared__ R s_sum[6];
    if (threadIdx.x < 6 && active)
    {
        const int32_t w = threadIdx.x;
        const R *x = w == 5 ? s_ec : w == 2 || w == 4 ? s_qb : s_qa;
        const R *y = w == 0 ? s_qa : s_qb;
        R acc = 0;
        if (w < 3)
            for (int32_t i = 0; i < nf; ++i) acc += s_w[i] * x[i] * y[i];
        else
            for (int32_t i = 0; i < nf; ++i) acc += s_w[i] * x[i];
        s_sum[w] = acc;
    }
    __syncthreads();
    if (threadIdx.x == 0 && active)
    {
        R l1, l2;
        uct_solve(s_sum[0], s_sum[1], s_sum[2], s_sum[3], s_sum[4], l1, l2);
        s_l[0] = l1; s_l[1] = l2;
    }
    __syncthreads();
    if (active)
        for (int32_t i = threadIdx.x; i < nf; i += blockDim.x)
        {
            const int32_t f = pid(d.e2f[f0 + i]);
            const R omega = s_w[i] * (1.0 - (s_qa[i] * s_l[0] + s_qb[i] * s_l[1]));
            s_ec[i] = omega * s_aef[i] * s_sig[i] * Ef[4 * size_t(f) + 3];
        }
    __syncthreads();
    if (threadIdx.x == 0)
    {
        R out = E_in ? E_in[e] : 0.0;
        if (active)
        {
            R Eu = 0;
            for (int32_t i = 0; i < nf; ++i) Eu += s_ec[i];
            out += s_sum[5] + 2.0 * cuct * L * Eu;
        }
        E_out[e] = apply_bc ? edge_bc(d, P, e, out) : out;
    }
}

// B -= dt d1 E of one face (Common/induction/Faraday.cpp:15-36), or with a per-edge step dte B -= d1 (dte E)
template <class R>
__device__ __forceinline__ void faraday_face(const DevMesh &d, const R *E, const double *dte, const R *dt_dev, double dt_val, R *B, int32_t f)
{
    if (f >= d.nf) return;
    if (d.fL[f] < 0 && d.fR[f] < 0) return;
    R circ = 0.0;
    if (dte)
    {
        for (int32_t k = d.f2e_ptr[f]; k < d.f2e_ptr[f + 1]; ++k)
        {
            const int32_t v = d.f2e[k], e = pid(v);
            circ += psg(v) * dte[e] * E[e];
        }
        B[f] -= circ;
        return;
    }
    if (d.fdeg == 3)
    {
        // triangles: the three edge entries in one 12-byte load, then the gathers, summed in entry order
        const int3 q = reinterpret_cast<const int3 *>(d.f2e)[f];
        const R x = E[pid(q.x)], y = E[pid(q.y)], z = E[pid(q.z)];
        circ += psg(q.x) * x;
        circ += psg(q.y) * y;
        circ += psg(q.z) * z;
    }
    else
        for (int32_t k = d.f2e_ptr[f]; k < d.f2e_ptr[f + 1]; ++k)
        {
            const int32_t v = d.f2e[k];
            circ += psg(v) * E[pid(v)];
        }
    const R dt = dt_dev ? dt_dev[0] : dt_val;
    B[f] -= dt * circ;
}

// One edge of valence at most `vmax` per thread (IdealEMF.cpp:59-128)
template <class R>
__device__ __forceinline__ void edge_emf_light(const DevMesh &d, const Params &P, const R *Ef, const R *u_cell, double cuct, int32_t vmax,
                                               int32_t e, const R *E_in, R *E_out, int32_t apply_bc)
{
    if (e >= d.ne) return;
    const int32_t f0 = d.e2f_ptr[e], f1 = d.e2f_ptr[e + 1];
    const int32_t nf = f1 - f0;
    if (nf > vmax) return;
    R out = E_in ? E_in[e] : 0.0;
    const int32_t c0 = d.ec_ptr[e], c1 = d.ec_ptr[e + 1];
    const int32_t nc = c1 - c0;
    const bool fast = nf <= kEmfFast && nc <= kEmfFast;
    // common valence: the row indices are loaded once, together, before their gathers
    int32_t fid[kEmfFast], cid[kEmfFast];
    bool any_fluid = false;
    if (fast)
    {
#pragma unroll
        for (int i = 0; i < kEmfFast; ++i)
        {
            if (i < nf) fid[i] = pid(d.e2f[f0 + i]);
            if (i < nc) cid[i] = d.ec_cell[c0 + i];
        }
#pragma unroll
        for (int k = 0; k < kEmfFast; ++k)
            if (k < nc) any_fluid |= d.mat[cid[k]] == 0;
    }
    else
        for (int32_t k = c0; k < c1 && !any_fluid; ++k) any_fluid = d.mat[d.ec_cell[k]] == 0;
    if (nf > 0 && d.elen[e] > 0 && any_fluid)
    {
        const V3 t = L3(d.evec, e);
        const double L = d.elen[e];
        const V3 th = (1.0 / L) * t;
        R Ec = 0;
        if (fast)
        {
            V3T<R> ef[kEmfFast];
#pragma unroll
            for (int i = 0; i < kEmfFast; ++i)
                if (i < nf) ef[i] = emf_of(Ef, fid[i]);
#pragma unroll
            for (int i = 0; i < kEmfFast; ++i)
                if (i < nf) Ec += d.efw[f0 + i] * dot(ef[i], t);
        }
        else
            for (int32_t i = f0; i < f1; ++i) Ec += d.efw[i] * dot(emf_of(Ef, pid(d.e2f[i])), t);
        V3 e1, e2;
        plane_basis(th, e1, e2);
        R M11 = 0, M12 = 0, M22 = 0, g1 = 0, g2 = 0, Eu = 0;
        if (fast)
        {
            // the edge's cell velocities and the per-face terms stay in registers, so the second pass re-reads
            // nothing (same operations in the same order as the general path)
            V3T<R> uc[kEmfFast];
#pragma unroll
            for (int k = 0; k < kEmfFast; ++k)
                if (k < nc) uc[k] = L3(u_cell, cid[k]);
            R fqa[kEmfFast], fqb[kEmfFast], faef[kEmfFast], fsig[kEmfFast];
#pragma unroll
            for (int i = 0; i < kEmfFast; ++i)
                if (i < nf)
                {
                    const int32_t f = fid[i];
                    V3 m, nrm;
                    face_dirs(d, f, e, th, m, nrm);
                    R aef = 0.0;
#pragma unroll
                    for (int k = 0; k < kEmfFast; ++k)
                        if (k < nc) aef = mx(aef, fabs(dot(uc[k], m)));
                    const R sig = dot(th, cross(m, nrm));
                    const V3T<R> qv = (aef * sig) * nrm;
                    const R qa = dot(qv, e1), qb = dot(qv, e2), w = d.efw[f0 + i];
                    M11 += w * qa * qa;
                    M12 += w * qa * qb;
                    M22 += w * qb * qb;
                    g1 += w * qa;
                    g2 += w * qb;
                    fqa[i] = qa; fqb[i] = qb; faef[i] = aef; fsig[i] = sig;
                }
            R l1, l2;
            uct_solve(M11, M12, M22, g1, g2, l1, l2);
            // the face weight and flux are loaded again (cache hits) rather than held across the solve
#pragma unroll
            for (int i = 0; i < kEmfFast; ++i)
                if (i < nf)
                {
                    const R omega = d.efw[f0 + i] * (1.0 - (fqa[i] * l1 + fqb[i] * l2));
                    Eu += omega * faef[i] * fsig[i] * Ef[4 * size_t(fid[i]) + 3];
                }
        }
        else
        {
            for (int32_t i = f0; i < f1; ++i)
            {
                const int32_t f = pid(d.e2f[i]);
                V3 m, nrm;
                face_dirs(d, f, e, th, m, nrm);
                const R aef = edge_amax(d, u_cell, c0, c1, m);
                const V3T<R> qv = (aef * dot(th, cross(m, nrm))) * nrm;
                const R qa = dot(qv, e1), qb = dot(qv, e2), w = d.efw[i];
                M11 += w * qa * qa;
                M12 += w * qa * qb;
                M22 += w * qb * qb;
                g1 += w * qa;
                g2 += w * qb;
            }
            R l1, l2;
            uct_solve(M11, M12, M22, g1, g2, l1, l2);
            for (int32_t i = f0; i < f1; ++i)
            {
                const int32_t f = pid(d.e2f[i]);
                V3 m, nrm;
                face_dirs(d, f, e, th, m, nrm);
                const R aef = edge_amax(d, u_cell, c0, c1, m);
                const V3T<R> qv = (aef * dot(th, cross(m, nrm))) * nrm;
                const R qa = dot(qv, e1), qb = dot(qv, e2), w = d.efw[i];
                const R omega = w * (1.0 - (qa * l1 + qb * l2));
                const R sig = dot(th, cross(m, nrm));
                Eu += omega * aef * sig * Ef[4 * size_t(f) + 3];
            }
        }
        out += Ec + 2.0 * cuct * L * Eu;
    }
    E_out[e] = apply_bc ? edge_bc(d, P, e, out) : out;
}
} // namespace
} // namespace mhdg
