// Explicit stage of the fused step (mercury::Solver::step_first_order, MercuryUns/driver/Solver.cpp:228-277) on the
// resident state, in the layouts of explicit_step.h.  Every sum runs in the order of the reference and of the
// single-operation kernels of explicit.hip, so the step is theirs bit for bit.
//
// Four launches on a step without an implicit part, each a set of roles that are independent of each other:
//   prepare          primitives, cell fields, CFL step
//   states           limited gradients -> face states, cell current | face EMF candidates | final CFL minimum
//   fluxes           Rusanov fluxes | edge EMF, high-valence edges first
//   update           owner gather, sources, forward Euler, floors | constrained transport
// On small meshes a kernel lasts as long as one thread's chain of dependent loads and divisions, so roles side by side
// save whole launches; on large ones a role gets the registers and LDS of its launch's largest, which cost nothing
// measurable (8M tetrahedra: 6181 us per step with the face EMFs in the states' launch, 6200 in one of their own).
//
// Measured, microseconds per explicit step, against one kernel per operation with gradients in memory (8 launches; one
// MI355X): 9.5k tetrahedra 90 -> 36, 60k 113 -> 58, 484k 547 -> 400, 1.95M 1982 -> 1547, 7.83M 7723 -> 6196.  At 7.83M
// prepare takes 617 us (994 before), states 2331 and fluxes 2403 (5660 for the gradients, fluxes, EMF candidates and
// edge sums before), update 846 (1073).  prepare, the flux half of fluxes and update run at 5.0-5.5 TB/s of their bytes
// (the streaming copy reaches 6.1); states is bound by its FP64 instructions and the loads' latency at three waves per
// SIMD, the edge half of fluxes by the L1's outstanding requests.  The roles' blocks follow one another: taking them in
// turn, one or eight each, let the two working sets evict each other (484k: fluxes 153 -> 213 us, states 154 -> 206).
#include <algorithm>
#include <cmath>
#include <stdexcept>
#include <type_traits>

#include "ctx.h"
#include "explicit_step.h"
#include "step_cell.h"

namespace mhdg
{
// ---------------------------------------------------------------------------------------------------- set-up tables
__global__ void __launch_bounds__(256) k_face_geo(DevMesh d, double *geo)
{
    const int32_t f = gid();
    if (f >= d.nf) return;
    const double A = d.famag[f];
    const V3 n = (1.0 / A) * L3(d.farea, f);
    double *g = geo + 4 * size_t(f);
    g[0] = n.x; g[1] = n.y; g[2] = n.z; g[3] = A;
}
// one thread per face: its entries in the rows of its two cells, and which flux it carries (FluxRHS.cpp:36-62)
__global__ void __launch_bounds__(256) k_face_entries(DevMesh d, int2 *fent, int8_t *fcls)
{
    const int32_t f = gid();
    if (f >= d.nf) return;
    const int32_t l = d.fL[f], r = d.fR[f];
    // of a cell that sees the face from both sides, the entry of that side
    auto entry = [&](int32_t c, int32_t v) {
        int32_t any = -1;
        for (int32_t k = c < 0 ? 0 : d.c2f_ptr[c]; c >= 0 && k < d.c2f_ptr[c + 1]; ++k)
        {
            if (d.c2f[k] == v) return k;
            if (pid(d.c2f[k]) == f && any < 0) any = k;
        }
        return any;
    };
    fent[f] = make_int2(entry(l, f), entry(r, ~f));
    const bool any = (l >= 0 && d.mat[l] == 0) || (r >= 0 && d.mat[r] == 0);
    int8_t cls;
    if (d.kind[f] == kSkip || !any) cls = kFluxNone;
    else if (l >= 0 && r >= 0 && d.kind[f] == kInterior) cls = kFluxInner;
    else
    {
        int32_t c;
        if (l >= 0 && r >= 0)
        {
            // the fluid cell, the lower id first (FluxRHS.cpp:57-62)
            const int32_t first = l < r ? l : r, second = l < r ? r : l;
            c = d.mat[first] == 1 ? second : first;
        }
        else c = l >= 0 ? l : r;
        cls = c == l ? kFluxLeft : kFluxRight;
    }
    fcls[f] = cls;
}
// columns [first, first + n) of the cell records as a dense n-per-cell array, for a getter: one launch ahead of the copy to
// the host (B_ind of 4k hexahedra 17 us without it, 30 with; of 484k tetrahedra 798 and 804)
__global__ void __launch_bounds__(256) k_rec_get(const double *rec, int32_t rs, int32_t first, int32_t n, int32_t nc, double *out)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < int64_t(n) * nc) out[i] = rec[size_t(rs) * size_t(i / n) + size_t(first + i % n)];
}

namespace
{
constexpr int kStatesThreads = 128; // block of the (cell, ion) kernels: 20 KB of face states staged per block on tetrahedra
constexpr int kRoleThreads = 256;
constexpr int kBatch = 2; // neighbour rows in flight per thread in the gradients (all four at once spilled at three waves per SIMD)

// cell_vector_add (fv.h) with the unit normal given: (s / |A|) a is s ((1 / |A|) a) bit for bit
__device__ __forceinline__ void vector_add(double (&M)[3][3], double (&r)[3], double s, double A, const V3 &n, double flux)
{
    if (A <= 0) return;
    const double nv[3] = {s * n.x, s * n.y, s * n.z};
    const double phi = s * flux;
    for (int i = 0; i < 3; ++i)
    {
        r[i] += nv[i] * phi;
        for (int j = 0; j < 3; ++j) M[i][j] += A * nv[i] * nv[j];
    }
}
// The face sum of cell_dt (fv.h) for one ion: one face's term
__device__ __forceinline__ double dt_term(const Params &P, const double *w, double cs2, double vA2, double rho_tot, const V3 &b, const V3 &n,
                                          double A)
{
    const double vAn2 = P.inver_MA2 * dot(b, n) * dot(b, n) / rho_tot;
    const double term = cs2 + vA2;
    const double cf = sqrt(0.5 * (term + sqrt(mx(0.0, term * term - 4 * cs2 * vAn2))));
    return (fabs(w[1] * n.x + w[2] * n.y + w[3] * n.z) + cf) * A;
}
// Cell field of Phi and the CFL step of the ions [s0, s1) of cell c, whose primitives are W[5 s] (Solver.cpp:94-125,
// MercurySources.cpp:104-145).  Up to DEG faces stay in registers; DEG 0 walks the row twice.
template <int DEG>
__device__ __forceinline__ void cell_fields(const DevMesh &d, const Params &P, int32_t c, const double *Phi,
                                            const double *Badd, const double *W, int32_t s0, int32_t s1, bool fluid, V3 &bi, V3 &bt,
                                            double &dtc)
{
    constexpr int N = DEG > 0 ? DEG : 1;
    int32_t k0, nk;
    row_of<DEG>(d, c, k0, nk);
    double M[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, r[3] = {0, 0, 0};
    V3 n[N];
    double A[N];
    const V3 ba = L3(Badd, c);
    const double vol = d.cvol[c];
    if constexpr (DEG > 0)
    {
        int32_t v[N];
        double fl[N];
        row_ids<DEG>(d.c2f, k0, v);
#pragma unroll
        for (int i = 0; i < DEG; ++i) { n[i] = geo_normal(d, pid(v[i]), A[i]); fl[i] = Phi[pid(v[i])]; }
#pragma unroll
        for (int i = 0; i < DEG; ++i) vector_add(M, r, psg(v[i]), A[i], n[i], fl[i]);
    }
    else
        for (int32_t k = k0; k < k0 + nk; ++k)
        {
            const int32_t v = d.c2f[k];
            double a;
            const V3 m = geo_normal(d, pid(v), a);
            vector_add(M, r, psg(v), a, m, Phi[pid(v)]);
        }
    bi = cell_vector_solve(M, r);
    bt = V3(bi.x + ba.x, bi.y + ba.y, bi.z + ba.z);
    dtc = __builtin_inf();
    if (!fluid) return;
    double rho = W[0];
    for (int s = 1; s < P.ns; ++s) rho = rho + W[5 * s];
    const double rho_tot = mx(rho, P.rho_floor_dt);
    const double vA2 = P.inver_MA2 * dot(bt, bt) / rho_tot;
    for (int s = s0; s < s1; ++s)
    {
        const double *w = W + 5 * s;
        const double cs2 = P.gamma * w[4] / mx(w[0], 1e-30);
        double denom = 0;
        if constexpr (DEG > 0)
        {
#pragma unroll
            for (int i = 0; i < DEG; ++i) denom += dt_term(P, w, cs2, vA2, rho_tot, bt, n[i], A[i]);
        }
        else
            for (int32_t k = k0; k < k0 + nk; ++k)
            {
                double a;
                const V3 m = geo_normal(d, pid(d.c2f[k]), a);
                denom += dt_term(P, w, cs2, vA2, rho_tot, bt, m, a);
            }
        if (denom > 0) dtc = mn(dtc, P.cfl * vol / denom);
    }
}
} // namespace

// Solver::prepare + cell_time_steps + alpha of the frozen Hall state (as k_prepare), two ions, one thread per cell; the
// block's 128-byte records are staged in LDS (17 doubles a row: no bank conflicts) and written as one range.
template <int DEG>
__global__ void __launch_bounds__(256) k_step_prepare2(DevMesh d, Params P, SpC Us, const double *Phi, const double *Badd, StepFields F,
                                                       double *dt_part)
{
    __shared__ double stage[256 * 17];
    const int32_t block = near_block(d, int32_t(blockIdx.x), 0, int32_t(gridDim.x)), c = block * 256 + int32_t(threadIdx.x);
    double dtc = __builtin_inf();
    if (c < d.nc)
    {
        double W[10];
#pragma unroll
        for (int s = 0; s < 2; ++s)
        {
            const Prim a = to_prim(Us.p[s] + 5 * size_t(c), P.gamma, P.rho_floor, P.p_floor);
            W[5 * s] = a.rho; W[5 * s + 1] = a.u; W[5 * s + 2] = a.v; W[5 * s + 3] = a.w; W[5 * s + 4] = a.p;
        }
        const bool fluid = d.mat[c] == 0;
        const V3 xc = L3(d.ccen, c);
        V3 bi, bt, up;
        cell_fields<DEG>(d, P, c, Phi, Badd, W, 0, 2, fluid, bi, bt, dtc);
        double al = 0.0;
        if (fluid)
        {
            const double n0 = ion_density(P, 0, W[0]), n1 = ion_density(P, 1, W[5]);
            const double ne = n0 + n1;
            const double ne_eff = sqrt(ne * ne + P.ne_floor * P.ne_floor);
            const double x0 = ne > 1e-300 ? n0 / ne : 1.0, x1 = ne > 1e-300 ? n1 / ne : 0.0;
            up = V3(x0 * W[1], x0 * W[2], x0 * W[3]);
            up = V3(up.x + x1 * W[6], up.y + x1 * W[7], up.z + x1 * W[8]);
            al = (P.hall && ne_eff > 0) ? d.taper[c] * P.hall_coef / ne_eff : 0.0;
        }
        st3(F.Btot, c, bt);
        st3(F.uplus, c, up);
        F.alpha[c] = al;
        double *q = stage + 17 * threadIdx.x;
#pragma unroll
        for (int m = 0; m < 10; ++m) q[m] = W[m];
        q[10] = bi.x; q[11] = bi.y; q[12] = bi.z; q[13] = xc.x; q[14] = xc.y; q[15] = xc.z;
    }
    __syncthreads();
    const int32_t c0 = block * 256, n_here = min(256, d.nc - c0);
    for (int32_t i = threadIdx.x; i < 16 * n_here; i += 256) F.rec[16 * size_t(c0) + i] = stage[17 * (i >> 4) + (i & 15)];
    __syncthreads();
    const double m = block_min(dtc, stage);
    if (threadIdx.x == 0) dt_part[block] = m;
}

// The same for more than two ions: one thread per (cell, ion), the ions of a cell side by side, so the record rows and
// the time step's face sums are spread over them; the sums over the ions run in their order from LDS.
template <int DEG>
__global__ void __launch_bounds__(256) k_step_prepare_many(DevMesh d, Params P, SpC Us, const double *Phi, const double *Badd, StepFields F,
                                                           double *dt_part)
{
    __shared__ double sW[256 * 5], sn[256];
    const int32_t ns = P.ns, per = 256 / ns, t = threadIdx.x, cl = t / ns, s = t - cl * ns;
    const int32_t c = near_block(d, int32_t(blockIdx.x), 0, int32_t(gridDim.x)) * per + cl;
    const bool act = cl < per && c < d.nc;
    double dtc = __builtin_inf();
    if (act)
    {
        const Prim a = to_prim(Us.p[s] + 5 * size_t(c), P.gamma, P.rho_floor, P.p_floor);
        double *w = sW + 5 * t, *row = F.rec + size_t(F.rs) * size_t(c) + 5 * s;
        w[0] = a.rho; w[1] = a.u; w[2] = a.v; w[3] = a.w; w[4] = a.p;
        row[0] = a.rho; row[1] = a.u; row[2] = a.v; row[3] = a.w; row[4] = a.p;
        sn[t] = ion_density(P, s, a.rho);
    }
    __syncthreads();
    if (act)
    {
        const double *W = sW + 5 * cl * ns, *n = sn + cl * ns;
        const bool fluid = d.mat[c] == 0;
        V3 bi, bt;
        cell_fields<DEG>(d, P, c, Phi, Badd, W, s, s + 1, fluid, bi, bt, dtc);
        double ne = n[0];
        for (int q = 1; q < ns; ++q) ne = ne + n[q];
        if (s < 3)
        {
            // component s of the cell's vectors
            double up = 0.0;
            if (fluid)
                for (int q = 0; q < ns; ++q)
                {
                    const double chi = ne > 1e-300 ? n[q] / ne : (q == 0 ? 1.0 : 0.0);
                    up = q == 0 ? chi * W[1 + s] : up + chi * W[5 * q + 1 + s];
                }
            const size_t o = 3 * size_t(c) + size_t(s);
            double *row = F.rec + size_t(F.rs) * size_t(c) + 5 * ns;
            F.uplus[o] = up;
            F.Btot[o] = s == 0 ? bt.x : s == 1 ? bt.y : bt.z;
            row[s] = s == 0 ? bi.x : s == 1 ? bi.y : bi.z;
            row[3 + s] = d.ccen[o];
        }
        if (s == 0)
        {
            const double ne_eff = sqrt(ne * ne + P.ne_floor * P.ne_floor);
            F.alpha[c] = (fluid && P.hall && ne_eff > 0) ? d.taper[c] * P.hall_coef / ne_eff : 0.0;
        }
    }
    __syncthreads();
    const double m = block_min(dtc, sW);
    if (t == 0) dt_part[blockIdx.x] = m;
}

namespace
{
// ------------------------------------------------------------------------------------------------------------ roles
// Limited gradients (Reconstruction.cpp:80-142) of one ion of a cell, and from them the cell's states at its faces
// (FluxRHS.cpp:16-27): thread (cell, ion), the ions of a cell side by side.  All of a row's neighbour records and face
// centres are loaded before the first is used (a load behind the test for a boundary face waited for it).  The
// neighbour's offset and weight are formed from the centres in the records, as the set-up forms them (tables.cpp), which
// reads 128 bytes a cell less than their tables.  Also cell_current (Current.cpp:9-31): the faces' terms are split over
// the cell's threads and summed in face order.
template <int DEG, int NS>
__device__ __forceinline__ void states_role(const DevMesh &d, const Params &P, const StepFields &F, int32_t block, double *stage)
{
    constexpr int N = DEG > 0 ? DEG : 1;
    const int32_t ns = NS > 0 ? NS : P.ns, per = kStatesThreads / ns, t = threadIdx.x, cl = t / ns, s = t - cl * ns;
    const int32_t c0 = block * per, c = c0 + cl;
    const bool act = cl < per && c < d.nc;
    const size_t rs = NS == 2 ? 16 : size_t(F.rs);
    const int32_t ob = 5 * ns; // the field, then the centre, after the ions
    double *jst = stage;       // cross products of the current first, the face states after them
    int32_t k0 = 0, nk = 0;
    if (act) row_of<DEG>(d, c, k0, nk);
    const double *own = F.rec + rs * size_t(act ? c : 0);
    int32_t v[N];
    if constexpr (DEG > 0)
    {
        if (act)
        {
            int32_t o[N];
            row_ids<DEG>(d.c2f, k0, v);
            row_ids<DEG>(d.c2n, k0, o);
            const V3 bc(own[ob], own[ob + 1], own[ob + 2]);
            const int32_t lanes = ns < DEG ? ns : DEG;
#pragma unroll
            for (int i = 0; i < DEG; ++i)
                if (i % lanes == s)
                {
                    const double *r = F.rec + rs * size_t(o[i] >= 0 ? o[i] : c) + ob;
                    const V3 bo(r[0], r[1], r[2]), area = L3(d.farea, pid(v[i]));
                    V3 bf = bc;
                    if (o[i] >= 0) bf = 0.5 * (bc + bo);
                    const V3 x = cross(psg(v[i]) * area, bf);
                    double *j = jst + 3 * (cl * DEG + i);
                    j[0] = x.x; j[1] = x.y; j[2] = x.z;
                }
        }
        __syncthreads();
    }
    if (act && s == 0)
    {
        V3 sum;
        if constexpr (DEG > 0)
        {
#pragma unroll
            for (int i = 0; i < DEG; ++i)
            {
                const double *j = jst + 3 * (cl * DEG + i);
                sum += V3(j[0], j[1], j[2]);
            }
        }
        else
        {
            const V3 bc(own[ob], own[ob + 1], own[ob + 2]);
            for (int32_t k = k0; k < k0 + nk; ++k)
            {
                const int32_t q = d.c2f[k], o = d.c2n[k];
                V3 bf = bc;
                if (o >= 0)
                {
                    const double *r = F.rec + rs * size_t(o) + ob;
                    bf = 0.5 * (bc + V3(r[0], r[1], r[2]));
                }
                sum += cross(psg(q) * L3(d.farea, pid(q)), bf);
            }
        }
        const double invV = 1.0 / d.cvol[c];
        st3(F.J, c, V3(sum.x * invV, sum.y * invV, sum.z * invV));
    }
    if constexpr (DEG > 0) __syncthreads(); // the cross products are read; stage takes the face states
    if (act)
    {
        double wc[5], lo[5], hi[5], r[5][3], g[5][3];
        const V3 xc(own[ob + 3], own[ob + 4], own[ob + 5]);
        for (int m = 0; m < 5; ++m) { wc[m] = own[5 * s + m]; lo[m] = hi[m] = wc[m]; r[m][0] = r[m][1] = r[m][2] = 0.0; }
        const bool valid = P.second_order && d.svalid[c];
        double fs[5];
        for (int m = 0; m < 5; ++m) fs[m] = P.fs[s][m];
        auto boundary_offset = [&](int32_t q) {
            double A;
            const V3 n = psg(q) * geo_normal(d, pid(q), A);
            return (2.0 * dot(L3(d.fcen, pid(q)) - xc, n)) * n;
        };
        auto accumulate = [&](const V3 &dd, const double *wn) {
            const double w = 1.0 / dot(dd, dd);
            for (int m = 0; m < 5; ++m)
            {
                const double dq = wn[m] - wc[m];
                r[m][0] += w * dd.x * dq; r[m][1] += w * dd.y * dq; r[m][2] += w * dd.z * dq;
                lo[m] = mn(lo[m], wn[m]);
                hi[m] = mx(hi[m], wn[m]);
            }
        };
        const double *I = d.sinv + 6 * size_t(c);
        V3 dx[N];
        if constexpr (DEG > 0)
        {
            int32_t nb[N];
            row_ids<DEG>(d.snb, k0, nb);
#pragma unroll
            for (int i0 = 0; i0 < DEG; i0 += kBatch)
            {
                double wn[kBatch][5];
                V3 xn[kBatch];
#pragma unroll
                for (int u = 0; u < kBatch; ++u)
                {
                    const double *q = F.rec + rs * size_t(nb[i0 + u] >= 0 ? nb[i0 + u] : c);
                    for (int m = 0; m < 5; ++m) wn[u][m] = q[5 * s + m];
                    xn[u] = V3(q[ob + 3], q[ob + 4], q[ob + 5]);
                }
                if (valid)
#pragma unroll
                    for (int u = 0; u < kBatch; ++u)
                    {
                        const int i = i0 + u;
                        V3 dd = xn[u] - xc;
                        if (nb[i] < 0)
                        {
                            if (nb[i] == kNoStencil) continue;
                            dd = boundary_offset(v[i]);
                            stencil_ghost(d, s, static_cast<const double *>(nullptr), wc, fs, v[i], nb[i], wn[u]);
                        }
                        accumulate(dd, wn[u]);
                    }
            }
#pragma unroll
            for (int i = 0; i < DEG; ++i) dx[i] = L3(d.fcen, pid(v[i])) - xc;
        }
        else if (valid)
            for (int32_t k = k0; k < k0 + nk; ++k)
            {
                const int32_t nb = d.snb[k], q = d.c2f[k];
                if (nb == kNoStencil) continue;
                double wn[5];
                V3 dd;
                if (nb >= 0)
                {
                    const double *x = F.rec + rs * size_t(nb);
                    for (int m = 0; m < 5; ++m) wn[m] = x[5 * s + m];
                    dd = V3(x[ob + 3], x[ob + 4], x[ob + 5]) - xc;
                }
                else
                {
                    stencil_ghost(d, s, static_cast<const double *>(nullptr), wc, fs, q, nb, wn);
                    dd = boundary_offset(q);
                }
                accumulate(dd, wn);
            }
        const double I0 = I[0], I1 = I[1], I2 = I[2], I3 = I[3], I4 = I[4], I5 = I[5];
        // The smallest of the faces' quotients room / dl is that of the largest |dl| of its sign (the room, at least 0, is the
        // same for them and a rounded division is monotone), so each primitive divides twice, or three times with the
        // relative limit, whatever the number of faces, and behind no branch: a division per face, each in its own, made
        // 28 of them a serial chain (60k tetrahedra 59.3 -> 57.6 us a step, 7.83M 6235 -> 6196; ten ions, 1.1M cells: the states
        // 1153 -> 1116 us, and 1065 with the fourth wave per SIMD that 38 registers fewer allow).
        auto reach = [&](int m, const V3 &x, double &up, double &down) {
            const double dl = g[m][0] * x.x + g[m][1] * x.y + g[m][2] * x.z;
            up = mx(up, dl);
            down = mn(down, dl);
        };
        auto quotient = [](double room, double dl, double psi) {
            const bool counts = fabs(dl) > 1e-300;
            return mn(psi, (counts ? room : 1.0) / (counts ? dl : 1.0));
        };
        for (int m = 0; m < 5; ++m)
        {
            g[m][0] = g[m][1] = g[m][2] = 0.0;
            if (!valid) continue;
            g[m][0] = I0 * r[m][0] + I1 * r[m][1] + I2 * r[m][2];
            g[m][1] = I1 * r[m][0] + I3 * r[m][1] + I4 * r[m][2];
            g[m][2] = I2 * r[m][0] + I4 * r[m][1] + I5 * r[m][2];
            const bool rel = P.rel_limit > 0 && (m == 0 || m == 4);
            double psi = 1.0, up = 0.0, down = 0.0;
            if constexpr (DEG > 0)
            {
#pragma unroll
                for (int i = 0; i < DEG; ++i) reach(m, dx[i], up, down);
            }
            else
                for (int32_t k = k0; k < k0 + nk; ++k) reach(m, L3(d.fcen, pid(d.c2f[k])) - xc, up, down);
            psi = quotient(hi[m] - wc[m], up, psi);
            psi = quotient(lo[m] - wc[m], down, psi);
            if (rel) psi = quotient(P.rel_limit * wc[m], mx(up, -down), psi);
            psi = mx(0.0, mn(1.0, psi));
            g[m][0] = psi * g[m][0]; g[m][1] = psi * g[m][1]; g[m][2] = psi * g[m][2];
        }
        auto face_state_of = [&](const V3 &x, double *out) {
            double q[5];
            for (int m = 0; m < 5; ++m) q[m] = wc[m] + g[m][0] * x.x + g[m][1] * x.y + g[m][2] * x.z;
            const bool ok = q[0] > 0 && q[4] > 0;
            for (int m = 0; m < 5; ++m) out[m] = ok ? q[m] : wc[m];
        };
        if constexpr (DEG > 0)
        {
#pragma unroll
            for (int i = 0; i < DEG; ++i) face_state_of(dx[i], stage + 5 * ((cl * DEG + i) * ns + s));
        }
        else
            for (int32_t k = k0; k < k0 + nk; ++k) face_state_of(L3(d.fcen, pid(d.c2f[k])) - xc, F.FS + 5 * (size_t(k) * size_t(ns) + s));
    }
    if constexpr (DEG > 0)
    {
        __syncthreads();
        const int32_t n_here = min(per, d.nc - c0) * (DEG * ns * 5 / 2);
        double2 *dst = reinterpret_cast<double2 *>(F.FS + size_t(c0) * size_t(DEG * 5 * ns));
        const double2 *src = reinterpret_cast<const double2 *>(stage);
        for (int32_t i = t; i < n_here; i += kStatesThreads) dst[i] = src[i];
    }
}

// Ideal EMF candidate of a face (IdealEMF.cpp:32-55), with Phi / |A| for the edge sum
__device__ __forceinline__ void face_emf_role(const DevMesh &d, const StepFields &F, const double *Phi, const double *PhiAdd, int32_t f)
{
    if (f >= d.nf) return;
    const int32_t l = d.fL[f], r = d.fR[f];
    double A;
    const V3 n = geo_normal(d, f, A);
    const double ph = Phi[f], Bn_tot = (ph + PhiAdd[f]) / A;
    const double *Bi = F.rec + 5 * F.ns;
    V3 E;
    if (l >= 0 && r >= 0)
    {
        const V3 uL = L3(F.uplus, l), uR = L3(F.uplus, r), tL = L3(F.Btot, l), tR = L3(F.Btot, r);
        const V3 iL = L3(Bi + size_t(F.rs) * size_t(l), 0), iR = L3(Bi + size_t(F.rs) * size_t(r), 0);
        const V3 fl = dot(uL, n) * tL - Bn_tot * uL, fr = dot(uR, n) * tR - Bn_tot * uR;
        const double a = mx(fabs(dot(uL, n)), fabs(dot(uR, n)));
        E = 0.5 * (fl + fr) - (0.5 * a) * (iR - iL);
    }
    else if (const int32_t c = l >= 0 ? l : r; c >= 0) // zero on a face without a cell
    {
        const V3 u = L3(F.uplus, c);
        E = dot(u, n) * L3(F.Btot, c) - Bn_tot * u;
    }
    E = -1.0 * cross(n, E);
    double2 *out = reinterpret_cast<double2 *>(F.Ef + 4 * size_t(f));
    out[0] = make_double2(E.x, E.y);
    out[1] = make_double2(E.z, ph / A);
}

// min of the blocks' time steps, at most dt_max, on the device and into host memory (one block)
__device__ __forceinline__ void dt_role(const double *part, int32_t n, double dt_max, double *out, double *sh, HostBox *box, uint64_t ticket)
{
    const int32_t t = threadIdx.x, nt = blockDim.x;
    double v = __builtin_inf();
    for (int32_t i = t; i < n; i += 4 * nt)
    {
        double x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = i + u * nt < n ? part[i + u * nt] : __builtin_inf();
#pragma unroll
        for (int u = 0; u < 4; ++u) v = mn(v, x[u]);
    }
    v = mn(block_min(v, sh), dt_max);
    __syncthreads(); // every thread has read the minimum
    if (t == 0) out[0] = sh[0] = v;
    __syncthreads();
    publish(box, ticket, sh, 1);
}

// Rusanov flux through a face (FluxRHS.cpp:43-70) for one ion: thread (face, ion), the ions of a face side by side
template <int NS>
__device__ __forceinline__ void flux_role(const DevMesh &d, const Params &P, const StepFields &F, int32_t block, double *stage)
{
    const int32_t ns = NS > 0 ? NS : P.ns, per = kRoleThreads / ns, t = threadIdx.x, fl = t / ns, s = t - fl * ns;
    const int32_t f0 = block * per, f = f0 + fl;
    if (fl < per && f < d.nf)
    {
        const int2 e = F.fent[f];
        const int8_t cls = F.fcls[f];
        double out[5] = {0, 0, 0, 0, 0};
        if (cls != kFluxNone)
        {
            double A;
            const V3 n = geo_normal(d, f, A);
            auto state = [&](int32_t k) {
                const double *q = F.FS + 5 * (size_t(k) * size_t(ns) + s);
                return Prim{q[0], q[1], q[2], q[3], q[4]};
            };
            Prim L, R;
            if (cls == kFluxInner) { L = state(e.x); R = state(e.y); }
            else
            {
                const Prim in = state(cls == kFluxLeft ? e.x : e.y);
                double fs[5];
                for (int m = 0; m < 5; ++m) fs[m] = P.fs[s][m];
                const Prim gh = ghost_state(d.kind[f], s, in, (cls == kFluxLeft ? 1.0 : -1.0) * n, fs);
                if (cls == kFluxLeft) { L = in; R = gh; } else { R = in; L = gh; }
            }
            const double nv[3] = {n.x, n.y, n.z};
            double flux[5];
            rusanov(L, R, nv, P.gamma, flux);
            for (int m = 0; m < 5; ++m) out[m] = flux[m] * A;
        }
        for (int m = 0; m < 5; ++m) stage[5 * t + m] = out[m];
    }
    __syncthreads();
    const int32_t n_here = min(per, d.nf - f0) * 5 * ns;
    double *dst = F.FA + size_t(f0) * size_t(5 * ns);
    for (int32_t i = t; i < n_here; i += kRoleThreads) dst[i] = stage[i];
}

// Owner gather of the fluxes in ascending face order (FluxRHS.cpp:71-72), Lorentz and production sources
// (MercurySources.cpp:20-63), forward Euler and floors (Solver.cpp:246-252, 171-191): thread (cell, ion)
template <int DEG, int NS>
__device__ __forceinline__ void update_role(const DevMesh &d, const Params &P, const StepFields &F, const double *dt_dev, const SpW &Us,
                                            int32_t block)
{
    const int32_t ns = NS > 0 ? NS : P.ns, per = kRoleThreads / ns, t = threadIdx.x, cl = t / ns, s = t - cl * ns;
    const int32_t c = block * per + cl;
    if (cl >= per || c >= d.nc || d.mat[c] != 0) return;
    const double dt = dt_dev[0], V = d.cvol[c];
    const double *row = F.rec + (NS == 2 ? 16 : size_t(F.rs)) * size_t(c);
    double *u = Us.p[s] + 5 * size_t(c);
    double rhs[5];
    cell_rhs<DEG>(d, P, F, c, s, ns, row, V, dt, rhs);
    double q[5];
    for (int m = 0; m < 5; ++m) q[m] = u[m] + dt * rhs[m];
    const double ke = q[0] > 0 ? 0.5 * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]) / q[0] : 0.0;
    if (!(q[0] >= P.rho_floor)) to_cons(Prim{P.rho_floor, 0, 0, 0, P.p_floor}, P.gamma, q);
    else if ((P.gamma - 1.0) * (q[4] - ke) < P.p_floor)
    {
        const Prim w = to_prim(q, P.gamma, P.rho_floor, P.p_floor);
        to_cons(w, P.gamma, q);
    }
    for (int m = 0; m < 5; ++m) u[m] = q[m];
}
} // namespace

// cell_current (Current.cpp:9-31) alone, of the fields in the records, for a caller that wants the derived fields of a state
// and takes no step (7.83M tetrahedra: 493 us; the states, which form it on the side for a step, 1729)
template <int DEG> __global__ void __launch_bounds__(kRoleThreads) k_step_current(DevMesh d, StepFields F)
{
    constexpr int N = DEG > 0 ? DEG : 1;
    const int32_t c = gid(d);
    if (c >= d.nc) return;
    int32_t k0, nk;
    row_of<DEG>(d, c, k0, nk);
    auto field = [&](int32_t q) { return L3(F.rec + size_t(F.rs) * size_t(q) + 5 * F.ns, 0); };
    const V3 bc = field(c);
    V3 sum;
    auto add = [&](int32_t v, int32_t o, const V3 &bo) {
        V3 bf = bc;
        if (o >= 0) bf = 0.5 * (bc + bo);
        sum += cross(psg(v) * L3(d.farea, pid(v)), bf);
    };
    if constexpr (DEG > 0)
    {
        int32_t v[N], o[N];
        V3 bo[N];
        row_ids<DEG>(d.c2f, k0, v);
        row_ids<DEG>(d.c2n, k0, o);
#pragma unroll
        for (int i = 0; i < DEG; ++i) bo[i] = field(o[i] >= 0 ? o[i] : c);
#pragma unroll
        for (int i = 0; i < DEG; ++i) add(v[i], o[i], bo[i]);
    }
    else
        for (int32_t k = k0; k < k0 + nk; ++k) add(d.c2f[k], d.c2n[k], field(d.c2n[k] >= 0 ? d.c2n[k] : c));
    const double invV = 1.0 / d.cvol[c];
    st3(F.J, c, V3(sum.x * invV, sum.y * invV, sum.z * invV));
}

template <int DEG, int NS>
__global__ void __launch_bounds__(kStatesThreads, DEG == 4 && NS == 0 ? 4 : 3) k_step_states(DevMesh d, Params P, StepFields F, const double *Phi, const double *PhiAdd,
                                                                   int32_t n_cell, int32_t n_face, const double *dt_part, int32_t n_part,
                                                                   double dt_max, double *dt_dev, HostBox *box, uint64_t ticket)
{
    // the larger of the staged face states (5 DEG per thread) and the reduction of the time step
    __shared__ double stage[kStatesThreads * (DEG > 0 ? 5 * DEG : 1)];
    const int32_t b = blockIdx.x;
    if (b < n_cell) states_role<DEG, NS>(d, P, F, near_block(d, b, 0, n_cell), stage);
    else if (b < n_cell + n_face) face_emf_role(d, F, Phi, PhiAdd, near_block(d, b, n_cell, n_face) * kStatesThreads + int32_t(threadIdx.x));
    else dt_role(dt_part, n_part, dt_max, dt_dev, stage, box, ticket);
}
// Dynamic LDS: the heavy edges' rows (fv.h) when there are any
template <int NS>
__global__ void __launch_bounds__(kRoleThreads) k_step_fluxes(DevMesh d, Params P, StepFields F, double *E, const int32_t *heavy, int32_t n_heavy,
                                                              int32_t hv, int32_t n_edge)
{
    extern __shared__ double shared[];
    const int32_t b = blockIdx.x;
    if (b < n_heavy) edge_emf_heavy<double>(d, P, F.Ef, F.uplus, P.cuct, heavy[b], nullptr, E, 1, shared, hv);
    else if (b < n_heavy + n_edge)
        edge_emf_light<double>(d, P, F.Ef, F.uplus, P.cuct, kLightMax,
                               near_block(d, b, n_heavy, n_edge) * kRoleThreads + int32_t(threadIdx.x), nullptr, E, 1);
    else flux_role<NS>(d, P, F, near_block(d, b, n_heavy + n_edge, int32_t(gridDim.x) - n_heavy - n_edge), shared);
}
template <int DEG, int NS>
__global__ void __launch_bounds__(kRoleThreads) k_step_update(DevMesh d, Params P, StepFields F, const double *dt_dev, SpW Us, int32_t n_cell,
                                                              const double *E, double *Phi)
{
    const int32_t b = blockIdx.x;
    if (b < n_cell) update_role<DEG, NS>(d, P, F, dt_dev, Us, near_block(d, b, 0, n_cell));
    else faraday_face(d, E, nullptr, dt_dev, 0.0, Phi, near_block(d, b, n_cell, int32_t(gridDim.x) - n_cell) * kRoleThreads + int32_t(threadIdx.x));
}
} // namespace mhdg

using namespace mhdg;

namespace
{
void chk(hipError_t e, const char *w)
{
    if (e != hipSuccess) throw std::runtime_error(std::string(w) + ": " + hipGetErrorString(e));
}
inline int blocks(int64_t n, int64_t per) { return static_cast<int>((n + per - 1) / per); }
// calls f with the row length of the mesh's cells (0: rows of varying length) and the ion count (0: more than two) as
// template arguments
template <class Fn> void by_shape(int32_t cdeg, int32_t ns, Fn f)
{
    auto with_ns = [&](auto deg) {
        if (ns == 2) f(deg, std::integral_constant<int, 2>{});
        else f(deg, std::integral_constant<int, 0>{});
    };
    if (cdeg == 4) with_ns(std::integral_constant<int, 4>{});
    else if (cdeg == 6) with_ns(std::integral_constant<int, 6>{});
    else with_ns(std::integral_constant<int, 0>{});
}
} // namespace

#define LAUNCH(NAME, ...)                                                                                                    \
    do                                                                                                                       \
    {                                                                                                                        \
        prof_begin(NAME);                                                                                                    \
        hipLaunchKernelGGL(__VA_ARGS__);                                                                                     \
        prof_end();                                                                                                          \
    } while (0)

StepFields mhdg_ctx::step_fields(double *Bt, double *up, double *cur, double *al)
{
    const size_t F = nf, C = nc, ns = size_t(P.ns);
    auto D = [&](size_t n) { return static_cast<double *>(alloc(n * sizeof(double))); };
    StepFields o = sf; // the face tables
    o.rs = step_row(P.ns);
    o.ns = P.ns;
    o.rec = D(size_t(o.rs) * C);
    chk(hipMemset(o.rec, 0, size_t(o.rs) * C * 8), "memset");
    o.Btot = Bt; o.uplus = up; o.J = cur; o.alpha = al;
    o.FS = D(5 * ns * c2f_nnz);
    o.FA = D(5 * ns * F);
    o.Ef = D(4 * F);
    return o;
}

StepRun mhdg_ctx::resident_run()
{
    StepRun r{};
    for (int s = 0; s < P.ns; ++s) r.U[s] = U[s];
    r.Phi = Phi; r.F = sf; r.E = E_expl; r.dt_part = dt_part; r.dt_dev = dt_dev;
    return r;
}

void mhdg_ctx::step_build()
{
    const size_t F = nf;
    sf = step_fields(Btot, uplus, J, alpha);
    int2 *fent = static_cast<int2 *>(alloc(F * sizeof(int2)));
    int8_t *fcls = static_cast<int8_t *>(alloc(F));
    hipLaunchKernelGGL(k_face_entries, dim3(blocks(nf, 256)), dim3(256), 0, stream, d, fent, fcls);
    check_launch("face entries");
    sf.fent = fent; sf.fcls = fcls;
}

void mhdg_ctx::launch_prepare(const StepRun &x)
{
    SpC Uc{};
    for (int s = 0; s < P.ns; ++s) Uc.p[s] = x.U[s];
    by_shape(cdeg, P.ns, [&](auto deg, auto ns) {
        constexpr int DEG = decltype(deg)::value;
        if constexpr (decltype(ns)::value == 2)
            LAUNCH("prepare", k_step_prepare2<DEG>, dim3(blocks(nc, 256)), dim3(256), 0, stream, d, P, Uc, static_cast<const double *>(x.Phi),
                   static_cast<const double *>(Badd), x.F, x.dt_part);
        else
            LAUNCH("prepare", k_step_prepare_many<DEG>, dim3(blocks(nc, 256 / P.ns)), dim3(256), 0, stream, d, P, Uc,
                   static_cast<const double *>(x.Phi), static_cast<const double *>(Badd), x.F, x.dt_part);
    });
}

void mhdg_ctx::launch_states(const StepRun &x, int32_t n_face, double *dt_out, double dt_max)
{
    const int32_t n_cell = blocks(nc, kStatesThreads / P.ns), n_part = blocks(nc, P.ns == 2 ? 256 : 256 / P.ns);
    by_shape(cdeg, P.ns, [&](auto deg, auto ns) {
        LAUNCH("states", (k_step_states<decltype(deg)::value, decltype(ns)::value>), dim3(n_cell + n_face + (dt_out ? 1 : 0)),
               dim3(kStatesThreads), 0, stream, d, P, x.F, static_cast<const double *>(x.Phi), static_cast<const double *>(PhiAdd), n_cell, n_face,
               static_cast<const double *>(x.dt_part), n_part, dt_max, dt_out, dt_box, ticket);
    });
}

void mhdg_ctx::launch_current(const StepRun &x)
{
    by_shape(cdeg, P.ns, [&](auto deg, auto) {
        LAUNCH("current", k_step_current<decltype(deg)::value>, dim3(blocks(nc, kRoleThreads)), dim3(kRoleThreads), 0, stream, d, x.F);
    });
}

double mhdg_ctx::explicit_stage(const StepRun &x, double dt_max, StageEnd end)
{
    // nothing before this wrote U or Phi (only derived fields), so the state is unchanged when it throws
    auto checked = [](double v) {
        if (!std::isfinite(v) || v <= 0) throw std::runtime_error("invalid time step");
        return v;
    };
    launch_prepare(x);
    // Strang split of the ions' gyration (Solver.cpp:237-241): half a step, then prepare again.  The rotation changes
    // U, so the time step is checked first, as the reference throws before it touches the state (Solver.cpp:236).
    const bool split = P.induce_coeff > 0 && P.lorentz;
    double gdt = 0;
    if (split)
    {
        LAUNCH("dt_final", k_dt_final<double>, dim3(1), dim3(256), 0, stream, static_cast<const double *>(x.dt_part), blocks(nc, 256), dt_max, x.dt_dev);
        d2h(&gdt, x.dt_dev, 8);
        checked(gdt);
        LAUNCH("gyrate", k_gyrate, dim3(blocks(nc, 256)), dim3(256), 0, stream, d, P, x.U[0], x.U[1], static_cast<const double *>(x.F.Btot),
               static_cast<const double *>(x.dt_dev), 0.5);
        launch_prepare(x);
    }
    ++ticket;
    launch_states(x, blocks(nf, kStatesThreads), split ? nullptr : x.dt_dev, dt_max);
    const int n_edge = blocks(ne, kRoleThreads), n_flux = blocks(nf, kRoleThreads / P.ns);
    const size_t lds = sizeof(double) * std::max<size_t>(5 * kRoleThreads, n_heavy ? kEmfHeavyRows * size_t(max_valence) : 0);
    auto kflux = P.ns == 2 ? k_step_fluxes<2> : k_step_fluxes<0>;
    LAUNCH("fluxes", kflux, dim3(n_heavy + n_edge + n_flux), dim3(kRoleThreads), lds, stream, d, P, x.F, x.E, static_cast<const int32_t *>(heavy),
           n_heavy, max_valence, n_edge);
    check_launch("explicit stage");
    if (end == kStageNone) return 0.0;
    if (!split) gdt = checked(wait_box(dt_box)[0]); // written while the states were formed
    SpW Us{};
    for (int s = 0; s < P.ns; ++s) Us.p[s] = x.U[s];
    const int n_cell = blocks(nc, kRoleThreads / P.ns), n_face = end == kStageState ? blocks(nf, kRoleThreads) : 0;
    by_shape(cdeg, P.ns, [&](auto deg, auto ns) {
        LAUNCH("update", (k_step_update<decltype(deg)::value, decltype(ns)::value>), dim3(n_cell + n_face), dim3(kRoleThreads), 0, stream, d, P,
               x.F, static_cast<const double *>(x.dt_dev), Us, n_cell, static_cast<const double *>(x.E), x.Phi);
    });
    check_launch("cell update");
    return gdt;
}

void mhdg_ctx::get_record(int32_t first, int32_t n, double *host)
{
    double *dense = stage(7, size_t(n) * size_t(nc));
    hipLaunchKernelGGL(k_rec_get, dim3(blocks(int64_t(n) * nc, 256)), dim3(256), 0, stream, static_cast<const double *>(sf.rec), sf.rs, first, n,
                       nc, dense);
    check_launch("record");
    d2h(host, dense, size_t(n) * size_t(nc) * 8);
}
