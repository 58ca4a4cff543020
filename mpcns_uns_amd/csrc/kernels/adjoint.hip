// Reverse mode (adjoint) of the explicit stage of the Mercury step (MercuryUns/driver/Solver.cpp:228-277 with
// the Hall solve inactive): the gradient of the shell magnetic energy after n steps with respect to the
// initial state, the background flux and field, the free-stream states and the imposed inflow EMF.
//
// The forward sweep is the resident step's own (explicit_step.hip) on fields of its own, and keeps the state (U, Phi) of
// every step; the reverse sweep recomputes a step's fields from it (the last step's are still there) and runs the
// transposed kernels, written out by hand from the branch that the values take (limiters, upwinding, floors, argmax, the
// CFL minimum; a tie takes the operand that the value computation keeps).  Five launches a step:
//   update      edges: Faraday and the UCT sum | cells: the update and its sources | the cell that sets the time step
//   faces       Rusanov fluxes | face EMF candidates | the time step's adjoint
//   gradients   limited gradients: adjoints of the face states -> of the primitives of the stencil
//   cells       the neighbours' parts, current, CFL cell, u+, primitive recovery, field reconstruction
//   flux        the reconstruction's parts of the face flux
// Sums run in a fixed order (adjoint.h), so the result is deterministic.
//
// Measured at 484k tetrahedra, five steps (one MI355X): a reverse step takes 890 us, its fields' recomputation 350; with
// local Jacobians from forward-mode columns and 20 adjoints per (cell, face) entry and ion instead of 5 it took 5100 and
// 520, and the host summed block parts five times a step.  The whole call, gradients in host memory: 36.3 -> 13.1 ms.
// update 283 us (two-thirds of it the edges, bound by their chains of dependent gathers at three waves per SIMD; in two
// launches 216 + 105), faces 224 and cells 174 (4-5 TB/s of slots and gathered rows), gradients 199 (its FP64 instructions:
// two divisions per face, primitive and ion, as the forward).
#include <algorithm>
#include <stdexcept>
#include <string>
#include <type_traits>

#include "ctx.h"
#include "step_cell.h"

namespace mhdg
{
namespace
{
constexpr int kAdjNs = 2;       // species of the adjoint (the two Mercury ions); a cell's or face's two threads are neighbours
constexpr int kAdjThreads = 256;
constexpr int kGradThreads = 128; // 20 KB of face states staged per block on tetrahedra
constexpr int kHeavyRows = 7;     // doubles staged per face of a high-valence edge (and one int)

// sums of v over the block's threads of the same parity (the ion of a two-thread entity), K values each, added to
// part[K * ion + j]; sh holds blockDim doubles
template <int K> __device__ void add_by_ion(const double (&v)[K], double *sh, double *part)
{
    const int t = threadIdx.x;
    for (int j = 0; j < K; ++j)
    {
        __syncthreads();
        sh[t] = v[j];
        __syncthreads();
        for (int s = blockDim.x / 2; s > 1; s >>= 1)
        {
            if (t < s) sh[t] += sh[t + s];
            __syncthreads();
        }
        if (t < kAdjNs) part[K * t + j] += sh[t];
    }
}
// sum over the block's threads, on thread 0
__device__ double block_sum(double v, double *sh)
{
    const int t = threadIdx.x;
    __syncthreads();
    sh[t] = v;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1)
    {
        if (t < s) sh[t] += sh[t + s];
        __syncthreads();
    }
    return sh[0];
}

// M^-1 b of the reconstruction's symmetric matrix M = sum |A| n n^T (upper triangle), zero where the reconstruction is
// (Reconstruct.cpp:11-45): with it the transpose of b_c = cell_vector(flux) is d(b . b_c) / d flux_f = n_f . M^-1 b
__device__ __forceinline__ V3 normal_solve(const double (&M)[6], const V3 &b)
{
    const double c0 = M[3] * M[5] - M[4] * M[4], c1 = M[2] * M[4] - M[1] * M[5], c2 = M[1] * M[4] - M[2] * M[3];
    const double det = M[0] * c0 + M[1] * c1 + M[2] * c2;
    const double sc = mx(mx(mx(M[0], M[3]), M[5]), 1e-300);
    if (fabs(det) < 1e-12 * sc * sc * sc) return V3();
    const double inv = 1.0 / det, c3 = M[0] * M[5] - M[2] * M[2], c4 = M[1] * M[2] - M[0] * M[4], c5 = M[0] * M[3] - M[1] * M[1];
    return V3(inv * (c0 * b.x + c1 * b.y + c2 * b.z), inv * (c1 * b.x + c3 * b.y + c4 * b.z), inv * (c2 * b.x + c4 * b.y + c5 * b.z));
}

// Floors of the update (Solver.cpp:171-191) transposed: b = (d floors(q) / dq)^T b
__device__ __forceinline__ void floors_adjoint(const Params &P, const double (&q)[5], double (&b)[5])
{
    const double ke = q[0] > 0 ? 0.5 * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]) / q[0] : 0.0;
    if (!(q[0] >= P.rho_floor))
    {
        for (int m = 0; m < 5; ++m) b[m] = 0.0;
        return;
    }
    if (!((P.gamma - 1.0) * (q[4] - ke) < P.p_floor)) return;
    // to_cons(to_prim(q)) with the pressure at its floor: the energy follows the kinetic part; the momenta are kept
    const double u = q[1] / q[0], v = q[2] / q[0], w = q[3] / q[0];
    const double uu = u * u + v * v + w * w;
    if (!((P.gamma - 1.0) * (q[4] - 0.5 * q[0] * uu) < P.p_floor)) return;
    b[0] -= 0.5 * uu * b[4];
    b[1] += u * b[4]; b[2] += v * b[4]; b[3] += w * b[4];
    b[4] = 0.0;
}

// ------------------------------------------------------------------------------------------------------------ roles
// Faraday (Common/induction/Faraday.cpp:15-36) and the UCT sum of an edge with the boundary EMF (IdealEMF.cpp:59-128,
// Solver.cpp:162-167), transposed.  Eb_e = -dt sum over the active faces of sgn Phib_f; the same sum times E_e is the
// edge's part of d/d dt.  -> the edge's EMF adjoint for its UCT sum (zero: none), parts[0] dt, [1..3] the inflow EMF.
struct EdgeSeed { double Eb; double part[4]; };
__device__ __forceinline__ EdgeSeed edge_seed(const DevMesh &d, int32_t e, double acc, double dt, const double *E)
{
    EdgeSeed o{-dt * acc, {-E[e] * acc, 0.0, 0.0, 0.0}};
    const int8_t mode = d.emode[e];
    if (mode == 2)
    {
        const V3 t = L3(d.evec, e);
        o.part[1] = o.Eb * t.x; o.part[2] = o.Eb * t.y; o.part[3] = o.Eb * t.z;
    }
    if (mode == 1 || mode == 2) o.Eb = 0.0;
    return o;
}
__device__ __forceinline__ double flux_bar(const DevMesh &d, const AdjFields &G, int32_t v)
{
    const int32_t f = pid(v);
    return G.all_active || d.fL[f] >= 0 || d.fR[f] >= 0 ? psg(v) * G.Phib[f] : 0.0;
}
// (l1, l2) = uct_solve(M11, M12, M22, g1, g2) (fv.h) transposed: sb = (d(l1, l2) / d in)^T (l1b, l2b)
__device__ __forceinline__ void uct_solve_adjoint(const double (&in)[5], double l1, double l2, double l1b, double l2b, double (&sb)[5])
{
    const double tr = in[0] + in[2], eps = 1e-14 * tr, a = in[0] + eps, b = in[2] + eps, det = a * b - in[1] * in[1];
    for (int q = 0; q < 5; ++q) sb[q] = 0.0;
    if (!(tr > 0 && det > 0)) return;
    const double inv = 1.0 / det, n1 = l1b * inv, n2 = l2b * inv, db = -(n1 * l1 + n2 * l2);
    const double ab = in[4] * n2 + b * db, bb = in[3] * n1 + a * db, eb = 1e-14 * (ab + bb);
    sb[0] = ab + eb;
    sb[1] = -(in[4] * n1 + in[3] * n2) - 2.0 * in[1] * db;
    sb[2] = bb + eb;
    sb[3] = b * n1 - in[1] * n2;
    sb[4] = a * n2 - in[1] * n1;
}
// One face of the edge's UCT sum: the direction m, aef = max_k |u_k . m| (first strict maximum, of cell k, kept as ~k for a
// negative u_k . m; kNoCell: none), a, b: sig times the normal's components in the edge's plane; q = aef (a, b)
constexpr int32_t kNoCell = INT32_MIN;
struct UctFace { V3 m; double aef, sig, a, b; int32_t k; };
__device__ __forceinline__ UctFace uct_geometry(const DevMesh &d, int32_t f, int32_t e, const V3 &th, const V3 &e1, const V3 &e2)
{
    UctFace o;
    V3 nrm;
    face_dirs(d, f, e, th, o.m, nrm);
    o.sig = dot(th, cross(o.m, nrm));
    o.a = o.sig * dot(nrm, e1);
    o.b = o.sig * dot(nrm, e2);
    o.aef = 0.0; o.k = kNoCell;
    return o;
}
__device__ __forceinline__ void uct_max(UctFace &o, int32_t k, const V3 &u)
{
    const double x = dot(u, o.m);
    if (o.aef < fabs(x)) { o.aef = fabs(x); o.k = x < 0 ? ~k : k; }
}
// adjoint of aef, with the face's eF row written; w, pf: the face's weight and Phi / |A|
__device__ __forceinline__ double uct_face_adjoint(double w, double pf, double A, double aef, double sig, double a, double b, double l1,
                                                   double l2, double Eub, double Eb, const V3 &t, const double (&sb)[5], double *eF)
{
    const double qa = aef * a, qb = aef * b;
    const double omega = w * (1.0 - (qa * l1 + qb * l2)), omb = Eub * aef * sig * pf;
    const double qab = -omb * w * l1 + 2.0 * w * qa * sb[0] + w * qb * sb[1] + w * sb[3];
    const double qbb = -omb * w * l2 + w * qa * sb[1] + 2.0 * w * qb * sb[2] + w * sb[4];
    double2 *o = reinterpret_cast<double2 *>(eF);
    o[0] = make_double2(Eb * w * t.x, Eb * w * t.y);
    o[1] = make_double2(Eb * w * t.z, Eub * omega * aef * sig / A);
    return Eub * omega * sig * pf + qab * a + qbb * b;
}

// One edge per thread.  The usual valence keeps the row's cell velocities and per-face terms in registers; longer rows
// walk them again, their cells' sums in the slots.
__device__ __forceinline__ void edge_adjoint_light(const DevMesh &d, const StepFields &F, const AdjFields &G, double cuct, double dt,
                                                   const double *E, int32_t e, double (&part)[4])
{
    if (e >= d.ne) return;
    const int32_t f0 = d.e2f_ptr[e], nf = d.e2f_ptr[e + 1] - f0;
    if (nf > kLightMax) return;
    const int32_t c0 = d.ec_ptr[e], nc = d.ec_ptr[e + 1] - c0;
    double *eC = G.eC + 3 * size_t(c0), *eF = G.eF + 4 * size_t(f0);
    const bool fast = nf <= kEmfFast && nc <= kEmfFast;
    int32_t vid[kEmfFast], cid[kEmfFast];
    double acc = 0.0;
    bool any_fluid = false;
    if (fast)
    {
#pragma unroll
        for (int i = 0; i < kEmfFast; ++i)
        {
            if (i < nf) vid[i] = d.e2f[f0 + i];
            if (i < nc) cid[i] = d.ec_cell[c0 + i];
        }
#pragma unroll
        for (int i = 0; i < kEmfFast; ++i)
        {
            if (i < nf) acc += flux_bar(d, G, vid[i]);
            if (i < nc) any_fluid |= d.mat[cid[i]] == 0;
        }
    }
    else
    {
        for (int32_t i = 0; i < nf; ++i) acc += flux_bar(d, G, d.e2f[f0 + i]);
        for (int32_t k = 0; k < nc && !any_fluid; ++k) any_fluid = d.mat[d.ec_cell[c0 + k]] == 0;
    }
    const EdgeSeed seed = edge_seed(d, e, acc, dt, E);
    for (int q = 0; q < 4; ++q) part[q] = seed.part[q];
    const double Eb = seed.Eb, L = d.elen[e];
    if (!(Eb != 0.0 && nf > 0 && L > 0 && any_fluid))
    {
        for (int32_t i = 0; i < 4 * nf; ++i) eF[i] = 0.0;
        for (int32_t k = 0; k < 3 * nc; ++k) eC[k] = 0.0;
        return;
    }
    const V3 t = L3(d.evec, e), th = (1.0 / L) * t;
    V3 e1, e2;
    plane_basis(th, e1, e2);
    const double Eub = 2.0 * cuct * L * Eb;
    double M[5] = {0, 0, 0, 0, 0}, l1, l2, l1b = 0, l2b = 0, sb[5];
    // the face's terms of the 2x2 system and of its multipliers' adjoints, which do not depend on the solution
    auto sums = [&](const UctFace &u, int32_t f, double w) {
        const double qa = u.aef * u.a, qb = u.aef * u.b, x = Eub * u.aef * u.sig * F.Ef[4 * size_t(f) + 3] * w;
        M[0] += w * qa * qa; M[1] += w * qa * qb; M[2] += w * qb * qb; M[3] += w * qa; M[4] += w * qb;
        l1b -= x * qa;
        l2b -= x * qb;
    };
    auto adjoint = [&](const UctFace &u, int32_t f, int32_t i) {
        return psg(u.k) * uct_face_adjoint(d.efw[f0 + i], F.Ef[4 * size_t(f) + 3], d.geo[4 * size_t(f) + 3], u.aef, u.sig, u.a, u.b, l1, l2, Eub,
                                           Eb, t, sb, eF + 4 * i);
    };
    if (fast)
    {
        // kept for the second pass: the maxima only (all terms of six faces, with the cells' velocities, spilled at three
        // waves per SIMD); the directions are formed again from cached rows
        double aef[kEmfFast];
        int32_t km[kEmfFast];
        {
            V3 uc[kEmfFast];
#pragma unroll
            for (int k = 0; k < kEmfFast; ++k)
                if (k < nc) uc[k] = L3(F.uplus, cid[k]);
#pragma unroll
            for (int i = 0; i < kEmfFast; ++i)
                if (i < nf)
                {
                    const int32_t f = pid(vid[i]);
                    UctFace u = uct_geometry(d, f, e, th, e1, e2);
#pragma unroll
                    for (int k = 0; k < kEmfFast; ++k)
                        if (k < nc) uct_max(u, k, uc[k]);
                    sums(u, f, d.efw[f0 + i]);
                    aef[i] = u.aef; km[i] = u.k;
                }
        }
        uct_solve(M[0], M[1], M[2], M[3], M[4], l1, l2);
        uct_solve_adjoint(M, l1, l2, l1b, l2b, sb);
        V3 ub[kEmfFast];
#pragma unroll
        for (int i = 0; i < kEmfFast; ++i)
            if (i < nf)
            {
                const int32_t f = pid(vid[i]);
                UctFace u = uct_geometry(d, f, e, th, e1, e2);
                u.aef = aef[i]; u.k = km[i];
                const double g = adjoint(u, f, i);
#pragma unroll
                for (int k = 0; k < kEmfFast; ++k)
                    if (pid(u.k) == k) ub[k] += g * u.m;
            }
#pragma unroll
        for (int k = 0; k < kEmfFast; ++k)
            if (k < nc) st3(eC, k, ub[k]);
        return;
    }
    auto face = [&](int32_t f) {
        UctFace u = uct_geometry(d, f, e, th, e1, e2);
        for (int32_t k = 0; k < nc; ++k) uct_max(u, k, L3(F.uplus, d.ec_cell[c0 + k]));
        return u;
    };
    for (int32_t k = 0; k < 3 * nc; ++k) eC[k] = 0.0;
    for (int32_t i = 0; i < nf; ++i)
    {
        const int32_t f = pid(d.e2f[f0 + i]);
        sums(face(f), f, d.efw[f0 + i]);
    }
    uct_solve(M[0], M[1], M[2], M[3], M[4], l1, l2);
    uct_solve_adjoint(M, l1, l2, l1b, l2b, sb);
    for (int32_t i = 0; i < nf; ++i)
    {
        const int32_t f = pid(d.e2f[f0 + i]);
        const UctFace u = face(f);
        const double g = adjoint(u, f, i);
        if (u.k != kNoCell)
        {
            double *o = eC + 3 * pid(u.k);
            o[0] += g * u.m.x; o[1] += g * u.m.y; o[2] += g * u.m.z;
        }
    }
}

// One high-valence edge per block (valence > kLightMax: the pole axes): the faces in parallel, each one's maximum over the
// cells read from LDS, the sums by one thread in face order, the cells' sums by a thread per cell in face order.
// sh: kHeavyRows rows of hv doubles and one of ints (hv at least the valence; more cells than that are read in place).
__device__ __forceinline__ void edge_adjoint_heavy(const DevMesh &d, const StepFields &F, const AdjFields &G, double cuct, double dt,
                                                   const double *E, int32_t e, double *sh, int32_t hv, double *part)
{
    double *x = sh, *y = sh + hv, *z = sh + 2 * hv, *sa = sh + 3 * hv, *sbv = sh + 4 * hv, *saef = sh + 5 * hv, *ssig = sh + 6 * hv;
    int32_t *sk = reinterpret_cast<int32_t *>(sh + kHeavyRows * hv); // UctFace::k
    __shared__ double s_r[9];
    const int32_t f0 = d.e2f_ptr[e], nf = d.e2f_ptr[e + 1] - f0;
    const int32_t c0 = d.ec_ptr[e], nc = d.ec_ptr[e + 1] - c0;
    const int32_t t0 = threadIdx.x, nt = blockDim.x;
    double *eC = G.eC + 3 * size_t(c0), *eF = G.eF + 4 * size_t(f0);
    for (int32_t i = t0; i < nf; i += nt) sa[i] = flux_bar(d, G, d.e2f[f0 + i]);
    bool any_fluid = false;
    for (int32_t k = 0; k < nc && !any_fluid; ++k) any_fluid = d.mat[d.ec_cell[c0 + k]] == 0;
    __syncthreads();
    if (t0 == 0)
    {
        double acc = 0.0;
        for (int32_t i = 0; i < nf; ++i) acc += sa[i];
        const EdgeSeed seed = edge_seed(d, e, acc, dt, E);
        s_r[0] = seed.Eb;
        part[0] = seed.part[0];
        for (int q = 1; q < 4; ++q) part[q] += seed.part[q];
    }
    __syncthreads();
    const double Eb = s_r[0], L = d.elen[e];
    if (!(Eb != 0.0 && L > 0 && any_fluid)) // the same for every thread
    {
        for (int32_t i = t0; i < 4 * nf; i += nt) eF[i] = 0.0;
        for (int32_t k = t0; k < 3 * nc; k += nt) eC[k] = 0.0;
        return;
    }
    const V3 t = L3(d.evec, e), th = (1.0 / L) * t;
    V3 e1, e2;
    plane_basis(th, e1, e2);
    const double Eub = 2.0 * cuct * L * Eb;
    const bool staged = nc <= hv;
    if (staged)
        for (int32_t k = t0; k < nc; k += nt)
        {
            const V3 u = L3(F.uplus, d.ec_cell[c0 + k]);
            x[k] = u.x; y[k] = u.y; z[k] = u.z;
        }
    __syncthreads();
    for (int32_t i = t0; i < nf; i += nt)
    {
        UctFace u = uct_geometry(d, pid(d.e2f[f0 + i]), e, th, e1, e2);
        if (staged)
            for (int32_t k = 0; k < nc; ++k) uct_max(u, k, V3(x[k], y[k], z[k]));
        else
            for (int32_t k = 0; k < nc; ++k) uct_max(u, k, L3(F.uplus, d.ec_cell[c0 + k]));
        sa[i] = u.a; sbv[i] = u.b; saef[i] = u.aef; ssig[i] = u.sig;
        sk[i] = u.k;
    }
    __syncthreads(); // the staged velocities are read
    for (int32_t i = t0; i < nf; i += nt)
    {
        x[i] = d.efw[f0 + i];
        y[i] = F.Ef[4 * size_t(pid(d.e2f[f0 + i])) + 3];
    }
    __syncthreads();
    if (t0 == 0)
    {
        double M[5] = {0, 0, 0, 0, 0}, l1, l2, l1b = 0, l2b = 0, sb[5];
        for (int32_t i = 0; i < nf; ++i)
        {
            const double w = x[i], qa = saef[i] * sa[i], qb = saef[i] * sbv[i];
            M[0] += w * qa * qa; M[1] += w * qa * qb; M[2] += w * qb * qb; M[3] += w * qa; M[4] += w * qb;
        }
        uct_solve(M[0], M[1], M[2], M[3], M[4], l1, l2);
        for (int32_t i = 0; i < nf; ++i)
        {
            const double q = Eub * saef[i] * ssig[i] * y[i] * x[i] * saef[i];
            l1b -= q * sa[i];
            l2b -= q * sbv[i];
        }
        uct_solve_adjoint(M, l1, l2, l1b, l2b, sb);
        s_r[1] = l1; s_r[2] = l2;
        for (int q = 0; q < 5; ++q) s_r[3 + q] = sb[q];
    }
    __syncthreads();
    const double l1 = s_r[1], l2 = s_r[2], sb[5] = {s_r[3], s_r[4], s_r[5], s_r[6], s_r[7]};
    for (int32_t i = t0; i < nf; i += nt)
    {
        const int32_t f = pid(d.e2f[f0 + i]);
        V3 m, nrm;
        face_dirs(d, f, e, th, m, nrm);
        const double g = psg(sk[i]) * uct_face_adjoint(x[i], y[i], d.geo[4 * size_t(f) + 3], saef[i], ssig[i], sa[i], sbv[i], l1, l2, Eub, Eb, t, sb, eF + 4 * i);
        sk[i] = pid(sk[i]); // kNoCell becomes INT32_MAX, no cell's
        x[i] = g * m.x; y[i] = g * m.y; z[i] = g * m.z; // this thread's entries only until the barrier
    }
    __syncthreads();
    for (int32_t k = t0; k < nc; k += nt)
    {
        V3 s;
        for (int32_t i = 0; i < nf; ++i)
            if (sk[i] == k) s += V3(x[i], y[i], z[i]);
        st3(eC, k, s);
    }
}

// Forward Euler update with floors, flux divergence and Lorentz sources, transposed: Ub (in: adjoint of U^{n+1}; out: its
// part through the update), the sources' parts of W, J, B_tot, the right-hand side's adjoint; thread (cell, ion).
// -> the thread's part of d/d dt
template <int DEG>
__device__ __forceinline__ double update_adjoint_role(const DevMesh &d, const Params &P, const StepFields &F, const AdjFields &G, const SpC &Us,
                                                      const SpW &Ub, double dt, int32_t block)
{
    const int32_t t = threadIdx.x, s = t & 1, c = block * (kAdjThreads / kAdjNs) + (t >> 1);
    if (c >= d.nc) return 0.0;
    double dtb = 0.0, rb[5] = {0, 0, 0, 0, 0}, wb[5] = {0, 0, 0, 0, 0}, neb = 0.0, nsb = 0.0;
    V3 jb, bb;
    const double V = d.cvol[c];
    const double *row = F.rec + 16 * size_t(c), *W = row + 5 * s;
    const bool fluid = d.mat[c] == 0; // the same for the cell's two threads
    if (fluid)
    {
        double rhs[5], q[5], qb[5];
        cell_rhs<DEG>(d, P, F, c, s, kAdjNs, row, V, dt, rhs);
        const double *u = Us.p[s] + 5 * size_t(c);
        double *ub = Ub.p[s] + 5 * size_t(c);
        for (int m = 0; m < 5; ++m) { q[m] = u[m] + dt * rhs[m]; qb[m] = ub[m]; }
        floors_adjoint(P, q, qb);
        for (int m = 0; m < 5; ++m)
        {
            ub[m] = qb[m];
            rb[m] = dt * qb[m];
            dtb += rhs[m] * qb[m];
        }
        if (P.lorentz)
        {
            // S = k chi' J x B, chi' = n_s / D, D = sqrt(n_e^2 + floor^2); out += S, energy += u . S + dt S^2 / (2 rho)
            const V3 Jc = L3(F.J, c), B = L3(F.Btot, c), C = cross(Jc, B), vel(W[1], W[2], W[3]);
            const double ns = ion_density(P, s, W[0]), ne = ion_density(P, 0, row[0]) + ion_density(P, 1, row[5]);
            const double D = sqrt(ne * ne + P.ne_floor * P.ne_floor), ws = ns / D;
            const V3 S = (P.inver_MA2 * ws) * C;
            V3 Sb(rb[1] + rb[4] * vel.x, rb[2] + rb[4] * vel.y, rb[3] + rb[4] * vel.z);
            wb[1] = rb[4] * S.x; wb[2] = rb[4] * S.y; wb[3] = rb[4] * S.z;
            const double rho = mx(W[0], 0.0);
            if (rho > 1e-30)
            {
                const double SS = dot(S, S), h = 0.5 * rb[4] / rho;
                Sb += (2.0 * h * dt) * S;
                wb[0] -= h * dt * SS / rho;
                dtb += h * SS;
            }
            const double wsb = P.inver_MA2 * dot(Sb, C);
            const V3 Cb = (P.inver_MA2 * ws) * Sb;
            jb = cross(B, Cb);
            bb = cross(Cb, Jc);
            if (D > 0)
            {
                nsb = wsb / D;
                neb = -wsb * ws * ne / (D * D);
            }
        }
    }
    // the two ions' parts of n_e, J and B_tot
    neb += __shfl_xor(neb, 1);
    jb += V3(__shfl_xor(jb.x, 1), __shfl_xor(jb.y, 1), __shfl_xor(jb.z, 1));
    bb += V3(__shfl_xor(bb.x, 1), __shfl_xor(bb.y, 1), __shfl_xor(bb.z, 1));
    if (fluid && W[0] >= 0) wb[0] += (nsb + neb) / P.M_s[s] * P.M_ref;
    for (int m = 0; m < 5; ++m)
    {
        G.rv[10 * size_t(c) + 5 * s + m] = rb[m] / V;
        G.Wb[10 * size_t(c) + 5 * s + m] = wb[m];
    }
    if (s == 0) st3(G.Jv, c, (1.0 / V) * jb);
    else st3(G.Btb, c, bb);
    return dtb;
}

// The first cell whose CFL step is dt (the blocks' minima in part), and the derivatives of its step by its primitives
// and field (MercurySources.cpp:104-145; the ion, and the branches, that give the minimum)
__device__ void dt_cell_role(const DevMesh &d, const Params &P, const StepFields &F, const AdjFields &G, const double *part, int32_t n_part,
                             double dt)
{
    __shared__ int32_t s_b, s_c;
    const int32_t t = threadIdx.x;
    if (t == 0) s_b = s_c = INT32_MAX;
    __syncthreads();
    for (int32_t i = t; i < n_part; i += kAdjThreads)
        if (part[i] == dt) { atomicMin(&s_b, i); break; }
    __syncthreads();
    auto field = [&](int32_t c, const double *(&w)[kMaxSpecies]) {
        for (int s = 0; s < kAdjNs; ++s) w[s] = F.rec + 16 * size_t(c) + 5 * s;
        return L3(F.Btot, c);
    };
    if (s_b != INT32_MAX)
    {
        const int32_t c = s_b * 256 + t;
        const double *w[kMaxSpecies];
        if (c < d.nc && d.mat[c] == 0)
        {
            const V3 b = field(c, w);
            if (cell_dt<double>(d, P, c, w, b, 0) == dt) atomicMin(&s_c, c);
        }
    }
    __syncthreads();
    if (t != 0) return;
    const int32_t c = s_c;
    if (c == INT32_MAX)
    {
        G.dt_cell[0] = -1;
        ++G.dt_cell[1];
        return;
    }
    const double *w[kMaxSpecies];
    const V3 b = field(c, w);
    const double k = P.inver_MA2, rsum = w[0][0] + w[1][0], rt = mx(rsum, P.rho_floor_dt), vA2 = k * dot(b, b) / rt;
    double denom[kAdjNs] = {0, 0};
    int ion = 0;
    double best = __builtin_inf();
    for (int s = 0; s < kAdjNs; ++s)
    {
        const double cs2 = P.gamma * w[s][4] / mx(w[s][0], 1e-30);
        for (int32_t i = d.c2f_ptr[c]; i < d.c2f_ptr[c + 1]; ++i)
        {
            double A;
            const V3 n = geo_normal(d, pid(d.c2f[i]), A);
            const double vAn2 = k * dot(b, n) * dot(b, n) / rt, term = cs2 + vA2;
            denom[s] += (fabs(w[s][1] * n.x + w[s][2] * n.y + w[s][3] * n.z) + sqrt(0.5 * (term + sqrt(mx(0.0, term * term - 4 * cs2 * vAn2))))) * A;
        }
        const double x = P.cfl * d.cvol[c] / denom[s];
        if (denom[s] > 0 && x < best) { best = x; ion = s; }
    }
    const double *q = w[ion];
    const double rs = mx(q[0], 1e-30), cs2 = P.gamma * q[4] / rs, db = -best / denom[ion];
    double cs2b = 0, vA2b = 0, rtb = 0;
    V3 ub, bb;
    for (int32_t i = d.c2f_ptr[c]; i < d.c2f_ptr[c + 1]; ++i)
    {
        double A;
        const V3 n = geo_normal(d, pid(d.c2f[i]), A);
        const double bn = dot(b, n), vAn2 = k * bn * bn / rt, term = cs2 + vA2, disc = mx(0.0, term * term - 4 * cs2 * vAn2), sq = sqrt(disc);
        const double cf = sqrt(0.5 * (term + sq)), un = q[1] * n.x + q[2] * n.y + q[3] * n.z;
        const double xb = cf > 0 ? 0.5 * (0.5 * db * A / cf) : 0.0, discb = sq > 0 && disc > 0 ? 0.5 * xb / sq : 0.0;
        const double termb = xb + 2.0 * term * discb, vAnb = -4.0 * cs2 * discb;
        cs2b += termb - 4.0 * vAn2 * discb;
        vA2b += termb;
        bb += (2.0 * k * bn / rt * vAnb) * n;
        rtb -= vAn2 * vAnb / rt;
        ub += ((un < 0 ? -db : db) * A) * n;
    }
    bb += (2.0 * k / rt * vA2b) * b;
    rtb -= vA2 * vA2b / rt;
    double *o = G.dtb + 1;
    for (int m = 0; m < 10; ++m) o[m] = 0.0;
    if (!(rsum < P.rho_floor_dt)) o[0] = o[5] = rtb;
    double *oi = o + 5 * ion;
    if (!(q[0] < 1e-30)) oi[0] -= cs2 / rs * cs2b;
    oi[1] = ub.x; oi[2] = ub.y; oi[3] = ub.z;
    oi[4] = P.gamma / rs * cs2b;
    o[10] = bb.x; o[11] = bb.y; o[12] = bb.z;
    G.dt_cell[0] = c;
}

// Rusanov flux (Common/physics/Euler.h:29-49) transposed: Lb, Rb = (dF/dL)^T Fb, (dF/dR)^T Fb
__device__ __forceinline__ void rusanov_adjoint(const Prim &L, const Prim &R, const V3 &n, double gamma, const double (&Fb)[5], double (&Lb)[5],
                                                double (&Rb)[5])
{
    const double unL = L.u * n.x + L.v * n.y + L.w * n.z, unR = R.u * n.x + R.v * n.y + R.w * n.z;
    const double cL = sqrt(gamma * L.p / L.rho), cR = sqrt(gamma * R.p / R.rho);
    const double sL = fabs(unL) + cL, sR = fabs(unR) + cR, s = mx(sL, sR);
    const double g1 = 1.0 / (gamma - 1.0);
    double UL[5], UR[5];
    to_cons(L, gamma, UL);
    to_cons(R, gamma, UR);
    double sb = 0.0;
    for (int m = 0; m < 5; ++m) sb -= 0.5 * Fb[m] * (UR[m] - UL[m]);
    auto side = [&](const Prim &w, double un, double c, double E, double h, double speed, double (&o)[5]) {
        // flux with adjoint Fb / 2, conserved state with h Fb, speed |un| + c with `speed`
        const V3 u(w.u, w.v, w.w), Gm(0.5 * Fb[1], 0.5 * Fb[2], 0.5 * Fb[3]);
        const double G0 = 0.5 * Fb[0], G4 = 0.5 * Fb[4], Gu = dot(Gm, u), Eb = un * G4 + h * Fb[4];
        const double unb = w.rho * (G0 + Gu) + G4 * (E + w.p) + (un < 0 ? -speed : speed);
        o[0] = un * (G0 + Gu) + h * (Fb[0] + 2.0 * Gu) + 0.5 * dot(u, u) * Eb;
        const V3 ub = (w.rho * (un + 2.0 * h)) * Gm + (w.rho * Eb) * u + unb * n;
        o[1] = ub.x; o[2] = ub.y; o[3] = ub.z;
        o[4] = dot(Gm, n) + un * G4 + g1 * Eb;
        if (speed != 0.0 && c > 0)
        {
            o[0] -= 0.5 * speed * c / w.rho;
            o[4] += 0.5 * speed * gamma / (c * w.rho);
        }
    };
    const bool right = sL < sR;
    side(L, unL, cL, UL[4], 0.5 * s, right ? 0.0 : sb, Lb);
    side(R, unR, cR, UR[4], -0.5 * s, right ? sb : 0.0, Rb);
}

// Face fluxes transposed: thread (face, ion).  Replaces the face states of the face's entries by their adjoints and adds
// the free stream's part to the block's.
__device__ __forceinline__ void flux_adjoint_role(const DevMesh &d, const Params &P, const StepFields &F, const AdjFields &G, int32_t block,
                                                  double *sh)
{
    const int32_t t = threadIdx.x, s = t & 1, f = block * (kAdjThreads / kAdjNs) + (t >> 1);
    double fsb[5] = {0, 0, 0, 0, 0};
    bool inflow = false;
    if (f < d.nf)
    {
        const int2 e = F.fent[f];
        const int8_t cls = F.fcls[f];
        double Lb[5] = {0, 0, 0, 0, 0}, Rb[5] = {0, 0, 0, 0, 0};
        double *qL = F.FS + 5 * (size_t(e.x < 0 ? 0 : e.x) * kAdjNs + s), *qR = F.FS + 5 * (size_t(e.y < 0 ? 0 : e.y) * kAdjNs + s);
        if (cls != kFluxNone)
        {
            const int32_t l = d.fL[f], r = d.fR[f];
            double A, Fb[5] = {0, 0, 0, 0, 0};
            const V3 n = geo_normal(d, f, A);
            // the cell that sees the face outward loses the flux
            if (e.x >= 0)
                for (int m = 0; m < 5; ++m) Fb[m] -= G.rv[10 * size_t(l) + 5 * s + m];
            if (e.y >= 0)
                for (int m = 0; m < 5; ++m) Fb[m] += G.rv[10 * size_t(r) + 5 * s + m];
            bool nz = false;
            for (int m = 0; m < 5; ++m) { Fb[m] *= A; nz = nz || Fb[m] != 0.0; }
            auto state = [](const double *q) { return Prim{q[0], q[1], q[2], q[3], q[4]}; };
            if (nz && cls == kFluxInner) rusanov_adjoint(state(qL), state(qR), n, P.gamma, Fb, Lb, Rb);
            else if (nz)
            {
                const bool left = cls == kFluxLeft;
                const int8_t kind = d.kind[f];
                const V3 no = (left ? 1.0 : -1.0) * n;
                const Prim in = state(left ? qL : qR);
                double fs[5];
                for (int m = 0; m < 5; ++m) fs[m] = P.fs[s][m];
                const Prim gh = ghost_state(kind, s, in, no, fs);
                double ib[5], gb[5];
                if (left) rusanov_adjoint(in, gh, n, P.gamma, Fb, ib, gb);
                else rusanov_adjoint(gh, in, n, P.gamma, Fb, gb, ib);
                if (kind == kInflow)
                {
                    inflow = true;
                    for (int m = 0; m < 5; ++m) fsb[m] = gb[m];
                }
                else if (!(kind == kWall && s == 1)) // the ghost is the cell's own state, mirrored at a wall
                {
                    if (kind == kWall)
                    {
                        const double w = 2.0 * (no.x * gb[1] + no.y * gb[2] + no.z * gb[3]);
                        gb[1] -= w * no.x; gb[2] -= w * no.y; gb[3] -= w * no.z;
                    }
                    for (int m = 0; m < 5; ++m) ib[m] += gb[m];
                }
                for (int m = 0; m < 5; ++m) (left ? Lb : Rb)[m] = ib[m];
            }
        }
        if (e.x >= 0)
            for (int m = 0; m < 5; ++m) qL[m] = Lb[m];
        if (e.y >= 0)
            for (int m = 0; m < 5; ++m) qR[m] = Rb[m];
    }
    if (__syncthreads_or(inflow)) add_by_ion<5>(fsb, sh, G.f_part + 10 * size_t(block));
}

// Face EMF candidate E_f = -n x F (IdealEMF.cpp:32-55) transposed: the edges' parts of E_f and of the induced flux are
// gathered; u+, B_tot and B_ind parts of the face's cells to their slots
__device__ __forceinline__ void face_emf_adjoint_role(const DevMesh &d, const StepFields &F, const AdjFields &G, const double *Phi,
                                                      const double *PhiAdd, int32_t f)
{
    if (f >= d.nf) return;
    V3 Eb;
    double pb = 0.0;
    auto edge = [&](int32_t pos) {
        const double2 a = ld2(G.eF + 4 * size_t(pos)), b = ld2(G.eF + 4 * size_t(pos) + 2);
        Eb += V3(a.x, a.y, b.x);
        pb += b.y;
    };
    if (d.fdeg == 3)
    {
        const int3 q = reinterpret_cast<const int3 *>(G.f2e_pos)[f];
        edge(q.x); edge(q.y); edge(q.z);
    }
    else
        for (int32_t k = d.f2e_ptr[f]; k < d.f2e_ptr[f + 1]; ++k) edge(G.f2e_pos[k]);
    const int32_t l = d.fL[f], r = d.fR[f];
    const int2 e = F.fent[f];
    double A;
    const V3 n = geo_normal(d, f, A), Fb = cross(n, Eb);
    const double Bn = (Phi[f] + PhiAdd[f]) / A;
    const double *Bi = F.rec + 5 * kAdjNs;
    double Bnb = 0.0;
    auto put = [&](int32_t k, const V3 &ub, const V3 &bt, const V3 &bi) {
        if (k < 0) return;
        double *o = G.sE + 9 * size_t(k);
        o[0] = ub.x; o[1] = ub.y; o[2] = ub.z; o[3] = bt.x; o[4] = bt.y; o[5] = bt.z; o[6] = bi.x; o[7] = bi.y; o[8] = bi.z;
    };
    if (l >= 0 && r >= 0)
    {
        const V3 uL = L3(F.uplus, l), uR = L3(F.uplus, r), tL = L3(F.Btot, l), tR = L3(F.Btot, r);
        const V3 db = L3(Bi + 16 * size_t(r), 0) - L3(Bi + 16 * size_t(l), 0), h = 0.5 * Fb;
        const double vL = dot(uL, n), vR = dot(uR, n);
        const bool right = fabs(vL) < fabs(vR);
        const double a = right ? fabs(vR) : fabs(vL), ab = -dot(h, db), v = right ? vR : vL;
        V3 ubL = dot(tL, h) * n - Bn * h, ubR = dot(tR, h) * n - Bn * h;
        (right ? ubR : ubL) += (v < 0 ? -ab : ab) * n;
        Bnb = -(dot(uL, h) + dot(uR, h));
        put(e.x, ubL, vL * h, a * h);
        put(e.y, ubR, vR * h, -a * h);
    }
    else
    {
        const int32_t c = l >= 0 ? l : r;
        if (c < 0) { G.Phib[f] += pb; return; }
        const V3 u = L3(F.uplus, c);
        Bnb = -dot(u, Fb);
        put(c == l ? e.x : e.y, dot(L3(F.Btot, c), Fb) * n - Bn * Fb, dot(u, n) * Fb, V3());
    }
    G.Phib[f] += pb + Bnb / A;
    G.PhiAddb[f] += Bnb / A;
}
} // namespace

// ---------------------------------------------------------------------------------------------------------- kernels
// Dynamic LDS: the heavy edges' rows when there are any
template <int DEG>
__global__ void __launch_bounds__(kAdjThreads, 3) k_adj_update(DevMesh d, Params P, StepFields F, AdjFields G, SpC Us, SpW Ub, const double *E,
                                                            double dt, const int32_t *heavy, int32_t n_heavy, int32_t hv, int32_t n_dt,
                                                            const double *dt_part, int32_t n_part, int32_t n_edge)
{
    extern __shared__ double rows[];
    __shared__ double sh[kAdjThreads];
    const int32_t b = blockIdx.x;
    if (b < n_heavy) edge_adjoint_heavy(d, F, G, P.cuct, dt, E, heavy[b], rows, hv, G.e_part + 4 * size_t(b));
    else if (b < n_heavy + n_dt) dt_cell_role(d, P, F, G, dt_part, n_part, dt);
    else if (b < n_heavy + n_dt + n_edge)
    {
        const int32_t i = near_block(d, b, n_heavy + n_dt, n_edge);
        double part[4] = {0, 0, 0, 0};
        edge_adjoint_light(d, F, G, P.cuct, dt, E, i * kAdjThreads + int32_t(threadIdx.x), part);
        double *o = G.e_part + 4 * size_t(n_heavy + i);
        const double s = block_sum(part[0], sh);
        if (threadIdx.x == 0) o[0] = s;
        // edges with the imposed EMF are few, at the inflow boundary
        if (__syncthreads_or(part[1] != 0.0 || part[2] != 0.0 || part[3] != 0.0))
            for (int q = 1; q < 4; ++q)
            {
                const double x = block_sum(part[q], sh);
                if (threadIdx.x == 0) o[q] += x;
            }
    }
    else
    {
        const int32_t first = n_heavy + n_dt + n_edge, i = near_block(d, b, first, int32_t(gridDim.x) - first);
        const double s = block_sum(update_adjoint_role<DEG>(d, P, F, G, Us, Ub, dt, i), sh);
        if (threadIdx.x == 0) G.c_part[i] = s;
    }
}

__global__ void __launch_bounds__(kAdjThreads) k_adj_faces(DevMesh d, Params P, StepFields F, AdjFields G, const double *Phi, const double *PhiAdd,
                                                           int32_t n_epart, int32_t n_cpart, int32_t n_emf)
{
    __shared__ double sh[kAdjThreads];
    const int32_t b = blockIdx.x;
    if (b == 0)
    {
        // adjoint of the time step: the edges' and the cells' parts
        double v = 0.0;
        for (int32_t i = threadIdx.x; i < n_epart; i += kAdjThreads) v += G.e_part[4 * size_t(i)];
        for (int32_t i = threadIdx.x; i < n_cpart; i += kAdjThreads) v += G.c_part[i];
        v = block_sum(v, sh);
        if (threadIdx.x == 0) G.dtb[0] = v;
    }
    else if (b <= n_emf) face_emf_adjoint_role(d, F, G, Phi, PhiAdd, near_block(d, b, 1, n_emf) * kAdjThreads + int32_t(threadIdx.x));
    else flux_adjoint_role(d, P, F, G, near_block(d, b, 1 + n_emf, int32_t(gridDim.x) - 1 - n_emf), sh);
}

// Limited gradients (Reconstruction.cpp:80-142) and the states formed from them (FluxRHS.cpp:16-27), transposed: thread
// (cell, ion), with the forward's operations up to the limiters.  In: the adjoints of the cell's face states; Wb +=
// the cell's own part, the entries receive the parts of the stencil neighbours' primitives.
template <int DEG>
__global__ void __launch_bounds__(kGradThreads, DEG == 6 ? 2 : 3) k_adj_gradients(DevMesh d, Params P, StepFields F, AdjFields G)
{
    constexpr int N = DEG > 0 ? DEG : 1, kCells = kGradThreads / kAdjNs;
    __shared__ double stage[kGradThreads * (DEG > 0 ? 5 * DEG : 1)];
    const int32_t t = threadIdx.x, s = t & 1, cl = t >> 1;
    const int32_t c0 = near_block(d, int32_t(blockIdx.x), 0, int32_t(gridDim.x)) * kCells, c = c0 + cl;
    const int32_t n_here = min(kCells, d.nc - c0) * (DEG * kAdjNs * 5 / 2);
    if constexpr (DEG > 0)
    {
        const double2 *src = reinterpret_cast<const double2 *>(F.FS + size_t(c0) * size_t(DEG * 5 * kAdjNs));
        double2 *dst = reinterpret_cast<double2 *>(stage);
        for (int32_t i = t; i < n_here; i += kGradThreads) dst[i] = src[i];
        __syncthreads();
    }
    double fsb[5] = {0, 0, 0, 0, 0};
    bool inflow = false;
    if (c < d.nc)
    {
        int32_t k0, nk, v[N], nb[N];
        row_of<DEG>(d, c, k0, nk);
        if constexpr (DEG > 0) { row_ids<DEG>(d.c2f, k0, v); row_ids<DEG>(d.snb, k0, nb); nk = DEG; }
        const double *own = F.rec + 16 * size_t(c);
        const V3 xc(own[13], own[14], own[15]);
        auto face = [&](int i) { return DEG > 0 ? v[i] : d.c2f[k0 + i]; };
        auto across = [&](int i) { return DEG > 0 ? nb[i] : d.snb[k0 + i]; };
        auto bar = [&](int i) { return DEG > 0 ? stage + 5 * ((cl * DEG + i) * kAdjNs + s) : F.FS + 5 * (size_t(k0 + i) * kAdjNs + s); };
        auto offset = [&](int i) {
            const int32_t o = across(i);
            if (o >= 0)
            {
                const double *q = F.rec + 16 * size_t(o);
                return V3(q[13], q[14], q[15]) - xc;
            }
            double A;
            const V3 n = psg(face(i)) * geo_normal(d, pid(face(i)), A);
            return (2.0 * dot(L3(d.fcen, pid(face(i))) - xc, n)) * n;
        };
        V3 dd_r[N], dx_r[N];
        if constexpr (DEG > 0)
        {
#pragma unroll
            for (int i = 0; i < DEG; ++i) { dd_r[i] = offset(i); dx_r[i] = L3(d.fcen, pid(v[i])) - xc; }
        }
        auto dd = [&](int i) { return DEG > 0 ? dd_r[i] : offset(i); };
        auto dx = [&](int i) { return DEG > 0 ? dx_r[i] : L3(d.fcen, pid(face(i))) - xc; };
        const bool valid = P.second_order && d.svalid[c];
        double wc[5], lo[5], hi[5], g[5][3], psi[5], wcb[5];
        int32_t hs[5], ls[5], act[5]; // entry of the extremes (-1: the cell); entry that limits, + 64 by the relative limit, or -1
        for (int m = 0; m < 5; ++m)
        {
            wc[m] = lo[m] = hi[m] = own[5 * s + m];
            hs[m] = ls[m] = act[m] = -1;
            g[m][0] = g[m][1] = g[m][2] = 0.0;
            psi[m] = 1.0;
        }
        if (valid)
        {
            double fs[5], r[5][3] = {};
            for (int m = 0; m < 5; ++m) fs[m] = P.fs[s][m];
#pragma unroll
            for (int i = 0; i < (DEG > 0 ? DEG : nk); ++i)
            {
                const int32_t o = across(i);
                if (o == kNoStencil) continue;
                double wn[5];
                if (o >= 0)
                    for (int m = 0; m < 5; ++m) wn[m] = F.rec[16 * size_t(o) + 5 * s + m];
                else stencil_ghost(d, s, static_cast<const double *>(nullptr), wc, fs, face(i), o, wn);
                const V3 q = dd(i);
                const double w = 1.0 / dot(q, q);
                for (int m = 0; m < 5; ++m)
                {
                    const double dq = wn[m] - wc[m];
                    r[m][0] += w * q.x * dq; r[m][1] += w * q.y * dq; r[m][2] += w * q.z * dq;
                    if (wn[m] < lo[m]) { lo[m] = wn[m]; ls[m] = i; }
                    if (hi[m] < wn[m]) { hi[m] = wn[m]; hs[m] = i; }
                }
            }
            const double *I = d.sinv + 6 * size_t(c);
            const double I0 = I[0], I1 = I[1], I2 = I[2], I3 = I[3], I4 = I[4], I5 = I[5];
#pragma unroll
            for (int m = 0; m < 5; ++m)
            {
                g[m][0] = I0 * r[m][0] + I1 * r[m][1] + I2 * r[m][2];
                g[m][1] = I1 * r[m][0] + I3 * r[m][1] + I4 * r[m][2];
                g[m][2] = I2 * r[m][0] + I4 * r[m][1] + I5 * r[m][2];
                const bool rel = P.rel_limit > 0 && (m == 0 || m == 4);
                // psi = max(0, min(1, quotients)): the first smallest quotient below 1 counts, unless it is not above 0
#pragma unroll
                for (int i = 0; i < (DEG > 0 ? DEG : nk); ++i)
                {
                    const V3 x = dx(i);
                    const double dl = g[m][0] * x.x + g[m][1] * x.y + g[m][2] * x.z;
                    const double q = (dl > 0 ? hi[m] - wc[m] : lo[m] - wc[m]) / dl;
                    if (fabs(dl) > 1e-300 && q < psi[m]) { psi[m] = q; act[m] = i; }
                }
                if (rel)
#pragma unroll
                    for (int i = 0; i < (DEG > 0 ? DEG : nk); ++i)
                    {
                        const V3 x = dx(i);
                        const double dl = fabs(g[m][0] * x.x + g[m][1] * x.y + g[m][2] * x.z), q = P.rel_limit * wc[m] / dl;
                        if (dl > 1e-300 && q < psi[m]) { psi[m] = q; act[m] = i + 64; }
                    }
                if (!(psi[m] > 0.0)) { psi[m] = 0.0; act[m] = -1; }
            }
        }
        // entries whose state is the linear one (else it is the cell's own): a face state depends on the gradient there
        uint64_t linear = 0;
        if (valid)
#pragma unroll
            for (int i = 0; i < (DEG > 0 ? DEG : nk); ++i)
            {
                const V3 x = dx(i);
                const double rr = wc[0] + psi[0] * g[0][0] * x.x + psi[0] * g[0][1] * x.y + psi[0] * g[0][2] * x.z;
                const double pp = wc[4] + psi[4] * g[4][0] * x.x + psi[4] * g[4][1] * x.y + psi[4] * g[4][2] * x.z;
                if (rr > 0 && pp > 0) linear |= uint64_t(1) << i;
            }
        const double *I = d.sinv + 6 * size_t(c);
        const double I0 = I[0], I1 = I[1], I2 = I[2], I3 = I[3], I4 = I[4], I5 = I[5];
#pragma unroll
        for (int m = 0; m < 5; ++m)
        {
            double own_b = 0.0, hb = 0.0, lb = 0.0;
            V3 ob;
#pragma unroll
            for (int i = 0; i < (DEG > 0 ? DEG : nk); ++i)
            {
                const double b = bar(i)[m];
                own_b += b;
                if (linear >> i & 1) ob += b * dx(i);
            }
            V3 tb;
            if (valid)
            {
                const V3 gm(g[m][0], g[m][1], g[m][2]);
                V3 gb = psi[m] * ob;
                if (act[m] >= 0)
                {
                    V3 x;
                    if constexpr (DEG > 0)
                    {
#pragma unroll
                        for (int i = 0; i < DEG; ++i)
                            if ((act[m] & 63) == i) x = dx_r[i];
                    }
                    else x = dx(act[m] & 63);
                    const double pb = dot(ob, gm), dl = dot(gm, x);
                    double db;
                    if (act[m] >= 64)
                    {
                        const double q = pb / fabs(dl);
                        own_b += P.rel_limit * q;
                        db = dl < 0 ? q * psi[m] : -q * psi[m];
                    }
                    else
                    {
                        const double q = pb / dl;
                        (dl > 0 ? hb : lb) = q;
                        own_b -= q;
                        db = -q * psi[m];
                    }
                    gb += db * x;
                }
                tb = V3(I0 * gb.x + I1 * gb.y + I2 * gb.z, I1 * gb.x + I3 * gb.y + I4 * gb.z, I2 * gb.x + I4 * gb.y + I5 * gb.z);
                if (hs[m] < 0) own_b += hb;
                if (ls[m] < 0) own_b += lb;
            }
#pragma unroll
            for (int i = 0; i < (DEG > 0 ? DEG : nk); ++i)
            {
                double q = 0.0;
                if (valid && across(i) != kNoStencil)
                {
                    const V3 x = dd(i);
                    q = dot(x, tb) / dot(x, x);
                    own_b -= q;
                    if (hs[m] == i) q += hb;
                    if (ls[m] == i) q += lb;
                }
                bar(i)[m] = q;
            }
            wcb[m] = own_b;
        }
        // ghosts (and a cell that is its own neighbour): their parts go back to the cell or the free stream
#pragma unroll
        for (int i = 0; i < (DEG > 0 ? DEG : nk); ++i)
        {
            const int32_t o = across(i);
            if (!valid || o == kNoStencil || (o >= 0 && o != c)) continue;
            const double *b = bar(i);
            const int8_t kind = o >= 0 ? kInterior : d.kind[-(o + 1)];
            if (kind == kInflow)
            {
                inflow = true;
                for (int m = 0; m < 5; ++m) fsb[m] += b[m];
            }
            else if (!(kind == kWall && s == 1))
            {
                for (int m = 0; m < 5; ++m) wcb[m] += b[m];
                if (kind == kWall)
                {
                    double A;
                    const V3 n = geo_normal(d, pid(face(i)), A); // its sign drops out
                    const double w = 2.0 * (n.x * b[1] + n.y * b[2] + n.z * b[3]);
                    wcb[1] -= w * n.x; wcb[2] -= w * n.y; wcb[3] -= w * n.z;
                }
            }
        }
        double *o = G.Wb + 10 * size_t(c) + 5 * s;
        for (int m = 0; m < 5; ++m) o[m] += wcb[m];
    }
    if constexpr (DEG > 0)
    {
        __syncthreads();
        double2 *dst = reinterpret_cast<double2 *>(F.FS + size_t(c0) * size_t(DEG * 5 * kAdjNs));
        const double2 *src = reinterpret_cast<const double2 *>(stage);
        for (int32_t i = t; i < n_here; i += kGradThreads) dst[i] = src[i];
    }
    if (__syncthreads_or(inflow)) add_by_ion<5>(fsb, stage, G.g_part + 10 * size_t(blockIdx.x));
}

// What is left of a cell: the parts its stencil neighbours, faces and edges hold for it, the current
// (Current.cpp:9-31), its CFL step if it set the step, u+ (Solver.cpp:110-118), the primitive recovery and the field
// reconstruction, transposed: Ub +=, Baddb +=, sPhi
template <int DEG>
__global__ void __launch_bounds__(kAdjThreads) k_adj_cells(DevMesh d, Params P, StepFields F, AdjFields G, SpC Us, SpW Ub, int32_t with_dt)
{
    constexpr int N = DEG > 0 ? DEG / 2 : 1;
    const int32_t t = threadIdx.x, s = t & 1, c = gid(d) >> 1;
    if (c >= d.nc) return; // both threads of a cell
    // the face normals' matrix of the reconstruction (Reconstruct.cpp:11-45), the faces' and edges' parts: this thread's half
    int32_t k0, nk;
    row_of<DEG>(d, c, k0, nk);
    double M[6] = {0, 0, 0, 0, 0, 0}, A[N], w[5];
    V3 n[N], up, bt, bi;
    const V3 jc = L3(G.Jv, c);
    auto half = [&](int32_t k, double &a, V3 &m) {
        const int32_t v = d.c2f[k], o = d.c2n[k];
        m = geo_normal(d, pid(v), a);
        const double *x = G.sE + 9 * size_t(k);
        up += V3(x[0], x[1], x[2]);
        bt += V3(x[3], x[4], x[5]);
        bi += V3(x[6], x[7], x[8]);
        const V3 area = (psg(v) * a) * m;
        bi += o >= 0 ? 0.5 * cross(jc - L3(G.Jv, o), area) : cross(jc, area);
        if (a <= 0) return;
        M[0] += a * m.x * m.x; M[1] += a * m.x * m.y; M[2] += a * m.x * m.z;
        M[3] += a * m.y * m.y; M[4] += a * m.y * m.z; M[5] += a * m.z * m.z;
    };
    for (int m = 0; m < 5; ++m) w[m] = G.Wb[10 * size_t(c) + 5 * s + m];
    if constexpr (DEG > 0)
    {
        int32_t op[DEG];
        row_ids<DEG>(G.opp, k0, op);
#pragma unroll
        for (int i = 0; i < DEG; ++i)
            if (op[i] >= 0)
                for (int m = 0; m < 5; ++m) w[m] += F.FS[10 * size_t(op[i]) + 5 * s + m];
#pragma unroll
        for (int i = 0; i < N; ++i) half(k0 + 2 * i + s, A[i], n[i]);
    }
    else
    {
        for (int32_t k = k0; k < k0 + nk; ++k)
            if (G.opp[k] >= 0)
                for (int m = 0; m < 5; ++m) w[m] += F.FS[10 * size_t(G.opp[k]) + 5 * s + m];
        for (int32_t k = k0 + s; k < k0 + nk; k += 2) half(k, A[0], n[0]);
    }
    for (int32_t j = G.cec_ptr[c] + s; j < G.cec_ptr[c + 1]; j += 2) up += L3(G.eC, G.cec[j]);
    auto both = [](double x) { return x + __shfl_xor(x, 1); };
    up = V3(both(up.x), both(up.y), both(up.z));
    bt = V3(both(bt.x), both(bt.y), both(bt.z)) + L3(G.Btb, c);
    bi = V3(both(bi.x), both(bi.y), both(bi.z));
    for (int q = 0; q < 6; ++q) M[q] = both(M[q]);
    if (with_dt && G.dt_cell[0] == c)
    {
        const double x = G.dtb[0];
        for (int m = 0; m < 5; ++m) w[m] += x * G.dtb[1 + 5 * s + m];
        bt += x * V3(G.dtb[11], G.dtb[12], G.dtb[13]);
    }
    const double *W = F.rec + 16 * size_t(c) + 5 * s;
    const V3 u(W[1], W[2], W[3]);
    const double rho = W[0];
    {
        // u+ = sum chi_s u_s, chi_s = n_s / n_e
        const double ns = ion_density(P, s, rho), ne = both(ns), inv = 1.0 / ne, x = ns * inv, b = dot(up, u), m = both(b * x);
        if (d.mat[c] == 0 && ne > 1e-300)
        {
            if (rho >= 0) w[0] += (b - m) * inv / P.M_s[s] * P.M_ref;
            w[1] += x * up.x; w[2] += x * up.y; w[3] += x * up.z;
        }
        else if (d.mat[c] == 0 && s == 0) { w[1] += up.x; w[2] += up.y; w[3] += up.z; }
    }
    {
        // to_prim (Euler.h:13-27)
        const double *U = Us.p[s] + 5 * size_t(c);
        double *o = Ub.p[s] + 5 * size_t(c);
        const double uu = dot(u, u), g = P.gamma - 1.0;
        const double eb = g * (U[4] - 0.5 * rho * uu) < P.p_floor ? 0.0 : g * w[4];
        const V3 mb = (1.0 / rho) * V3(w[1], w[2], w[3]) - eb * u;
        if (!(U[0] < P.rho_floor)) o[0] += w[0] - 0.5 * uu * eb - dot(u, mb);
        o[1] += mb.x; o[2] += mb.y; o[3] += mb.z;
        o[4] += eb;
    }
    if (s == 0) st3(G.Baddb, c, L3(G.Baddb, c) + bt);
    const V3 y = normal_solve(M, bi + bt);
    if constexpr (DEG > 0)
    {
#pragma unroll
        for (int i = 0; i < N; ++i) G.sPhi[k0 + 2 * i + s] = A[i] > 0 ? dot(n[i], y) : 0.0;
    }
    else
        for (int32_t k = k0 + s; k < k0 + nk; k += 2)
        {
            double a;
            const V3 q = geo_normal(d, pid(d.c2f[k]), a);
            G.sPhi[k] = a > 0 ? dot(q, y) : 0.0;
        }
}

// Shell energy transposed: J = sum over fluid cells with r0 <= |x| <= r1 of |b + B_add|^2 V; sets Baddb and sPhi
__global__ void __launch_bounds__(kAdjThreads) k_adj_energy(DevMesh d, const double *phi, const double *badd, double r0, double r1, AdjFields G)
{
    const int32_t c = gid();
    if (c >= d.nc) return;
    V3 bb;
    if (d.mat[c] == 0)
    {
        const double r = norm(L3(d.ccen, c));
        if (r >= r0 && r <= r1) bb = (2.0 * d.cvol[c]) * (cell_vector(d, c, phi) + L3(badd, c));
    }
    st3(G.Baddb, c, bb);
    double M[6] = {0, 0, 0, 0, 0, 0}, A;
    for (int32_t k = d.c2f_ptr[c]; k < d.c2f_ptr[c + 1]; ++k)
    {
        const V3 m = geo_normal(d, pid(d.c2f[k]), A);
        if (A <= 0) continue;
        M[0] += A * m.x * m.x; M[1] += A * m.x * m.y; M[2] += A * m.x * m.z;
        M[3] += A * m.y * m.y; M[4] += A * m.y * m.z; M[5] += A * m.z * m.z;
    }
    const V3 y = normal_solve(M, bb);
    for (int32_t k = d.c2f_ptr[c]; k < d.c2f_ptr[c + 1]; ++k)
    {
        const V3 m = geo_normal(d, pid(d.c2f[k]), A);
        G.sPhi[k] = A > 0 ? dot(m, y) : 0.0;
    }
}

// Face gather of the reconstruction parts: Phib_f += both cells' slots; the first one of a sweep sets Phib and PhiAddb
__global__ void __launch_bounds__(kAdjThreads) k_adj_flux(DevMesh d, const int2 *fent, AdjFields G, int32_t first)
{
    const int32_t f = gid(d);
    if (f >= d.nf) return;
    const int2 e = fent[f];
    const double x = (e.x >= 0 ? G.sPhi[e.x] : 0.0) + (e.y >= 0 ? G.sPhi[e.y] : 0.0);
    if (first) { G.Phib[f] = x; G.PhiAddb[f] = 0.0; }
    else G.Phib[f] += x;
}

// Sums of the sweep's block parts, one block each: the free stream (10) from the fluxes and the gradients together, E_inf (3)
__global__ void __launch_bounds__(kAdjThreads) k_adj_sums(AdjFields G, int32_t n_f, int32_t n_g, int32_t n_e)
{
    __shared__ double sh[kAdjThreads];
    const int32_t b = blockIdx.x;
    double v = 0.0;
    if (b < 10)
    {
        for (int32_t i = threadIdx.x; i < n_f; i += kAdjThreads) v += G.f_part[10 * size_t(i) + b];
        for (int32_t i = threadIdx.x; i < n_g; i += kAdjThreads) v += G.g_part[10 * size_t(i) + b];
    }
    else
        for (int32_t i = threadIdx.x; i < n_e; i += kAdjThreads) v += G.e_part[4 * size_t(i) + size_t(b - 9)];
    v = block_sum(v, sh);
    if (threadIdx.x == 0) G.sums[b] = v;
    if (b == 0 && threadIdx.x == 0) G.sums[13] = G.dt_cell[1];
}

// ----------------------------------------------------------------------------------------------- gather maps (once)
// per c2f entry: the entry on the other side of its face, if that cell's stencil neighbour there is this cell
__global__ void __launch_bounds__(256) k_adj_opposite(DevMesh d, const int2 *fent, int32_t *opp)
{
    const int32_t c = gid();
    if (c >= d.nc) return;
    for (int32_t k = d.c2f_ptr[c]; k < d.c2f_ptr[c + 1]; ++k)
    {
        const int2 e = fent[pid(d.c2f[k])];
        const int32_t o = k == e.x ? e.y : k == e.y ? e.x : -1, n = d.c2n[k];
        opp[k] = o >= 0 && n >= 0 && n != c && d.snb[o] == c ? o : -1;
    }
}
// per f2e entry: where the face stands in the edge's row; counts the entries without one, and the faces without a cell
__global__ void __launch_bounds__(256) k_adj_edge_pos(DevMesh d, int32_t *pos, int32_t *counts)
{
    const int32_t f = gid();
    if (f >= d.nf) return;
    if (d.fL[f] < 0 && d.fR[f] < 0) atomicAdd(counts + 1, 1);
    for (int32_t k = d.f2e_ptr[f]; k < d.f2e_ptr[f + 1]; ++k)
    {
        const int32_t e = pid(d.f2e[k]);
        int32_t at = -1;
        for (int32_t i = d.e2f_ptr[e]; i < d.e2f_ptr[e + 1] && at < 0; ++i)
            if (pid(d.e2f[i]) == f) at = i;
        if (at < 0) atomicAdd(counts, 1);
        pos[k] = at < 0 ? 0 : at;
    }
}
// edge-cell entries by cell: counts into ptr[c + 1], then their running sums, then the entries, sorted within a cell
__global__ void __launch_bounds__(256) k_adj_count(const int32_t *ec_cell, int32_t n, int32_t *ptr)
{
    const int32_t i = gid();
    if (i < n) atomicAdd(ptr + ec_cell[i] + 1, 1);
}
// running sums of each block's kScanTile values, and the blocks' totals; then the totals before a block added to its values
constexpr int kScanTile = 1024;
__device__ __forceinline__ int32_t scan_block(int32_t v, int32_t *sh)
{
    const int32_t t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
    for (int k = 1; k < kScanTile; k <<= 1)
    {
        const int32_t a = t >= k ? sh[t - k] : 0;
        __syncthreads();
        sh[t] += a;
        __syncthreads();
    }
    return sh[t];
}
__global__ void __launch_bounds__(kScanTile) k_adj_scan(int32_t *x, int32_t n, int32_t *total)
{
    __shared__ int32_t sh[kScanTile];
    const int32_t i = gid(), v = scan_block(i < n ? x[i] : 0, sh);
    if (i < n) x[i] = v;
    if (threadIdx.x == kScanTile - 1) total[blockIdx.x] = v;
}
__global__ void __launch_bounds__(kScanTile) k_adj_scan_add(int32_t *x, int32_t n, const int32_t *total)
{
    __shared__ int32_t sh[kScanTile];
    int32_t before = 0;
    for (int32_t b = threadIdx.x; b < int32_t(blockIdx.x); b += kScanTile) before += total[b];
    scan_block(before, sh);
    const int32_t i = gid();
    if (i < n) x[i] += sh[kScanTile - 1];
}
__global__ void __launch_bounds__(256) k_adj_fill(const int32_t *ec_cell, int32_t n, const int32_t *ptr, int32_t *used, int32_t *cec)
{
    const int32_t i = gid();
    if (i < n) cec[ptr[ec_cell[i]] + atomicAdd(used + ec_cell[i], 1)] = i;
}
__global__ void __launch_bounds__(256) k_adj_sort(int32_t nc, const int32_t *ptr, int32_t *cec)
{
    const int32_t c = gid();
    if (c >= nc) return;
    for (int32_t i = ptr[c] + 1; i < ptr[c + 1]; ++i)
    {
        const int32_t x = cec[i];
        int32_t j = i;
        for (; j > ptr[c] && cec[j - 1] > x; --j) cec[j] = cec[j - 1];
        cec[j] = x;
    }
}
} // namespace mhdg

using namespace mhdg;

namespace
{
inline int blocks(int64_t n, int64_t per) { return static_cast<int>((n + per - 1) / per); }
void chk(hipError_t e, const char *w)
{
    if (e != hipSuccess) throw std::runtime_error(std::string(w) + ": " + hipGetErrorString(e));
}
template <class Fn> void by_degree(int32_t cdeg, Fn f)
{
    if (cdeg == 4) f(std::integral_constant<int, 4>{});
    else if (cdeg == 6) f(std::integral_constant<int, 6>{});
    else f(std::integral_constant<int, 0>{});
}
} // namespace

#define LAUNCH(NAME, ...)                                                                                                    \
    do                                                                                                                       \
    {                                                                                                                        \
        prof_begin(NAME);                                                                                                    \
        hipLaunchKernelGGL(__VA_ARGS__);                                                                                     \
        prof_end();                                                                                                          \
    } while (0)

// Work arrays and gather maps of the adjoint (first use), and a state for every step and after the last
void mhdg_ctx::vjp_alloc(int n_steps)
{
    if (!aw.x.E)
    {
        const size_t C = nc, F = nf, E = ne, K = c2f_nnz;
        auto D = [&](size_t n) { return static_cast<double *>(alloc(n * sizeof(double))); };
        auto I = [&](size_t n) { return static_cast<int32_t *>(alloc(n * sizeof(int32_t))); };
        int32_t f2e_n = 0;
        d2h(&f2e_n, d.f2e_ptr + F, 4);
        int32_t *opp = I(K), *pos = I(size_t(f2e_n)), *ptr = I(C + 1), *cec = I(ec_nnz), *used = I(C + 2);
        chk(hipMemsetAsync(ptr, 0, 4 * (C + 1), stream), "memset");
        chk(hipMemsetAsync(used, 0, 4 * (C + 2), stream), "memset"); // per cell, then the two counts
        const dim3 b256(256);
        hipLaunchKernelGGL(k_adj_opposite, dim3(blocks(nc, 256)), b256, 0, stream, d, sf.fent, opp);
        hipLaunchKernelGGL(k_adj_edge_pos, dim3(blocks(nf, 256)), b256, 0, stream, d, pos, used + C);
        if (ec_nnz)
        {
            const int32_t n = int32_t(ec_nnz);
            hipLaunchKernelGGL(k_adj_count, dim3(blocks(n, 256)), b256, 0, stream, d.ec_cell, n, ptr);
            const dim3 tiles(blocks(int64_t(nc) + 1, kScanTile));
            int32_t *total = I(tiles.x);
            hipLaunchKernelGGL(k_adj_scan, tiles, dim3(kScanTile), 0, stream, ptr, nc + 1, total);
            hipLaunchKernelGGL(k_adj_scan_add, tiles, dim3(kScanTile), 0, stream, ptr, nc + 1, static_cast<const int32_t *>(total));
            hipLaunchKernelGGL(k_adj_fill, dim3(blocks(n, 256)), b256, 0, stream, d.ec_cell, n, static_cast<const int32_t *>(ptr), used, cec);
            hipLaunchKernelGGL(k_adj_sort, dim3(blocks(nc, 256)), b256, 0, stream, nc, static_cast<const int32_t *>(ptr), cec);
        }
        check_launch("vjp maps");
        int32_t counts[2];
        d2h(counts, used + C, 8);
        if (counts[0]) throw std::runtime_error("vjp: face missing from its edge's face list");
        AdjFields &g = aw.g;
        g.all_active = counts[1] == 0;
        g.opp = opp; g.f2e_pos = pos; g.cec_ptr = ptr; g.cec = cec;
        for (int s = 0; s < 2; ++s) aw.Ub[s] = D(5 * C);
        g.Wb = D(10 * C); g.rv = D(10 * C); g.Jv = D(3 * C); g.Btb = D(3 * C);
        g.sE = D(9 * K); g.sPhi = D(K); g.eF = D(4 * e2f_nnz); g.eC = D(3 * ec_nnz);
        g.Phib = D(F); g.PhiAddb = D(F); g.Baddb = D(3 * C);
        g.e_part = D(4 * size_t(n_heavy + blocks(ne, kAdjThreads))); g.c_part = D(size_t(blocks(nc, kAdjThreads / 2)));
        g.f_part = D(10 * size_t(blocks(nf, kAdjThreads / 2))); g.g_part = D(10 * size_t(blocks(nc, kGradThreads / 2)));
        g.dtb = D(16); g.dt_cell = I(2); g.sums = D(16);
        aw.x.F = step_fields(D(3 * C), D(3 * C), D(3 * C), D(C));
        aw.x.dt_part = D(size_t(blocks(nc, 256)) + 1); aw.x.dt_dev = D(1);
        aw.x.E = D(E);
    }
    if (int(aw.ck.size()) < n_steps + 1)
    {
        const size_t per = 10 * size_t(nc) + size_t(nf);
        for (int n = int(aw.ck.size()); n < n_steps + 1; ++n)
        {
            void *p = nullptr;
            chk(hipMalloc(&p, per * 8), "hipMalloc");
            aw.ck.push_back(static_cast<double *>(p));
        }
    }
}

// n explicit steps from the resident state (kept unchanged), J = shell energy of the final state, and the
// reverse sweep; gradients are left in aw.Ub, aw.g.Phib, aw.g.PhiAddb, aw.g.Baddb and fs_b (2x5), einf_b (3)
double mhdg_ctx::step_vjp(int n_steps, double dt_max, double r0, double r1, double *fs_b, double *einf_b)
{
    vjp_alloc(n_steps);
    const size_t C = nc, F = nf;
    const int nbc = blocks(nc, kAdjThreads), nbf = blocks(nf, kAdjThreads), n_edge = blocks(ne, kAdjThreads), n_cell = blocks(nc, kAdjThreads / 2),
              n_flux = blocks(nf, kAdjThreads / 2), n_grad = blocks(nc, kGradThreads / 2), n_epart = n_heavy + n_edge;
    const AdjFields &g = aw.g;
    // the state before step n, which the step overwrites in the copy for n + 1
    auto state = [&](int n) {
        double *ck = aw.ck[size_t(n)];
        aw.x.U[0] = ck; aw.x.U[1] = ck + 5 * C; aw.x.Phi = ck + 10 * C;
    };
    for (int s = 0; s < 2; ++s) chk(hipMemcpyAsync(aw.ck[0] + 5 * C * size_t(s), U[s], 5 * C * 8, hipMemcpyDeviceToDevice, stream), "copy");
    chk(hipMemcpyAsync(aw.ck[0] + 10 * C, Phi, F * 8, hipMemcpyDeviceToDevice, stream), "copy");
    std::vector<double> dts(static_cast<size_t>(n_steps));
    for (int n = 0; n < n_steps; ++n)
    {
        chk(hipMemcpyAsync(aw.ck[size_t(n) + 1], aw.ck[size_t(n)], (10 * C + F) * 8, hipMemcpyDeviceToDevice, stream), "copy");
        state(n + 1);
        dts[size_t(n)] = explicit_stage(aw.x, dt_max, kStageState);
    }
    state(n_steps);
    double Jv = 0;
    shell_energy<double>(aw.x.Phi, Badd, r0, r1, &Jv);
    // adjoint of the objective
    for (int s = 0; s < 2; ++s) chk(hipMemsetAsync(aw.Ub[s], 0, 5 * C * 8, stream), "memset");
    chk(hipMemsetAsync(g.e_part, 0, 8 * 4 * size_t(n_epart), stream), "memset");
    chk(hipMemsetAsync(g.f_part, 0, 8 * 10 * size_t(n_flux), stream), "memset");
    chk(hipMemsetAsync(g.g_part, 0, 8 * 10 * size_t(n_grad), stream), "memset");
    chk(hipMemsetAsync(g.dt_cell, 0, 8, stream), "memset");
    LAUNCH("adj_energy", k_adj_energy, dim3(nbc), dim3(kAdjThreads), 0, stream, d, static_cast<const double *>(aw.x.Phi),
           static_cast<const double *>(Badd), r0, r1, g);
    LAUNCH("adj_flux", k_adj_flux, dim3(nbf), dim3(kAdjThreads), 0, stream, d, aw.x.F.fent, g, 1);
    SpC Us{};
    SpW Ub{};
    for (int s = 0; s < 2; ++s) Ub.p[s] = aw.Ub[s];
    const size_t lds = n_heavy ? (kHeavyRows * sizeof(double) + sizeof(int32_t)) * size_t(max_valence) : 0;
    for (int n = n_steps - 1; n >= 0; --n)
    {
        // the step's fields from the state before it; the forward sweep's last ones are still there
        state(n);
        const bool again = n < n_steps - 1;
        if (again) explicit_stage(aw.x, dt_max, kStageNone);
        for (int s = 0; s < 2; ++s) Us.p[s] = aw.x.U[s];
        const double dt = dts[size_t(n)];
        const int n_dt = dt < dt_max ? 1 : 0; // else dt_max set the step
        by_degree(cdeg, [&](auto deg) {
            constexpr int DEG = decltype(deg)::value;
            LAUNCH("adj_update", k_adj_update<DEG>, dim3(n_heavy + n_dt + n_edge + n_cell), dim3(kAdjThreads), lds, stream, d, P, aw.x.F, g, Us, Ub,
                   static_cast<const double *>(aw.x.E), dt, static_cast<const int32_t *>(heavy), n_heavy, max_valence, n_dt,
                   static_cast<const double *>(aw.x.dt_part), blocks(nc, 256), n_edge);
            LAUNCH("adj_faces", k_adj_faces, dim3(1 + nbf + n_flux), dim3(kAdjThreads), 0, stream, d, P, aw.x.F, g,
                   static_cast<const double *>(aw.x.Phi), static_cast<const double *>(PhiAdd), n_epart, n_cell, nbf);
            LAUNCH("adj_gradients", k_adj_gradients<DEG>, dim3(n_grad), dim3(kGradThreads), 0, stream, d, P, aw.x.F, g);
            LAUNCH("adj_cells", k_adj_cells<DEG>, dim3(n_cell), dim3(kAdjThreads), 0, stream, d, P, aw.x.F, g, Us, Ub, n_dt);
        });
        LAUNCH("adj_flux", k_adj_flux, dim3(nbf), dim3(kAdjThreads), 0, stream, d, aw.x.F.fent, g, 0);
        check_launch("vjp reverse step");
        // written while the step's fields were formed, long before what was launched since ends
        if (again && wait_box(dt_box)[0] != dt) throw std::runtime_error("vjp: recomputed time step differs from the forward sweep");
    }
    LAUNCH("adj_sums", k_adj_sums, dim3(13), dim3(kAdjThreads), 0, stream, g, n_flux, n_grad, n_epart);
    check_launch("vjp sums");
    double h[14];
    d2h(h, g.sums, sizeof(h));
    if (h[13] != 0.0) throw std::runtime_error("vjp: CFL minimum cell not found");
    if (fs_b)
        for (int k = 0; k < 10; ++k) fs_b[k] = h[k];
    if (einf_b)
        for (int k = 0; k < 3; ++k) einf_b[k] = h[10 + k];
    return Jv;
}
