// Reverse mode (adjoint) of the explicit stage of the Mercury step (MercuryUns/driver/Solver.cpp:228-277 with
// the Hall solve inactive): the gradient of the shell magnetic energy after n steps with respect to the
// initial state, the background flux and field, the free-stream states and the imposed inflow EMF.
//
// The forward sweep is the resident step's own (explicit_step.hip) on fields of its own, and keeps the state (U, Phi) of
// every step; the reverse sweep recomputes a step's fields from it (the last step's are still there) and runs the
// transposed kernels from the branch that the values take (limiters, upwinding, floors, argmax, the CFL minimum; a tie takes
// the operand that the value computation keeps).  Six launches a step:
//   update      edges: Faraday and the UCT sum | faces: the time step's part of Faraday | cells: the update and its sources |
//               the cell that sets the time step | the free stream's sums of the step before in the sweep
//   faces       Rusanov fluxes | face EMF candidates | sums of the inflow EMF's and of the cells' time step's parts
//   mirror      the velocities that a wall couples
//   gradients   limited gradients: adjoints of the face states -> of the primitives of the stencil | the time step's adjoint
//   cells       the neighbours' parts, current, CFL cell, u+, primitive recovery, field reconstruction | free-stream blocks
//   flux        the reconstruction's parts of the face flux
//
// Every operation and every sum has a fixed place: each local derivative is the forward-mode column of its input (Tan below,
// Dual of dual.h) weighted and summed in the columns' order, gathers run in row order, sums over the mesh over 256-entity
// blocks in a tree and over the blocks in their order.  The order matters to more than the last digit: an input whose
// influence has not reached the objective (the inflow EMF, four layers away) has a gradient that is what the cancelling
// sums leave, 1e-60 to 1e-35 where the others are 1e-1, and another order leaves something else.
//
// Measured at 484k tetrahedra, five steps (one MI355X): a reverse step takes 1060 us, its fields' recomputation 350; with
// every column a pass of Dual arithmetic over the whole operation and 20 adjoints per (cell, face) entry and ion instead of
// 5 it took 5100 and 520, and the host summed block parts five times a step.  The whole call, gradients in host memory:
// 36.3 -> 13.9 ms.  update 302 us (two-thirds of it the edges, bound by their chains of dependent gathers at three waves per
// SIMD; in two launches 216 + 105), gradients 260 (its FP64 instructions, at two waves: three spilled, 300) and mirror 23
// (inside the gradients, where half of the waves have a wall cell, 322 for both), faces 245 and cells 214 (slots and
// gathered rows).  Sums with one derivative for all of a cell's or face's inputs, in whatever order is shortest, took 890.
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
constexpr int kSumStage = 2048;   // doubles staged per pass of a serial sum

// A value and its derivative along one input; what does not depend on the input stays a double.  The operations are those
// of Dual (dual.h) without the terms that a zero derivative makes zero, so a derivative has the bits of its Dual column.
struct Tan { double v, d; };
__device__ __forceinline__ Tan operator+(const Tan &a, const Tan &b) { return {a.v + b.v, a.d + b.d}; }
__device__ __forceinline__ Tan operator+(const Tan &a, double b) { return {a.v + b, a.d}; }
__device__ __forceinline__ Tan operator+(double a, const Tan &b) { return {a + b.v, b.d}; }
__device__ __forceinline__ Tan operator-(const Tan &a, const Tan &b) { return {a.v - b.v, a.d - b.d}; }
__device__ __forceinline__ Tan operator-(const Tan &a, double b) { return {a.v - b, a.d}; }
__device__ __forceinline__ Tan operator-(double a, const Tan &b) { return {a - b.v, -b.d}; }
__device__ __forceinline__ Tan operator-(const Tan &a) { return {-a.v, -a.d}; }
__device__ __forceinline__ Tan operator*(const Tan &a, const Tan &b) { return {a.v * b.v, a.d * b.v + a.v * b.d}; }
__device__ __forceinline__ Tan operator*(const Tan &a, double b) { return {a.v * b, a.d * b}; }
__device__ __forceinline__ Tan operator*(double a, const Tan &b) { return {a * b.v, a * b.d}; }
__device__ __forceinline__ Tan operator/(const Tan &a, const Tan &b)
{
    const double q = a.v / b.v;
    return {q, (a.d - q * b.d) / b.v};
}
__device__ __forceinline__ Tan operator/(const Tan &a, double b) { return {a.v / b, a.d / b}; }
__device__ __forceinline__ Tan operator/(double a, const Tan &b)
{
    const double q = a / b.v;
    return {q, -(q * b.d) / b.v};
}
__device__ __forceinline__ Tan tsqrt(const Tan &a)
{
    const double s = sqrt(a.v);
    return {s, s > 0 ? a.d / (2.0 * s) : 0.0};
}
__device__ __forceinline__ double tsqrt(double a) { return sqrt(a); }
__device__ __forceinline__ Tan tabs(const Tan &a) { return a.v < 0 ? -a : a; }
__device__ __forceinline__ double tabs(double a) { return fabs(a); }
// mx (dev.h) of operands of which one depends on the input
__device__ __forceinline__ Tan tmax(const Tan &a, double b) { return a.v < b ? Tan{b, 0.0} : a; }
__device__ __forceinline__ Tan tmax(double a, const Tan &b) { return a < b.v ? b : Tan{a, 0.0}; }
__device__ __forceinline__ double tmax(double a, double b) { return mx(a, b); }
__device__ __forceinline__ double der(const Tan &a) { return a.d; }
__device__ __forceinline__ double der(double) { return 0.0; }
// the input x itself where ON, else a value
template <bool ON> __device__ __forceinline__ auto seed(double x)
{
    if constexpr (ON) return Tan{x, 1.0};
    else return x;
}

// the neighbouring lane's value (lanes 2i and 2i + 1 exchange theirs)
__device__ __forceinline__ double swap_pair(double x)
{
    union { double d; int32_t i[2]; } u{x};
    u.i[0] = __builtin_amdgcn_update_dpp(0, u.i[0], 0xB1, 0xF, 0xF, true); // quad_perm [1, 0, 3, 2]
    u.i[1] = __builtin_amdgcn_update_dpp(0, u.i[1], 0xB1, 0xF, 0xF, true);
    return u.d;
}
// sum of the even lane's p in order, then the odd lane's, on both lanes of a pair
template <int N> __device__ __forceinline__ double pair_chain(const double (&p)[N], int32_t odd)
{
    double a = 0.0;
    for (int m = 0; m < N; ++m) a += p[m];
    double b = swap_pair(a);
    for (int m = 0; m < N; ++m) b += p[m];
    const double c = swap_pair(b);
    return odd ? b : c;
}

// sum over the block's threads, on every thread
__device__ __forceinline__ double block_sum(double v, double *sh)
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
// thread j < K: the sum over n rows of K values in the rows' order, the next stage's loads under way (blocks of NT
// threads; sh: kSumStage doubles)
template <int K, int NT> __device__ __forceinline__ double serial_sum(const double *x, int32_t n, double *sh)
{
    constexpr int32_t rows = kSumStage / K, per = (rows * K + NT - 1) / NT;
    const int32_t t = threadIdx.x;
    double v = 0.0, next[per];
    auto load = [&](int32_t r) {
#pragma unroll
        for (int32_t u = 0; u < per; ++u)
            if (r + rows > n ? t + u * NT < (n - r) * K : t + u * NT < rows * K) next[u] = x[size_t(r) * K + size_t(t + u * NT)];
    };
    if (n > 0) load(0);
    for (int32_t r = 0; r < n; r += rows)
    {
        __syncthreads();
#pragma unroll
        for (int32_t u = 0; u < per; ++u)
            if (t + u * NT < kSumStage) sh[t + u * NT] = next[u];
        __syncthreads();
        if (r + rows < n) load(r + rows);
        if (t < K)
#pragma unroll 8
            for (int32_t i = 0; i < min(rows, n - r); ++i) v += sh[i * K + t];
    }
    return v;
}

// the free stream's adjoint of a step: the face blocks' sums, then the cell blocks' (sh: kSumStage doubles)
__device__ __forceinline__ void free_stream_sums(const AdjFields &G, int32_t second_order, double *sh)
{
    const double a = serial_sum<10, kAdjThreads>(G.f_part, G.n_f, sh), b = serial_sum<10, kAdjThreads>(G.g_part, second_order ? G.n_c : 0, sh);
    if (threadIdx.x >= 10) return;
    const double x = G.sums[threadIdx.x] + a;
    G.sums[threadIdx.x] = second_order ? x + b : x;
}

// I = M^-1 of the reconstruction (Reconstruct.cpp:11-45) from M = sum |A| n n^T, in its operation order; false where it is zero
__device__ __forceinline__ bool normal_inverse(const double (&M)[3][3], double (&I)[3][3])
{
    const double det = M[0][0] * (M[1][1] * M[2][2] - M[1][2] * M[2][1]) - M[0][1] * (M[1][0] * M[2][2] - M[1][2] * M[2][0]) +
                       M[0][2] * (M[1][0] * M[2][1] - M[1][1] * M[2][0]);
    const double sc = mx(mx(mx(M[0][0], M[1][1]), M[2][2]), 1e-300);
    if (fabs(det) < 1e-12 * sc * sc * sc) return false;
    I[0][0] = (M[1][1] * M[2][2] - M[1][2] * M[2][1]) / det;
    I[0][1] = (M[0][2] * M[2][1] - M[0][1] * M[2][2]) / det;
    I[0][2] = (M[0][1] * M[1][2] - M[0][2] * M[1][1]) / det;
    I[1][0] = (M[1][2] * M[2][0] - M[1][0] * M[2][2]) / det;
    I[1][1] = (M[0][0] * M[2][2] - M[0][2] * M[2][0]) / det;
    I[1][2] = (M[0][2] * M[1][0] - M[0][0] * M[1][2]) / det;
    I[2][0] = (M[1][0] * M[2][1] - M[1][1] * M[2][0]) / det;
    I[2][1] = (M[0][1] * M[2][0] - M[0][0] * M[2][1]) / det;
    I[2][2] = (M[0][0] * M[1][1] - M[0][1] * M[1][0]) / det;
    return true;
}
__device__ __forceinline__ void normal_add(double (&M)[3][3], double A, const V3 &n)
{
    if (A <= 0) return;
    const double nv[3] = {n.x, n.y, n.z};
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) M[i][j] += A * nv[i] * nv[j];
}
// y with d(b . cell_vector) / d flux_f = n_f . y
__device__ __forceinline__ V3 normal_solve(const double (&M)[3][3], const V3 &b)
{
    double I[3][3];
    if (!normal_inverse(M, I)) return V3();
    return V3(I[0][0] * b.x + I[1][0] * b.y + I[2][0] * b.z, I[0][1] * b.x + I[1][1] * b.y + I[2][1] * b.z,
              I[0][2] * b.x + I[1][2] * b.y + I[2][2] * b.z);
}

// Forward Euler floors of the update (Solver.cpp:171-191)
template <class R> __device__ void floors(const Params &P, R q[5])
{
    const R ke = q[0] > 0 ? 0.5 * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]) / q[0] : R(0.0);
    if (!(q[0] >= P.rho_floor)) to_cons(PrimT<R>{P.rho_floor, 0, 0, 0, P.p_floor}, P.gamma, q);
    else if ((P.gamma - 1.0) * (q[4] - ke) < P.p_floor)
    {
        const PrimT<R> w = to_prim(q, P.gamma, P.rho_floor, P.p_floor);
        to_cons(w, P.gamma, q);
    }
}
// b = (d floors(q) / dq)^T b
__device__ __forceinline__ void floors_adjoint(const Params &P, const double (&q)[5], double (&b)[5])
{
    const double ke = q[0] > 0 ? 0.5 * (q[1] * q[1] + q[2] * q[2] + q[3] * q[3]) / q[0] : 0.0;
    if (q[0] >= P.rho_floor && !((P.gamma - 1.0) * (q[4] - ke) < P.p_floor)) return;
    double o[5];
#pragma unroll 1
    for (int j = 0; j < 5; ++j) // few cells
    {
        Dual x[5];
        for (int m = 0; m < 5; ++m) x[m] = Dual(q[m], m == j ? 1.0 : 0.0);
        floors<Dual>(P, x);
        double g = 0.0;
        for (int m = 0; m < 5; ++m) g += b[m] * x[m].d;
        o[j] = g;
    }
    for (int m = 0; m < 5; ++m) b[m] = o[m];
}

// ------------------------------------------------------------------------------------------------------------ roles
__device__ __forceinline__ double flux_bar(const DevMesh &d, const AdjFields &G, int32_t v)
{
    const int32_t f = pid(v);
    return G.all_active || d.fL[f] >= 0 || d.fR[f] >= 0 ? psg(v) * G.Phib[f] : 0.0;
}
// -Phib_f (d1 E)_f: the face's part of d/d dt through Faraday (Common/induction/Faraday.cpp:15-36)
__device__ __forceinline__ double faraday_dt(const DevMesh &d, const AdjFields &G, const double *E, int32_t f)
{
    if (f >= d.nf || (d.fL[f] < 0 && d.fR[f] < 0)) return 0.0;
    double circ = 0.0;
    if (d.fdeg == 3)
    {
        const int3 q = reinterpret_cast<const int3 *>(d.f2e)[f];
        const double x = E[pid(q.x)], y = E[pid(q.y)], z = E[pid(q.z)];
        circ += psg(q.x) * x;
        circ += psg(q.y) * y;
        circ += psg(q.z) * z;
    }
    else
        for (int32_t k = d.f2e_ptr[f]; k < d.f2e_ptr[f + 1]; ++k) circ += psg(d.f2e[k]) * E[pid(d.f2e[k])];
    return -G.Phib[f] * circ;
}
// l1b d l1 + l2b d l2 of (l1, l2) = uct_solve(M11, M12, M22, g1, g2) (fv.h) along its input J
template <int J> __device__ __forceinline__ double uct_column(const double (&in)[5], double l1b, double l2b)
{
    const auto M11 = seed<J == 0>(in[0]);
    const auto M12 = seed<J == 1>(in[1]);
    const auto M22 = seed<J == 2>(in[2]);
    const auto g1 = seed<J == 3>(in[3]);
    const auto g2 = seed<J == 4>(in[4]);
    const auto tr = M11 + M22, eps = 1e-14 * tr;
    const auto det = (M11 + eps) * (M22 + eps) - M12 * M12;
    const auto l1 = ((M22 + eps) * g1 - M12 * g2) / det;
    const auto l2 = ((M11 + eps) * g2 - M12 * g1) / det;
    return l1b * der(l1) + l2b * der(l2);
}
__device__ __forceinline__ void uct_solve_adjoint(const double (&in)[5], double l1b, double l2b, double (&sb)[5])
{
    const double tr = in[0] + in[2], eps = 1e-14 * tr, det = (in[0] + eps) * (in[2] + eps) - in[1] * in[1];
    for (int q = 0; q < 5; ++q) sb[q] = 0.0;
    if (!(tr > 0 && det > 0)) return;
    sb[0] = uct_column<0>(in, l1b, l2b);
    sb[1] = uct_column<1>(in, l1b, l2b);
    sb[2] = uct_column<2>(in, l1b, l2b);
    sb[3] = uct_column<3>(in, l1b, l2b);
    sb[4] = uct_column<4>(in, l1b, l2b);
}
// One face of the edge's UCT sum: the direction m, the normal, sig, aef = max_k |u_k . m| (first strict maximum, of cell k,
// kept as ~k for a negative u_k . m; kNoCell: none)
constexpr int32_t kNoCell = INT32_MIN;
struct UctFace { V3 m, nrm; double aef, sig; int32_t k; };
__device__ __forceinline__ UctFace uct_geometry(const DevMesh &d, int32_t f, int32_t e, const V3 &th)
{
    UctFace o;
    face_dirs(d, f, e, th, o.m, o.nrm);
    o.sig = dot(th, cross(o.m, o.nrm));
    o.aef = 0.0; o.k = kNoCell;
    return o;
}
__device__ __forceinline__ void uct_max(UctFace &o, int32_t k, const V3 &u)
{
    const double x = dot(u, o.m);
    if (o.aef < fabs(x)) { o.aef = fabs(x); o.k = x < 0 ? ~k : k; }
}
__device__ __forceinline__ void uct_q(const UctFace &u, const V3 &e1, const V3 &e2, double &qa, double &qb)
{
    const V3 qv = (u.aef * u.sig) * u.nrm;
    qa = dot(qv, e1);
    qb = dot(qv, e2);
}
// adjoint of aef, with the face's eF row written; w, pf: the face's weight and Phi / |A|
__device__ __forceinline__ double uct_face_adjoint(double w, double pf, double A, const UctFace &u, const V3 &e1, const V3 &e2, double l1,
                                                   double l2, double Eub, double Eb, const V3 &t, const double (&sb)[5], double *eF)
{
    double qa, qb;
    uct_q(u, e1, e2, qa, qb);
    const double omega = w * (1.0 - (qa * l1 + qb * l2));
    const double omb = Eub * u.aef * u.sig * pf;
    double aefb = Eub * omega * u.sig * pf;
    const double pfb = Eub * omega * u.aef * u.sig;
    const double qab = -omb * w * l1 + 2.0 * w * qa * sb[0] + w * qb * sb[1] + w * sb[3];
    const double qbb = -omb * w * l2 + w * qa * sb[1] + 2.0 * w * qb * sb[2] + w * sb[4];
    const V3 sn = u.sig * u.nrm;
    aefb += qab * dot(sn, e1) + qbb * dot(sn, e2);
    double2 *o = reinterpret_cast<double2 *>(eF);
    o[0] = make_double2(Eb * w * t.x, Eb * w * t.y);
    o[1] = make_double2(Eb * w * t.z, pfb / A);
    return aefb;
}

// Faraday and the UCT sum of an edge with the boundary EMF (IdealEMF.cpp:59-128, Solver.cpp:162-167), transposed:
// Eb_e = -dt sum over the active faces of sgn Phib_f.  One edge per thread; the usual valence keeps the row's cell
// velocities and per-face terms in registers; longer rows walk them again, their cells' sums in the slots.  einf: the
// edge's part of the imposed inflow EMF's adjoint (zero but on its edges).
__device__ __forceinline__ void edge_adjoint_light(const DevMesh &d, const StepFields &F, const AdjFields &G, double cuct, double dt, int32_t e,
                                                   double (&einf)[3])
{
    if (e >= d.ne) return;
    const int32_t f0 = d.e2f_ptr[e], nf = d.e2f_ptr[e + 1] - f0;
    const int8_t mode = d.emode[e];
    const bool heavy = nf > kLightMax; // a heavy block's, but for its part of the inflow EMF
    if (heavy && mode != 2) return;
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
    double Eb = -dt * acc;
    const V3 t = L3(d.evec, e);
    if (mode == 2) { einf[0] = Eb * t.x; einf[1] = Eb * t.y; einf[2] = Eb * t.z; }
    if (heavy) return;
    if (mode == 1 || mode == 2) Eb = 0.0;
    const double L = d.elen[e];
    if (!(Eb != 0.0 && nf > 0 && L > 0 && any_fluid))
    {
        for (int32_t i = 0; i < 4 * nf; ++i) eF[i] = 0.0;
        for (int32_t k = 0; k < 3 * nc; ++k) eC[k] = 0.0;
        return;
    }
    const V3 th = (1.0 / L) * t;
    V3 e1, e2;
    plane_basis(th, e1, e2);
    const double Eub = 2.0 * cuct * L * Eb;
    double M[5] = {0, 0, 0, 0, 0}, l1, l2, l1b = 0, l2b = 0, sb[5];
    // the face's terms of the 2x2 system and of its multipliers' adjoints, which do not depend on the solution
    auto sums = [&](const UctFace &u, int32_t f, double w) {
        double qa, qb;
        uct_q(u, e1, e2, qa, qb);
        M[0] += w * qa * qa; M[1] += w * qa * qb; M[2] += w * qb * qb; M[3] += w * qa; M[4] += w * qb;
        const double omb = Eub * u.aef * u.sig * F.Ef[4 * size_t(f) + 3];
        l1b -= omb * w * qa;
        l2b -= omb * w * qb;
    };
    auto adjoint = [&](const UctFace &u, int32_t f, int32_t i) {
        const double aefb = uct_face_adjoint(d.efw[f0 + i], F.Ef[4 * size_t(f) + 3], d.geo[4 * size_t(f) + 3], u, e1, e2, l1, l2, Eub, Eb, t, sb,
                                             eF + 4 * i);
        return aefb * psg(u.k);
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
                    UctFace u = uct_geometry(d, f, e, th);
#pragma unroll
                    for (int k = 0; k < kEmfFast; ++k)
                        if (k < nc) uct_max(u, k, uc[k]);
                    sums(u, f, d.efw[f0 + i]);
                    aef[i] = u.aef; km[i] = u.k;
                }
        }
        uct_solve(M[0], M[1], M[2], M[3], M[4], l1, l2);
        uct_solve_adjoint(M, l1b, l2b, sb);
        V3 ub[kEmfFast];
#pragma unroll
        for (int i = 0; i < kEmfFast; ++i)
            if (i < nf)
            {
                const int32_t f = pid(vid[i]);
                UctFace u = uct_geometry(d, f, e, th);
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
        UctFace u = uct_geometry(d, f, e, th);
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
    uct_solve_adjoint(M, l1b, l2b, sb);
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
__device__ __forceinline__ void edge_adjoint_heavy(const DevMesh &d, const StepFields &F, const AdjFields &G, double cuct, double dt, int32_t e,
                                                   double *sh, int32_t hv)
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
        const int8_t mode = d.emode[e];
        s_r[0] = mode == 1 || mode == 2 ? 0.0 : -dt * acc;
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
        UctFace u = uct_geometry(d, pid(d.e2f[f0 + i]), e, th);
        if (staged)
            for (int32_t k = 0; k < nc; ++k) uct_max(u, k, V3(x[k], y[k], z[k]));
        else
            for (int32_t k = 0; k < nc; ++k) uct_max(u, k, L3(F.uplus, d.ec_cell[c0 + k]));
        uct_q(u, e1, e2, sa[i], sbv[i]);
        saef[i] = u.aef; ssig[i] = u.sig;
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
            const double w = x[i], qa = sa[i], qb = sbv[i];
            M[0] += w * qa * qa; M[1] += w * qa * qb; M[2] += w * qb * qb; M[3] += w * qa; M[4] += w * qb;
        }
        uct_solve(M[0], M[1], M[2], M[3], M[4], l1, l2);
        for (int32_t i = 0; i < nf; ++i)
        {
            const double omb = Eub * saef[i] * ssig[i] * y[i];
            l1b -= omb * x[i] * sa[i];
            l2b -= omb * x[i] * sbv[i];
        }
        uct_solve_adjoint(M, l1b, l2b, sb);
        s_r[1] = l1; s_r[2] = l2;
        for (int q = 0; q < 5; ++q) s_r[3 + q] = sb[q];
    }
    __syncthreads();
    const double l1 = s_r[1], l2 = s_r[2], sb[5] = {s_r[3], s_r[4], s_r[5], s_r[6], s_r[7]};
    for (int32_t i = t0; i < nf; i += nt)
    {
        const int32_t f = pid(d.e2f[f0 + i]);
        UctFace u = uct_geometry(d, f, e, th);
        u.aef = saef[i]; u.k = sk[i];
        const double g = uct_face_adjoint(x[i], y[i], d.geo[4 * size_t(f) + 3], u, e1, e2, l1, l2, Eub, Eb, t, sb, eF + 4 * i) * psg(u.k);
        sk[i] = pid(u.k); // kNoCell becomes INT32_MAX, no cell's
        x[i] = g * u.m.x; y[i] = g * u.m.y; z[i] = g * u.m.z; // this thread's entries only until the barrier
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
// part through the update), the sources' parts of W, J, B_tot, the right-hand side's adjoint, the cell's part of d/d dt;
// thread (cell, ion)
template <int DEG>
__device__ __forceinline__ void update_adjoint_role(const DevMesh &d, const Params &P, const StepFields &F, const AdjFields &G, const SpC &Us,
                                                    const SpW &Ub, double dt, int32_t block)
{
    const int32_t t = threadIdx.x, s = t & 1, c = block * (kAdjThreads / kAdjNs) + (t >> 1);
    if (c >= d.nc) return;
    double dtb = 0.0, rb[5] = {0, 0, 0, 0, 0}, wb[5] = {0, 0, 0, 0, 0};
    V3 jb, bb;
    const double V = d.cvol[c];
    const double *row = F.rec + 16 * size_t(c), *W = row + 5 * s;
    if (d.mat[c] == 0) // the same for the cell's two threads
    {
        double rhs[5], q[5], qb[5], p[5];
        cell_rhs<DEG>(d, P, F, c, s, kAdjNs, row, V, dt, rhs);
        const double *u = Us.p[s] + 5 * size_t(c);
        double *ub = Ub.p[s] + 5 * size_t(c);
        for (int m = 0; m < 5; ++m) { q[m] = u[m] + dt * rhs[m]; qb[m] = ub[m]; }
        floors_adjoint(P, q, qb);
        for (int m = 0; m < 5; ++m)
        {
            ub[m] = qb[m];
            rb[m] = dt * qb[m];
            p[m] = rhs[m] * qb[m];
        }
        dtb = pair_chain(p, s);
        if (P.lorentz)
        {
            // S = ws J x B with ws = k n_s / D, D = sqrt(n_e^2 + floor^2); out += S, energy += u . S + dt S^2 / (2 rho).
            // Each input's column below is the derivative of the ion's S (sd) and energy term, weighted by rb and summed
            // over the two ions in order.
            const V3 Jc = L3(F.J, c), B = L3(F.Btot, c), C = cross(Jc, B), vel(W[1], W[2], W[3]);
            const double n0 = ion_density(P, 0, row[0]), n1 = ion_density(P, 1, row[5]), ns = s ? n1 : n0, ne = n0 + n1;
            const double D = sqrt(ne * ne + P.ne_floor * P.ne_floor), ws = ns / D, kw = P.inver_MA2 * ws;
            const V3 S = kw * C;
            const double rho = mx(W[0], 0.0), SS = dot(S, S), h = 0.5 * dt, hSS = h * SS, hq = hSS / rho;
            const bool kinetic = rho > 1e-30;
            auto column = [&](const V3 &sd, double rho_d) {
                const double SSd = (sd.x * S.x + S.x * sd.x) + (sd.y * S.y + S.y * sd.y) + (sd.z * S.z + S.z * sd.z);
                double e = vel.x * sd.x + vel.y * sd.y + vel.z * sd.z;
                if (kinetic) e += (h * SSd - hq * rho_d) / rho;
                const double x[4] = {rb[1] * sd.x, rb[2] * sd.y, rb[3] * sd.z, rb[4] * e};
                return pair_chain(x, s);
            };
            double rho_b[kAdjNs];
            for (int k = 0; k < kAdjNs; ++k)
            {
                const double nd = row[5 * k] < 0.0 ? 0.0 : 1.0 / P.M_s[k] * P.M_ref, Dd = D > 0 ? (nd * ne + ne * nd) / (2.0 * D) : 0.0;
                const double wd = ((k == s ? nd : 0.0) - ws * Dd) / D, kd = P.inver_MA2 * wd;
                rho_b[k] = column(V3(C.x * kd, C.y * kd, C.z * kd), k == s && !(W[0] < 0.0) ? 1.0 : 0.0);
            }
            wb[0] = s ? rho_b[1] : rho_b[0];
            wb[1] = rb[4] * S.x; wb[2] = rb[4] * S.y; wb[3] = rb[4] * S.z;
            jb.x = column(V3(0.0, -B.z * kw, B.y * kw), 0.0);
            jb.y = column(V3(B.z * kw, 0.0, -B.x * kw), 0.0);
            jb.z = column(V3(-B.y * kw, B.x * kw, 0.0), 0.0);
            bb.x = column(V3(0.0, Jc.z * kw, -Jc.y * kw), 0.0);
            bb.y = column(V3(-Jc.z * kw, 0.0, Jc.x * kw), 0.0);
            bb.z = column(V3(Jc.y * kw, -Jc.x * kw, 0.0), 0.0);
            const double x[1] = {rb[4] * (kinetic ? 0.5 * SS / rho : 0.0)};
            dtb += pair_chain(x, s);
        }
    }
    for (int m = 0; m < 5; ++m)
    {
        G.rv[10 * size_t(c) + 5 * s + m] = rb[m] / V;
        G.Wb[10 * size_t(c) + 5 * s + m] = wb[m];
    }
    if (s == 0) st3(G.Jv, c, (1.0 / V) * jb);
    else
    {
        st3(G.Btb, c, bb);
        G.dt_c[c] = dtb;
    }
}

// The first cell whose CFL step is dt (the blocks' minima in part), and the derivatives of its step by its primitives
// and field (MercurySources.cpp:104-145): one forward-mode column per thread
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
    if (s_b != INT32_MAX)
    {
        const int32_t c = s_b * 256 + t;
        const double *w[kMaxSpecies];
        if (c < d.nc && d.mat[c] == 0)
        {
            for (int s = 0; s < kAdjNs; ++s) w[s] = F.rec + 16 * size_t(c) + 5 * s;
            if (cell_dt<double>(d, P, c, w, L3(F.Btot, c), 0) == dt) atomicMin(&s_c, c);
        }
    }
    __syncthreads();
    const int32_t c = s_c;
    if (c == INT32_MAX)
    {
        if (t == 0) { G.dt_cell[0] = -1; ++G.dt_cell[1]; }
        return;
    }
    if (t == 0) G.dt_cell[0] = c;
    if (t >= 5 * kAdjNs + 3) return;
    Dual w[kAdjNs][5];
    const Dual *wp[kMaxSpecies];
    for (int s = 0; s < kAdjNs; ++s)
    {
        for (int m = 0; m < 5; ++m) w[s][m] = Dual(F.rec[16 * size_t(c) + 5 * s + m], t == 5 * s + m ? 1.0 : 0.0);
        wp[s] = w[s];
    }
    const int32_t o = t - 5 * kAdjNs;
    const V3 b = L3(F.Btot, c);
    const V3D bd(Dual(b.x, o == 0 ? 1.0 : 0.0), Dual(b.y, o == 1 ? 1.0 : 0.0), Dual(b.z, o == 2 ? 1.0 : 0.0));
    G.dtb[1 + t] = cell_dt<Dual>(d, P, c, wp, bd, 0).d;
}

// sum_m Fb_m dF_m of the Rusanov flux (Common/physics/Euler.h:29-49) along primitive J of one side: w the side's state,
// E its energy, U0, F0, s0 the other side's conserved state, flux and speed
template <int J, bool LEFT>
__device__ __forceinline__ double rusanov_column(const Prim &w, const V3 &n, double gamma, const double (&U0)[5], const double (&F0)[5], double s0,
                                                 const double (&Fb)[5])
{
    const auto rho = seed<J == 0>(w.rho);
    const auto u = seed<J == 1>(w.u);
    const auto v = seed<J == 2>(w.v);
    const auto ww = seed<J == 3>(w.w);
    const auto p = seed<J == 4>(w.p);
    const auto U1 = rho * u;
    const auto U2 = rho * v;
    const auto U3 = rho * ww;
    const auto U4 = p / (gamma - 1.0) + 0.5 * rho * (u * u + v * v + ww * ww);
    const auto un = u * n.x + v * n.y + ww * n.z;
    const auto F1 = rho * un * u + p * n.x;
    const auto F2 = rho * un * v + p * n.y;
    const auto F3 = rho * un * ww + p * n.z;
    const auto F4 = un * (U4 + p);
    const auto sw = tabs(un) + tsqrt(gamma * p / rho);
    auto flux = [&](const auto &U, const auto &F, int m) {
        if constexpr (LEFT) return Fb[m] * der(0.5 * (F + F0[m]) - 0.5 * tmax(sw, s0) * (U0[m] - U));
        else return Fb[m] * der(0.5 * (F0[m] + F) - 0.5 * tmax(s0, sw) * (U - U0[m]));
    };
    double g = 0.0;
    g += flux(rho, rho * un, 0);
    g += flux(U1, F1, 1);
    g += flux(U2, F2, 2);
    g += flux(U3, F3, 3);
    g += flux(U4, F4, 4);
    return g;
}
__device__ __forceinline__ void rusanov_side(const Prim &w, const V3 &n, double gamma, double (&U)[5], double (&F)[5], double &s)
{
    to_cons(w, gamma, U);
    const double un = w.u * n.x + w.v * n.y + w.w * n.z;
    F[0] = w.rho * un; F[1] = w.rho * un * w.u + w.p * n.x; F[2] = w.rho * un * w.v + w.p * n.y; F[3] = w.rho * un * w.w + w.p * n.z;
    F[4] = un * (U[4] + w.p);
    s = fabs(un) + sqrt(gamma * w.p / w.rho);
}
// Lb, Rb = (dF/dL)^T Fb, (dF/dR)^T Fb
__device__ __forceinline__ void rusanov_adjoint(const Prim &L, const Prim &R, const V3 &n, double gamma, const double (&Fb)[5], double (&Lb)[5],
                                                double (&Rb)[5])
{
    double UL[5], UR[5], FL[5], FR[5], sL, sR;
    rusanov_side(L, n, gamma, UL, FL, sL);
    rusanov_side(R, n, gamma, UR, FR, sR);
    Lb[0] = rusanov_column<0, true>(L, n, gamma, UR, FR, sR, Fb);
    Lb[1] = rusanov_column<1, true>(L, n, gamma, UR, FR, sR, Fb);
    Lb[2] = rusanov_column<2, true>(L, n, gamma, UR, FR, sR, Fb);
    Lb[3] = rusanov_column<3, true>(L, n, gamma, UR, FR, sR, Fb);
    Lb[4] = rusanov_column<4, true>(L, n, gamma, UR, FR, sR, Fb);
    Rb[0] = rusanov_column<0, false>(R, n, gamma, UL, FL, sL, Fb);
    Rb[1] = rusanov_column<1, false>(R, n, gamma, UL, FL, sL, Fb);
    Rb[2] = rusanov_column<2, false>(R, n, gamma, UL, FL, sL, Fb);
    Rb[3] = rusanov_column<3, false>(R, n, gamma, UL, FL, sL, Fb);
    Rb[4] = rusanov_column<4, false>(R, n, gamma, UL, FL, sL, Fb);
}

// Face fluxes transposed: thread (face, ion).  Replaces the face states of the face's entries by their adjoints; in the
// 256-face blocks with an inflow face the free stream's parts go to their rows.
__device__ __forceinline__ void flux_adjoint_role(const DevMesh &d, const Params &P, const StepFields &F, const AdjFields &G, int32_t block)
{
    const int32_t t = threadIdx.x, s = t & 1, f = block * (kAdjThreads / kAdjNs) + (t >> 1);
    if (f >= d.nf) return;
    double fsb[5] = {0, 0, 0, 0, 0};
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
        if (nz)
        {
            // one call for both kinds of face: of a boundary face one side is the ghost
            const bool left = cls != kFluxRight, inner = cls == kFluxInner;
            const int8_t kind = d.kind[f];
            const V3 no = (left ? 1.0 : -1.0) * n;
            Prim L, R, in = state(left ? qL : qR), other;
            if (inner) other = state(qR);
            else
            {
                double fs[5];
                for (int m = 0; m < 5; ++m) fs[m] = P.fs[s][m];
                other = ghost_state(kind, s, in, no, fs);
            }
            if (left) { L = in; R = other; } else { L = other; R = in; }
            rusanov_adjoint(L, R, n, P.gamma, Fb, Lb, Rb);
            if (!inner)
            {
                double ib[5], gb[5];
                for (int m = 0; m < 5; ++m) { ib[m] = left ? Lb[m] : Rb[m]; gb[m] = left ? Rb[m] : Lb[m]; }
                if (kind == kInflow)
                    for (int m = 0; m < 5; ++m) fsb[m] = gb[m];
                else if (!(kind == kWall && s == 1)) // the ghost is the cell's own state, mirrored at a wall
                {
                    if (kind == kWall)
                    {
                        const double ndg = no.x * gb[1] + no.y * gb[2] + no.z * gb[3];
                        gb[1] -= 2.0 * ndg * no.x; gb[2] -= 2.0 * ndg * no.y; gb[3] -= 2.0 * ndg * no.z;
                    }
                    for (int m = 0; m < 5; ++m) ib[m] += gb[m];
                }
                for (int m = 0; m < 5; ++m) { Lb[m] = left ? ib[m] : 0.0; Rb[m] = left ? 0.0 : ib[m]; }
            }
        }
    }
    if (e.x >= 0)
        for (int m = 0; m < 5; ++m) qL[m] = Lb[m];
    if (e.y >= 0)
        for (int m = 0; m < 5; ++m) qR[m] = Rb[m];
    const int32_t slot = G.fs_face[f >> 8];
    if (slot >= 0)
        for (int m = 0; m < 5; ++m) G.fsf[10 * (256 * size_t(slot) + size_t(f & 255)) + 5 * s + m] = fsb[m];
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
    if (l < 0 && r < 0) { G.Phib[f] += pb; return; }
    const int2 e = F.fent[f];
    double A;
    const V3 n = geo_normal(d, f, A), Fb = cross(n, Eb);
    const double Bn = (Phi[f] + PhiAdd[f]) / A;
    const double *Bi = F.rec + 5 * kAdjNs;
    double Bnb = 0.0;
    // the parts of cell c's u+ and B_tot from the adjoint fxb of its side
    auto side = [&](const V3 &u, const V3 &B, const V3 &fxb, V3 &ub, V3 &bt) {
        ub = dot(B, fxb) * n - Bn * fxb;
        bt = dot(u, n) * fxb;
        Bnb -= dot(u, fxb);
    };
    auto put = [&](int32_t k, const V3 &ub, const V3 &bt, const V3 &bi) {
        if (k < 0) return;
        double *o = G.sE + 9 * size_t(k);
        o[0] = ub.x; o[1] = ub.y; o[2] = ub.z; o[3] = bt.x; o[4] = bt.y; o[5] = bt.z; o[6] = bi.x; o[7] = bi.y; o[8] = bi.z;
    };
    if (l >= 0 && r >= 0)
    {
        const V3 uL = L3(F.uplus, l), uR = L3(F.uplus, r), tL = L3(F.Btot, l), tR = L3(F.Btot, r);
        const V3 db = L3(Bi + 16 * size_t(r), 0) - L3(Bi + 16 * size_t(l), 0), h = 0.5 * Fb;
        const double vL = dot(uL, n), vR = dot(uR, n), aL = fabs(vL), aR = fabs(vR), a = aL < aR ? aR : aL;
        V3 ubL, ubR, btL, btR;
        side(uL, tL, h, ubL, btL);
        side(uR, tR, h, ubR, btR);
        const double ab = -0.5 * dot(Fb, db);
        const bool right = aL < aR;
        const double sgn = (right ? vR : vL) < 0 ? -1.0 : 1.0;
        (right ? ubR : ubL) += (ab * sgn) * n;
        const V3 bi = (0.5 * a) * Fb;
        put(e.x, ubL, btL, bi);
        put(e.y, ubR, btR, -1.0 * bi);
    }
    else
    {
        const int32_t c = l >= 0 ? l : r;
        V3 ub, bt;
        side(L3(F.uplus, c), L3(F.Btot, c), Fb, ub, bt);
        put(c == l ? e.x : e.y, ub, bt, V3());
    }
    const double x = G.Phib[f] + pb;
    G.Phib[f] = x + Bnb / A;
    G.PhiAddb[f] += Bnb / A;
}
} // namespace

// ---------------------------------------------------------------------------------------------------------- kernels
// Dynamic LDS: the heavy edges' rows, and kSumStage doubles
template <int DEG>
__global__ void __launch_bounds__(kAdjThreads, 3) k_adj_update(DevMesh d, Params P, StepFields F, AdjFields G, SpC Us, SpW Ub, const double *E,
                                                            double dt, const int32_t *heavy, int32_t n_heavy, int32_t hv, int32_t n_dt,
                                                            const double *dt_part, int32_t n_part, int32_t n_sum, int32_t n_edge, int32_t n_face)
{
    extern __shared__ double rows[];
    __shared__ double sh[kAdjThreads];
    const int32_t t = threadIdx.x;
    int32_t b = blockIdx.x, first = n_heavy + n_dt + n_sum;
    if (b < n_heavy) edge_adjoint_heavy(d, F, G, P.cuct, dt, heavy[b], rows, hv);
    else if (b < n_heavy + n_dt) dt_cell_role(d, P, F, G, dt_part, n_part, dt);
    else if (b < first) free_stream_sums(G, P.second_order, rows); // of the step before in the sweep
    else if (b < first + n_edge)
    {
        const int32_t i = near_block(d, b, first, n_edge), slot = G.inflow_edge[i];
        double einf[3] = {0, 0, 0};
        edge_adjoint_light(d, F, G, P.cuct, dt, i * kAdjThreads + t, einf);
        if (slot >= 0)
            for (int q = 0; q < 3; ++q)
            {
                const double x = block_sum(einf[q], sh);
                if (t == 0) G.e_part[3 * size_t(slot) + q] = x;
            }
    }
    else if (first += n_edge; b < first + n_face)
    {
        const int32_t i = near_block(d, b, first, n_face);
        const double x = block_sum(faraday_dt(d, G, E, i * kAdjThreads + t), sh);
        if (t == 0) G.dt_f[i] = x;
    }
    else
    {
        first += n_face;
        update_adjoint_role<DEG>(d, P, F, G, Us, Ub, dt, near_block(d, b, first, int32_t(gridDim.x) - first));
    }
}

__global__ void __launch_bounds__(kAdjThreads) k_adj_faces(DevMesh d, Params P, StepFields F, AdjFields G, const double *Phi, const double *PhiAdd,
                                                           int32_t n_cell, int32_t n_emf)
{
    __shared__ double sh[kSumStage];
    const int32_t b = blockIdx.x, t = threadIdx.x;
    if (b == 0)
    {
        const double x = serial_sum<3, kAdjThreads>(G.e_part, G.n_e, sh);
        if (t < 3) G.sums[10 + t] += x;
    }
    else if (b <= n_cell)
    {
        const int32_t c = (b - 1) * kAdjThreads + t;
        const double x = block_sum(c < d.nc ? G.dt_c[c] : 0.0, sh);
        if (t == 0) G.dt_cp[b - 1] = x;
    }
    else if (b <= n_cell + n_emf)
        face_emf_adjoint_role(d, F, G, Phi, PhiAdd, near_block(d, b, 1 + n_cell, n_emf) * kAdjThreads + t);
    else flux_adjoint_role(d, P, F, G, near_block(d, b, 1 + n_cell + n_emf, int32_t(gridDim.x) - 1 - n_cell - n_emf));
}

namespace
{
// Whose value a stencil entry takes: the row's first entry of that neighbour, or one of these: the free stream's, none of
// the others', the cell's own (boundary values that follow it, mirrored velocities among them)
constexpr int32_t kFree = -1, kOther = -2, kOwnCell = -3;
// The stencil of one ion of a cell (Reconstruction.cpp:26-78): a fixed row in registers (its face offsets in `offsets`), or
// (DEG 0) walked in memory
template <int DEG> struct StencilRow
{
    static constexpr int N = DEG > 0 ? DEG : 1;
    const DevMesh &d;
    const Params &P;
    const StepFields &F;
    const double *offsets;
    int32_t c, s, k0, nk, v[N], nb[N], src[N];
    double wc[5], wn[N][5];
    V3 xc, wd[N];
    __device__ __forceinline__ StencilRow(const DevMesh &d, const Params &P, const StepFields &F, int32_t c, int32_t s, const double *offsets)
        : d(d), P(P), F(F), offsets(offsets), c(c), s(s)
    {
        const double *own = F.rec + 16 * size_t(c);
        row_of<DEG>(d, c, k0, nk);
        xc = V3(own[13], own[14], own[15]);
        for (int m = 0; m < 5; ++m) wc[m] = own[5 * s + m];
        if constexpr (DEG > 0)
        {
            row_ids<DEG>(d.c2f, k0, v);
            row_ids<DEG>(d.snb, k0, nb);
#pragma unroll
            for (int i = 0; i < DEG; ++i)
            {
                src[i] = find_source(i);
                find_value(i, wn[i]);
                wd[i] = find_weighted(i);
            }
        }
    }
    __device__ __forceinline__ int count() const { return DEG > 0 ? DEG : nk; }
    __device__ __forceinline__ int32_t face(int i) const { return DEG > 0 ? v[i] : d.c2f[k0 + i]; }
    __device__ __forceinline__ int32_t across(int i) const { return DEG > 0 ? nb[i] : d.snb[k0 + i]; }
    __device__ __forceinline__ int8_t kind(int i) const
    {
        const int32_t o = across(i);
        return o >= 0 ? int8_t(kInterior) : o == kNoStencil ? int8_t(kSkip) : d.kind[-(o + 1)];
    }
    __device__ __forceinline__ V3 normal(int i) const
    {
        double A;
        return psg(face(i)) * geo_normal(d, pid(face(i)), A);
    }
    __device__ __forceinline__ int32_t find_source(int i) const
    {
        const int32_t o = across(i);
        if (o < 0) return kind(i) == kInflow ? kFree : kind(i) == kWall && s == 1 ? kOther : kOwnCell;
        if (o == c) return kOwnCell;
        int32_t j = i;
#pragma unroll
        for (int q = (DEG > 0 ? DEG : i + 1) - 1; q >= 0; --q)
            if (q < i && across(q) == o) j = q;
        return j;
    }
    __device__ __forceinline__ void find_value(int i, double (&w)[5]) const
    {
        const int32_t o = across(i);
        double fs[5];
        for (int m = 0; m < 5; ++m) { fs[m] = P.fs[s][m]; w[m] = wc[m]; }
        if (o >= 0)
            for (int m = 0; m < 5; ++m) w[m] = F.rec[16 * size_t(o) + 5 * s + m];
        else if (o != kNoStencil) stencil_ghost(d, s, static_cast<const double *>(nullptr), wc, fs, face(i), o, w);
    }
    // the offset over its square, zero for an entry without a stencil
    __device__ __forceinline__ V3 find_weighted(int i) const
    {
        const int32_t o = across(i);
        if (o == kNoStencil) return V3();
        V3 q;
        if (o >= 0)
        {
            const double *r = F.rec + 16 * size_t(o);
            q = V3(r[13], r[14], r[15]) - xc;
        }
        else
        {
            const V3 n = normal(i);
            q = (2.0 * dot(L3(d.fcen, pid(face(i))) - xc, n)) * n;
        }
        return (1.0 / dot(q, q)) * q;
    }
    __device__ __forceinline__ int32_t source(int i) const { return DEG > 0 ? src[i] : find_source(i); }
    __device__ __forceinline__ V3 weighted(int i) const { return DEG > 0 ? wd[i] : find_weighted(i); }
    __device__ __forceinline__ V3 dx(int i) const { return DEG > 0 ? L3(offsets, i) : L3(d.fcen, pid(face(i))) - xc; }
    __device__ __forceinline__ double value(int i, int m) const
    {
        if constexpr (DEG > 0) return wn[i][m];
        else
        {
            double w[5];
            find_value(i, w);
            return m == 0 ? w[0] : m == 1 ? w[1] : m == 2 ? w[2] : m == 3 ? w[3] : w[4];
        }
    }
};
// the symmetric inverse of the stencil's normal matrix
struct StencilInverse
{
    double a, b, c, d, e, f;
    __device__ __forceinline__ explicit StencilInverse(const double *I) : a(I[0]), b(I[1]), c(I[2]), d(I[3]), e(I[4]), f(I[5]) {}
    __device__ __forceinline__ V3 operator()(const V3 &r) const
    {
        return V3(a * r.x + b * r.y + c * r.z, b * r.x + d * r.y + e * r.z, c * r.x + e * r.y + f * r.z);
    }
};
// A primitive's gradient g, its limiter psi and what sets it (kNoLimit: nothing): the room to an extreme or the relative
// limit over dl = g . x, x the offset of its face; and whose the extremes are (source)
enum : int32_t { kNoLimit, kRoom, kRelative };
struct Limited
{
    V3 g, x;
    double psi, dl;
    int32_t by, hs, ls;
    // the derivative of psi g along an input that moves g by gd, the extremes by hd and ld and the cell's value by wd
    __device__ __forceinline__ V3 column(const Params &P, const V3 &gd, double hd, double ld, double wd) const
    {
        double pd = 0.0;
        if (by != kNoLimit)
        {
            double dld = gd.x * x.x + gd.y * x.y + gd.z * x.z, num, den = dl;
            if (by == kRelative)
            {
                num = P.rel_limit * wd;
                if (dl < 0) { dld = -dld; den = -dl; }
            }
            else num = (dl > 0 ? hd : ld) - wd;
            pd = (num - psi * dld) / den;
        }
        return V3(pd * g.x + psi * gd.x, pd * g.y + psi * gd.y, pd * g.z + psi * gd.z);
    }
};
template <int DEG> __device__ __forceinline__ Limited limited(const Params &P, const StencilRow<DEG> &row, const StencilInverse &inv, int m)
{
    Limited L;
    const double w = m == 0 ? row.wc[0] : m == 1 ? row.wc[1] : m == 2 ? row.wc[2] : m == 3 ? row.wc[3] : row.wc[4];
    double lo = w, hi = w;
    V3 r;
    L.hs = L.ls = kOwnCell;
#pragma unroll
    for (int i = 0; i < row.count(); ++i)
    {
        const double q = row.value(i, m), dq = q - w;
        const V3 a = row.weighted(i);
        r.x += a.x * dq; r.y += a.y * dq; r.z += a.z * dq;
        if (q < lo) { lo = q; L.ls = row.source(i); }
        if (hi < q) { hi = q; L.hs = row.source(i); }
    }
    L.g = inv(r);
    L.psi = 1.0;
    L.by = kNoLimit;
    L.dl = 0.0;
    // psi = max(0, min(1, quotients)): the first smallest quotient below 1 counts, unless it is not above 0
#pragma unroll
    for (int i = 0; i < row.count(); ++i)
    {
        const V3 x = row.dx(i);
        const double dl = L.g.x * x.x + L.g.y * x.y + L.g.z * x.z, q = (dl > 0 ? hi - w : lo - w) / dl;
        if (fabs(dl) > 1e-300 && q < L.psi) { L.psi = q; L.by = kRoom; L.x = x; L.dl = dl; }
    }
    if (P.rel_limit > 0 && (m == 0 || m == 4))
#pragma unroll
        for (int i = 0; i < row.count(); ++i)
        {
            const V3 x = row.dx(i);
            const double dl = L.g.x * x.x + L.g.y * x.y + L.g.z * x.z, q = P.rel_limit * w / fabs(dl);
            if (fabs(dl) > 1e-300 && q < L.psi) { L.psi = q; L.by = kRelative; L.x = x; L.dl = dl; }
        }
    if (!(L.psi > 0.0)) { L.psi = 0.0; L.by = kNoLimit; }
    return L;
}
// Whether an entry's state is the linear one (else it is the cell's own): a face state depends on the gradient there.  A bit
// per entry of a fixed row; walked rows, which may be longer than a word, form it again.
template <int DEG> struct LinearEntries
{
    V3 a, b; // the limited gradients of density and pressure
    uint32_t bits = 0;
    __device__ __forceinline__ LinearEntries(const StencilRow<DEG> &row, const Limited &rho, const Limited &p)
        : a(rho.psi * rho.g.x, rho.psi * rho.g.y, rho.psi * rho.g.z), b(p.psi * p.g.x, p.psi * p.g.y, p.psi * p.g.z)
    {
        if constexpr (DEG > 0)
#pragma unroll
            for (int i = 0; i < DEG; ++i) bits |= uint32_t(positive(row, i)) << i;
    }
    __device__ __forceinline__ bool positive(const StencilRow<DEG> &row, int i) const
    {
        const V3 x = row.dx(i);
        const double rr = row.wc[0] + a.x * x.x + a.y * x.y + a.z * x.z, pp = row.wc[4] + b.x * x.x + b.y * x.y + b.z * x.z;
        return rr > 0 && pp > 0;
    }
    __device__ __forceinline__ bool operator()(const StencilRow<DEG> &row, int i) const { return DEG > 0 ? bits >> i & 1 : positive(row, i); }
};
} // namespace

// The first ion's velocities of a wall cell, which its mirror image couples: thread (wall cell, component j), the part of
// velocity j in the cell's limited gradients.  A launch of its own ahead of k_adj_gradients, which adds
// it: there the coupling's nine derivatives made half of the waves, those with a wall cell, wait for a few lanes.
template <int DEG> __global__ void __launch_bounds__(64, 2) k_adj_mirror(DevMesh d, Params P, StepFields F, AdjFields G)
{
    __shared__ double face_dx[DEG > 0 ? 64 * (3 * DEG + 1) : 1];
    const int32_t i0 = gid(), j = i0 % 3 + 1, slot = i0 / 3;
    if (slot >= G.n_wall) return;
    const int32_t c = G.wall_cell[slot];
    double *const offsets = face_dx + int32_t(threadIdx.x) * (3 * DEG + 1);
    const StencilRow<DEG> row(d, P, F, c, 0, offsets);
    if constexpr (DEG > 0)
#pragma unroll
        for (int i = 0; i < DEG; ++i) st3(offsets, i, L3(d.fcen, pid(row.v[i])) - row.xc); // this thread's own
    const StencilInverse inv(d.sinv + 6 * size_t(c));
    auto bar = [&](int i) { return F.FS + 5 * (size_t(row.k0 + i) * kAdjNs); };
    const LinearEntries<DEG> linear(row, limited(P, row, inv, 0), limited(P, row, inv, 4));
    double sum = 0.0;
#pragma unroll
    for (int m = 1; m <= 3; ++m)
    {
        const Limited L = limited(P, row, inv, m);
        const double w = m == 1 ? row.wc[1] : m == 2 ? row.wc[2] : row.wc[3], wd = m == j ? 1.0 : 0.0;
        double hd = wd, ld = wd, lo = w, hi = w;
        V3 gb, rd;
#pragma unroll
        for (int i = 0; i < row.count(); ++i)
        {
            if (linear(row, i)) gb += bar(i)[m] * row.dx(i);
            double nd = row.source(i) == kOwnCell ? wd : 0.0; // the entry's value along velocity j
            if (row.kind(i) == kWall)
            {
                const V3 n = row.normal(i);
                const double nj = j == 1 ? n.x : j == 2 ? n.y : n.z, nm = m == 1 ? n.x : m == 2 ? n.y : n.z;
                nd -= 2.0 * nj * nm;
            }
            const double q = row.value(i, m), dq = nd - wd;
            const V3 a = row.weighted(i);
            rd += V3(a.x * dq, a.y * dq, a.z * dq);
            if (q < lo) { lo = q; ld = nd; }
            if (hi < q) { hi = q; hd = nd; }
        }
        const V3 o = L.column(P, inv(rd), hd, ld, wd);
        sum += gb.x * o.x; sum += gb.y * o.y; sum += gb.z * o.z;
    }
    G.mirror[i0] = sum;
}

// Limited gradients (Reconstruction.cpp:80-142) and the states formed from them (FluxRHS.cpp:16-27), transposed: thread
// (cell, ion), with the forward's operations up to the limiters.  In: the adjoints of the cell's face states; Wb +=
// the cell's own part, the entries receive the parts of the stencil neighbours' primitives.
//
// A primitive's limited gradient is psi g with g = I sum_k w_k d_k (q_k - q_c), psi the limiting quotient, so its
// derivative along the primitive of a neighbour (or of the cell) needs one vector I w_k d_k (or I times minus their sum),
// the same for all five, and one quotient per limited primitive.
template <int DEG>
__global__ void __launch_bounds__(kGradThreads, 2) k_adj_gradients(DevMesh d, Params P, StepFields F, AdjFields G, int32_t n_cell)
{
    constexpr int kCells = kGradThreads / kAdjNs;
    constexpr int kStage = kGradThreads * (DEG > 0 ? 5 * DEG : 1);
    __shared__ double stage[kStage > kSumStage ? kStage : kSumStage];
    __shared__ double face_dx[DEG > 0 ? kCells * (3 * DEG + 1) : 1]; // a cell's two threads share them (an odd row: no bank conflicts)
    const int32_t t = threadIdx.x, s = t & 1, cl = t >> 1;
    if (blockIdx.x == 0)
    {
        // adjoint of the time step: the faces' and the cells' parts
        const double a = serial_sum<1, kGradThreads>(G.dt_f, (d.nf + 255) / 256, stage), b = serial_sum<1, kGradThreads>(G.dt_cp, (d.nc + 255) / 256, stage);
        if (t == 0) G.dtb[0] = a + b;
        return;
    }
    const int32_t c0 = near_block(d, int32_t(blockIdx.x), 1, n_cell) * kCells, c = c0 + cl;
    const int32_t n_here = min(kCells, d.nc - c0) * (DEG * kAdjNs * 5 / 2);
    double *const offsets = face_dx + cl * (3 * DEG + 1);
    if constexpr (DEG > 0)
    {
        if (c < d.nc)
        {
            const V3 xc(F.rec[16 * size_t(c) + 13], F.rec[16 * size_t(c) + 14], F.rec[16 * size_t(c) + 15]);
#pragma unroll
            for (int i = 0; i < DEG; i += 2) st3(offsets, i + s, L3(d.fcen, pid(d.c2f[DEG * c + i + s])) - xc);
        }
        const double2 *src = reinterpret_cast<const double2 *>(F.FS + size_t(c0) * size_t(DEG * 5 * kAdjNs));
        double2 *dst = reinterpret_cast<double2 *>(stage);
        for (int32_t i = t; i < n_here; i += kGradThreads) dst[i] = src[i];
        __syncthreads();
    }
    if (c < d.nc)
    {
        const int32_t slot = G.fs_cell[c >> 8], wall = s == 0 ? G.wall_slot[c] : -1;
        double *const wb = G.Wb + 10 * size_t(c) + 5 * s;
        double *const fsb = G.fsc + 10 * (256 * size_t(slot < 0 ? 0 : slot) + size_t(c & 255)) + 5 * s;
        if (slot >= 0)
            for (int m = 0; m < 5; ++m) fsb[m] = 0.0;
        int32_t k0, nk;
        row_of<DEG>(d, c, k0, nk);
        auto bar = [&](int i) { return DEG > 0 ? stage + 5 * ((cl * DEG + i) * kAdjNs + s) : F.FS + 5 * (size_t(k0 + i) * kAdjNs + s); };
        if (!(P.second_order && d.svalid[c])) // the states are the cell's own
#pragma unroll 1
            for (int m = 0; m < 5; ++m)
            {
                double sum = 0.0;
                for (int i = 0; i < nk; ++i) { sum += bar(i)[m]; bar(i)[m] = 0.0; }
                wb[m] += sum;
            }
        else
        {
            const StencilRow<DEG> row(d, P, F, c, s, offsets);
            const StencilInverse inv(d.sinv + 6 * size_t(c));
            Limited L = limited(P, row, inv, 0);
            const LinearEntries<DEG> linear(row, L, limited(P, row, inv, 4));
            // I times the sum of w d dq along the cell's own primitive; a value that follows the cell's adds nothing
            bool nz = false, inflow = false; // some gradient has an adjoint; a face of the inflow
            V3 rc;
#pragma unroll
            for (int i = 0; i < row.count(); ++i)
            {
                for (int m = 0; m < 5; ++m) nz = nz || (linear(row, i) && bar(i)[m] != 0.0);
                inflow = inflow || row.source(i) == kFree;
                if (row.source(i) != kOwnCell) rc -= row.weighted(i);
            }
            const V3 gc = inv(rc);
#pragma unroll
            for (int m = 0; m < 5; ++m)
            {
                if (m > 0) L = limited(P, row, inv, m);
                double sum = 0.0;
                V3 gb;
#pragma unroll
                for (int i = 0; i < row.count(); ++i)
                {
                    const double b = bar(i)[m];
                    sum += b;
                    if (linear(row, i)) gb += b * row.dx(i);
                }
                auto weigh = [&](const V3 &o) { return gb.x * o.x + gb.y * o.y + gb.z * o.z; };
                sum = wb[m] + sum;
                if (nz)
                {
                    if (wall >= 0 && m >= 1 && m <= 3) sum += G.mirror[3 * size_t(wall) + m - 1];
                    else sum += weigh(L.column(P, gc, L.hs == kOwnCell ? 1.0 : 0.0, L.ls == kOwnCell ? 1.0 : 0.0, 1.0));
                    if (inflow)
                    {
                        V3 r;
#pragma unroll
                        for (int i = 0; i < row.count(); ++i)
                            if (row.source(i) == kFree) r += row.weighted(i);
                        fsb[m] = weigh(L.column(P, inv(r), L.hs == kFree ? 1.0 : 0.0, L.ls == kFree ? 1.0 : 0.0, 0.0));
                    }
                }
                wb[m] = sum;
                // a neighbour's part, of its entries together, on the first of them
#pragma unroll
                for (int i = 0; i < row.count(); ++i)
                {
                    double q = 0.0;
                    if (nz && row.source(i) == i)
                    {
                        V3 r = row.weighted(i);
#pragma unroll
                        for (int j = 1; j < row.count(); ++j)
                            if (j > i && row.source(j) == i) r += row.weighted(j);
                        q = weigh(L.column(P, inv(r), L.hs == i ? 1.0 : 0.0, L.ls == i ? 1.0 : 0.0, 0.0));
                    }
                    bar(i)[m] = q;
                }
            }
        }
    }
    if constexpr (DEG > 0)
    {
        __syncthreads();
        double2 *dst = reinterpret_cast<double2 *>(F.FS + size_t(c0) * size_t(DEG * 5 * kAdjNs));
        const double2 *src = reinterpret_cast<const double2 *>(stage);
        for (int32_t i = t; i < n_here; i += kGradThreads) dst[i] = src[i];
    }
}

namespace
{
// sum_m b_m d(primitive m) / d U_J of the primitive recovery (Euler.h:13-27)
template <int J> __device__ __forceinline__ double prim_column(const Params &P, const double *U, const double (&b)[5])
{
    const auto U0 = seed<J == 0>(U[0]);
    const auto U1 = seed<J == 1>(U[1]);
    const auto U2 = seed<J == 2>(U[2]);
    const auto U3 = seed<J == 3>(U[3]);
    const auto U4 = seed<J == 4>(U[4]);
    const auto rho = tmax(U0, P.rho_floor);
    const auto u = U1 / rho;
    const auto v = U2 / rho;
    const auto w = U3 / rho;
    const auto ke = 0.5 * rho * (u * u + v * v + w * w);
    const auto p = tmax((P.gamma - 1.0) * (U4 - ke), P.p_floor);
    return b[0] * der(rho) + b[1] * der(u) + b[2] * der(v) + b[3] * der(w) + b[4] * der(p);
}
// the free stream's parts of a 256-entity block, 10 values: rows x of n entities, their sums to out, in block_sum's order
// (sh: 2560 doubles)
__device__ __forceinline__ void free_stream_block(const double *x, int32_t n, double *out, double *sh)
{
    const int32_t t = threadIdx.x;
    for (int j = 0; j < 10; ++j) sh[256 * j + t] = t < n ? x[10 * size_t(t) + j] : 0.0;
    __syncthreads();
    for (int k = 7; k >= 0; --k)
    {
        for (int32_t i = t; i < 10 << k; i += kAdjThreads)
        {
            double *v = sh + 256 * (i >> k) + (i & ((1 << k) - 1));
            v[0] += v[1 << k];
        }
        __syncthreads();
    }
    if (t < 10) out[t] = sh[256 * t];
}
} // namespace

// What is left of a cell: the parts its stencil neighbours, faces and edges hold for it, the current
// (Current.cpp:9-31), its CFL step if it set the step, u+ (Solver.cpp:110-118), the primitive recovery and the field
// reconstruction, transposed: Ub +=, Baddb +=, sPhi.  The entries' rows are loaded by the cell's two threads in turn and
// summed by both in entry order.  The first n_fs blocks sum the free stream's parts of a block of faces or cells each.
template <int DEG>
__global__ void __launch_bounds__(kAdjThreads, DEG == 4 ? 3 : 2) k_adj_cells(DevMesh d, Params P, StepFields F, AdjFields G, SpC Us, SpW Ub, int32_t with_dt,
                                                           int32_t n_fs)
{
    constexpr int N = DEG > 0 ? DEG / 2 : 1;
    __shared__ double sh[10 * kAdjThreads];
    const int32_t b = blockIdx.x, t = threadIdx.x, s = t & 1;
    if (b < G.n_f) return free_stream_block(G.fsf + 2560 * size_t(b), d.nf - 256 * G.block_face[b], G.f_part + 10 * size_t(b), sh);
    if (b < n_fs)
    {
        const int32_t i = b - G.n_f;
        return free_stream_block(G.fsc + 2560 * size_t(i), d.nc - 256 * G.block_cell[i], G.g_part + 10 * size_t(i), sh);
    }
    const int32_t c = (near_block(d, b, n_fs, int32_t(gridDim.x) - n_fs) * kAdjThreads + t) >> 1;
    if (c >= d.nc) return; // both threads of a cell
    int32_t k0, nk;
    row_of<DEG>(d, c, k0, nk);
    if constexpr (DEG > 0) nk = DEG;
    double M[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, A[N], w[5], e[9] = {};
    V3 n[N], cur;
    const V3 jc = L3(G.Jv, c);
    // x of the even entry, then (both) of the odd one
    auto pair = [&](double x, bool both, double &acc) {
        const double y = swap_pair(x);
        acc += s ? y : x;
        if (both) acc += s ? x : y;
    };
    // the entries i and i + 1 of the row: this thread's is i + s
    auto entries = [&](int i, double &a, V3 &m) {
        const bool both = i + 1 < nk, mine = i + s < nk;
        double x[9] = {};
        V3 j;
        a = 0.0;
        m = V3();
        if (mine)
        {
            const int32_t k = k0 + i + s, v = d.c2f[k], o = d.c2n[k];
            m = geo_normal(d, pid(v), a);
            const double *q = G.sE + 9 * size_t(k);
            for (int r = 0; r < 9; ++r) x[r] = q[r];
            const V3 area = psg(v) * L3(d.farea, pid(v));
            j = cross(jc, area);
            if (o >= 0) j = 0.5 * j + 0.5 * cross(L3(G.Jv, o), -1.0 * area);
        }
        for (int r = 0; r < 9; ++r) pair(x[r], both, e[r]);
        pair(j.x, both, cur.x); pair(j.y, both, cur.y); pair(j.z, both, cur.z);
        const V3 p(swap_pair(m.x), swap_pair(m.y), swap_pair(m.z));
        const double q = swap_pair(a);
        normal_add(M, s ? q : a, s ? p : m);
        normal_add(M, s ? a : q, s ? m : p);
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
        for (int i = 0; i < N; ++i) entries(2 * i, A[i], n[i]);
    }
    else
    {
        for (int32_t k = k0; k < k0 + nk; ++k)
            if (G.opp[k] >= 0)
                for (int m = 0; m < 5; ++m) w[m] += F.FS[10 * size_t(G.opp[k]) + 5 * s + m];
        for (int32_t i = 0; i < nk; i += 2) entries(i, A[0], n[0]);
    }
    V3 up;
    for (int32_t i = G.cec_ptr[c], end = G.cec_ptr[c + 1]; i < end; i += 2)
    {
        const bool both = i + 1 < end;
        V3 x;
        if (i + s < end) x = L3(G.eC, G.cec[i + s]);
        pair(x.x, both, up.x); pair(x.y, both, up.y); pair(x.z, both, up.z);
    }
    up += V3(e[0], e[1], e[2]);
    V3 bt = L3(G.Btb, c) + V3(e[3], e[4], e[5]);
    const V3 bi = V3(e[6], e[7], e[8]) + cur;
    if (with_dt && G.dt_cell[0] == c && G.dtb[0] != 0.0)
    {
        const double x = G.dtb[0];
        for (int m = 0; m < 5; ++m) w[m] += x * G.dtb[1 + 5 * s + m];
        bt += x * V3(G.dtb[11], G.dtb[12], G.dtb[13]);
    }
    const double *row = F.rec + 16 * size_t(c), *W = row + 5 * s;
    if (d.mat[c] == 0 && (up.x != 0.0 || up.y != 0.0 || up.z != 0.0))
    {
        // u+ = sum chi_s u_s, chi_s = n_s / n_e
        const double n0 = ion_density(P, 0, row[0]), n1 = ion_density(P, 1, row[5]), ne = n0 + n1;
        double chi = s == 0 ? 1.0 : 0.0;
        if (ne > 1e-300)
        {
            const double x0 = n0 / ne, x1 = n1 / ne, nd = W[0] < 0.0 ? 0.0 : 1.0 / P.M_s[s] * P.M_ref;
            const double d0 = ((s == 0 ? nd : 0.0) - x0 * nd) / ne, d1 = ((s == 1 ? nd : 0.0) - x1 * nd) / ne;
            w[0] += up.x * (d0 * row[1] + d1 * row[6]) + up.y * (d0 * row[2] + d1 * row[7]) + up.z * (d0 * row[3] + d1 * row[8]);
            chi = s == 0 ? x0 : x1;
        }
        w[1] += up.x * chi; w[2] += up.y * chi; w[3] += up.z * chi;
    }
    {
        const double *U = Us.p[s] + 5 * size_t(c);
        double *o = Ub.p[s] + 5 * size_t(c);
        o[0] += prim_column<0>(P, U, w);
        o[1] += prim_column<1>(P, U, w);
        o[2] += prim_column<2>(P, U, w);
        o[3] += prim_column<3>(P, U, w);
        o[4] += prim_column<4>(P, U, w);
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
    double M[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, A;
    for (int32_t k = d.c2f_ptr[c]; k < d.c2f_ptr[c + 1]; ++k)
    {
        const V3 m = geo_normal(d, pid(d.c2f[k]), A);
        normal_add(M, A, m);
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

// The last step's free-stream sums, and the flag of a time step whose cell was not found
__global__ void __launch_bounds__(kAdjThreads) k_adj_sums(AdjFields G, int32_t second_order)
{
    __shared__ double sh[kSumStage];
    free_stream_sums(G, second_order, sh);
    if (threadIdx.x == 0) G.sums[13] = G.dt_cell[1];
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
// the 256-entity blocks with an inflow face, a cell whose stencil has one, an edge of the imposed EMF; the cells with a wall
// in their stencil, numbered (the wall list's order does not matter: each cell's values are its own)
__global__ void __launch_bounds__(256) k_adj_inflow(DevMesh d, int32_t *face, int32_t *cell, int32_t *edge, int32_t *wall_slot, int32_t *wall_cell,
                                                    int32_t *n_wall)
{
    const int32_t i = gid();
    if (i < d.nf && d.kind[i] == kInflow) face[i >> 8] = 1;
    if (i < d.ne && d.emode[i] == 2) edge[i >> 8] = 1;
    if (i >= d.nc) return;
    bool wall = false;
    for (int32_t k = d.c2f_ptr[i]; k < d.c2f_ptr[i + 1]; ++k)
        if (d.snb[k] < 0 && d.snb[k] != kNoStencil)
        {
            const int8_t kind = d.kind[-(d.snb[k] + 1)];
            if (kind == kInflow) cell[i >> 8] = 1;
            wall |= kind == kWall;
        }
    wall_slot[i] = wall ? atomicAdd(n_wall, 1) : -1;
    if (wall) wall_cell[wall_slot[i]] = i;
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
        g.dt_f = D(size_t(blocks(nf, 256))); g.dt_c = D(C); g.dt_cp = D(size_t(blocks(nc, 256)));
        g.dtb = D(14); g.dt_cell = I(2); g.sums = D(14);
        // the 256-entity blocks at the inflow, numbered in their order
        const size_t nb[3] = {size_t(blocks(nf, 256)), size_t(blocks(nc, 256)), size_t(blocks(ne, 256))};
        const size_t n_flag = nb[0] + nb[1] + nb[2];
        int32_t *flag = I(n_flag + 1), *wall_slot = I(C), *wall_cell = I(C);
        std::vector<int32_t> h(n_flag + 1);
        chk(hipMemsetAsync(flag, 0, 4 * h.size(), stream), "memset");
        hipLaunchKernelGGL(k_adj_inflow, dim3(blocks(std::max({nc, nf, ne}), 256)), b256, 0, stream, d, flag, flag + nb[0], flag + nb[0] + nb[1],
                           wall_slot, wall_cell, flag + n_flag);
        check_launch("vjp inflow");
        d2h(h.data(), flag, 4 * h.size());
        g.wall_slot = wall_slot; g.wall_cell = wall_cell; g.n_wall = h[n_flag];
        g.mirror = D(3 * size_t(g.n_wall));
        std::vector<int32_t> block[3];
        for (size_t k = 0, i = 0; k < 3; ++k)
            for (size_t b = 0; b < nb[k]; ++b, ++i)
            {
                const bool on = h[i] != 0;
                h[i] = on ? int32_t(block[k].size()) : -1;
                if (on) block[k].push_back(int32_t(b));
            }
        chk(hipMemcpyAsync(flag, h.data(), 4 * h.size(), hipMemcpyHostToDevice, stream), "H2D");
        int32_t *list[2];
        for (int k = 0; k < 2; ++k)
        {
            list[k] = I(block[k].size());
            if (!block[k].empty()) chk(hipMemcpyAsync(list[k], block[k].data(), 4 * block[k].size(), hipMemcpyHostToDevice, stream), "H2D");
        }
        chk(hipStreamSynchronize(stream), "sync");
        g.fs_face = flag; g.fs_cell = flag + nb[0]; g.inflow_edge = flag + nb[0] + nb[1];
        g.block_face = list[0]; g.block_cell = list[1];
        g.n_f = int32_t(block[0].size()); g.n_c = int32_t(block[1].size()); g.n_e = int32_t(block[2].size());
        g.fsf = D(2560 * size_t(g.n_f)); g.fsc = D(2560 * size_t(g.n_c));
        g.f_part = D(10 * size_t(g.n_f)); g.g_part = D(10 * size_t(g.n_c)); g.e_part = D(3 * size_t(g.n_e));
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
              n_flux = blocks(nf, kAdjThreads / 2), n_grad = blocks(nc, kGradThreads / 2);
    const AdjFields &g = aw.g;
    const int n_fs = g.n_f + (P.second_order ? g.n_c : 0);
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
    chk(hipMemsetAsync(g.sums, 0, 8 * 14, stream), "memset");
    chk(hipMemsetAsync(g.dt_cell, 0, 8, stream), "memset");
    LAUNCH("adj_energy", k_adj_energy, dim3(nbc), dim3(kAdjThreads), 0, stream, d, static_cast<const double *>(aw.x.Phi),
           static_cast<const double *>(Badd), r0, r1, g);
    LAUNCH("adj_flux", k_adj_flux, dim3(nbf), dim3(kAdjThreads), 0, stream, d, aw.x.F.fent, g, 1);
    SpC Us{};
    SpW Ub{};
    for (int s = 0; s < 2; ++s) Ub.p[s] = aw.Ub[s];
    const size_t lds = std::max(sizeof(double) * kSumStage, n_heavy ? (kHeavyRows * sizeof(double) + sizeof(int32_t)) * size_t(max_valence) : 0);
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
            const int n_sum = n < n_steps - 1 ? 1 : 0;
            LAUNCH("adj_update", k_adj_update<DEG>, dim3(n_heavy + n_dt + n_sum + n_edge + nbf + n_cell), dim3(kAdjThreads), lds, stream, d, P,
                   aw.x.F, g, Us, Ub, static_cast<const double *>(aw.x.E), dt, static_cast<const int32_t *>(heavy), n_heavy, max_valence, n_dt,
                   static_cast<const double *>(aw.x.dt_part), nbc, n_sum, n_edge, nbf);
            LAUNCH("adj_faces", k_adj_faces, dim3(1 + nbc + nbf + n_flux), dim3(kAdjThreads), 0, stream, d, P, aw.x.F, g,
                   static_cast<const double *>(aw.x.Phi), static_cast<const double *>(PhiAdd), nbc, nbf);
            if (P.second_order && g.n_wall)
                LAUNCH("adj_mirror", k_adj_mirror<DEG>, dim3(blocks(3 * int64_t(g.n_wall), 64)), dim3(64), 0, stream, d, P, aw.x.F, g);
            LAUNCH("adj_gradients", k_adj_gradients<DEG>, dim3(1 + n_grad), dim3(kGradThreads), 0, stream, d, P, aw.x.F, g, n_grad);
            LAUNCH("adj_cells", k_adj_cells<DEG>, dim3(n_fs + n_cell), dim3(kAdjThreads), 0, stream, d, P, aw.x.F, g, Us, Ub, n_dt, n_fs);
        });
        LAUNCH("adj_flux", k_adj_flux, dim3(nbf), dim3(kAdjThreads), 0, stream, d, aw.x.F.fent, g, 0);
        check_launch("vjp reverse step");
        // written while the step's fields were formed, long before what was launched since ends
        if (again && wait_box(dt_box)[0] != dt) throw std::runtime_error("vjp: recomputed time step differs from the forward sweep");
    }
    if (n_steps > 0) LAUNCH("adj_sums", k_adj_sums, dim3(1), dim3(kAdjThreads), 0, stream, g, P.second_order);
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
