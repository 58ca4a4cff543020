// FP64 GMRES with the mixed-precision solve's orthogonalisation (precision 3): the reference system and iteration
// (ImplicitInduction::solve, Common/induction/ImplicitInduction.cpp:299-390: Jacobi, warm start, restarts, true
// residual per restart) with classical Gram-Schmidt in place of modified Gram-Schmidt: one multi-dot pass and one
// multi-axpy pass per Arnoldi step (DGKS re-projection when the first removed more than 1 - kDgks64 of the norm),
// all in FP64.  It is the FP64 counterpart of the mixed inner solve, so that the mixed path's gain over the reference
// iteration can be split into its precision part and its orthogonalisation part.
#include <algorithm>
#include <cmath>
#include <stdexcept>

#include "ctx.h"

using namespace mhdg;

namespace
{
constexpr double kDgks64 = 0.1; // as the mixed solve
inline int nbk(int64_t n) { return static_cast<int>((n + 255) / 256); }
} // namespace

#define LAUNCH(NAME, ...)                                                                                                    \
    do                                                                                                                       \
    {                                                                                                                        \
        prof_begin(NAME);                                                                                                    \
        hipLaunchKernelGGL(__VA_ARGS__);                                                                                     \
        prof_end();                                                                                                          \
    } while (0)

int mhdg_ctx::solve64_cgs(const double *Phi_n, const double *Eex, const int8_t *dir, double dt, double *Eout, double *rel_res)
{
    const int m = restart;
    const int max_it = cfg.ind_max_it;
    const double rtol = rtol_override > 0 ? rtol_override : cfg.ind_rtol;
    freeze(nullptr);
    LAUNCH("solve_init", k_solve_init, dim3(nbk(ne)), dim3(256), 0, stream, Eex, have_corr ? corr : nullptr, dir, d.m_e, d.d2, dt,
           dte_cur, ne, x0, invdiag, static_cast<float *>(nullptr), delta);
    rhs_residual(Phi_n, Eex, x0, dir, dt); // b = E_expl + F(Phi^n), r = b - A x0
    const double *nn = norms(rvec, bvec);
    const double bnorm = std::sqrt(std::max(nn[1], 1e-300));
    double beta = std::sqrt(nn[0]);
    int total = 0;
    Hessenberg hs(m);
    while (beta > rtol * bnorm && total < max_it)
    {
        LAUNCH("scale", k_div_scalar, dim3(nbk(ne)), dim3(256), 0, stream, rvec, scal, ne, V[0]);
        hs.start(beta);
        int j = 0;
        for (; j < m && total < max_it; ++j, ++total)
        {
            apply_op(nullptr, V[j], invdiag, dir, dt, 1, 1, nullptr, wvec);
            double hn;
            const double *h = arnoldi_cgs(ortho64(j), kDgks64, hn);
            const double est = hs.add(j, h, 0.0, hn);
            if (est <= rtol * bnorm || !(hn > 1e-300)) { ++j; ++total; break; }
        }
        prof_begin("gmres_update");
        solution_update<double>(Vptrs, hs.solve(j), j, invdiag, dir, ne, x0, delta, tmp, stream);
        prof_end();
        apply_op(nullptr, tmp, nullptr, dir, dt, 1, 0, bvec, rvec);
        beta = std::sqrt(norms(rvec, nullptr)[0]);
    }
    LAUNCH("solve_final", k_solve_final, dim3(nbk(ne)), dim3(256), 0, stream, x0, delta, Eex, dir, ne, Eout, corr);
    check_launch("solve final");
    have_corr = true;
    if (rel_res) *rel_res = beta / bnorm;
    return total;
}
