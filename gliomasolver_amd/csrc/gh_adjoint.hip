// gh_adjoint.hip -- discrete adjoint of the reaction-diffusion solve and the
// gradient of J = -logL w.r.t. (Dw, rho, T, x0, y0, z0).
//
// No reference counterpart (the reference has no derivatives).  Differentiable
// model: N fused steps u_{k+1} = F(u_k) = clamp(u_k + dt R(u_k)) of the
// operator of Glioma/Operators/ReactionDiffusionOperator.h with dt = T/N, where
//   R_c = ih2 sum_i d'_i (u_{n_i} - u_c) + rho u_c (1 - u_c)   (in the domain)
//   d'_i = Dbar_i (1 + o(opposite neighbour of face i))        (no-flux rule)
//   o(x) = [u_x < tau_x]                                       (chf < 0.1)
// The flags o, the in-domain test and the upper clamp are frozen along the
// trajectory (a.e. derivative); the lower clamp is taken as inactive.
// Dbar is homogeneous of degree 1 in (Dw, Dg = Dw/10), so dDbar/dDw = Dbar/Dw.
//
// Reverse sweep, per step, per cell c (lambda in FP64):
//   lambda_k[c] = m_c l_c (dom_c ? 1 + dt(-ih2 sum_i d'_i + rho(1 - 2u_c)) : 1)
//               + dt ih2 sum_i w_{n_i} Dbar_i (1 + o(c + 2 dir_i))
//   with w_e = m_e dom_e lambda_{k+1}[e], m_e = [u_{k+1,e} < 1]
// (the face of neighbour e towards c is doubled when e's opposite neighbour,
// c + 2 dir_i, is outside).  Parameter gradients accumulate per cell
//   dJ/dDw += w_c dt Rdiff_c / Dw, dJ/drho += w_c dt u_c(1-u_c), dJ/dT += w_c R_c / N
// with R_c = Rdiff_c + rho u_c (1 - u_c): all three are linear in the sums
// A = sum w_c Rdiff_c and B = sum w_c u_c (1 - u_c), which are accumulated in
// FP64 per wave (dt, rho, N and Dw are constant over the solve and applied
// once at the end); every wave owns the same cells in every step, so the
// accumulation order is fixed.  The states that fit the tape
// (TapeBuf) stay on it from the forward sweep, which writes them there; the
// steps before them are cut into segments of the tape's length, recomputed from
// checkpoints taken in the forward sweep.  With every segment recomputed, 343
// steps of 64^3 FP64 took 3.3 ms (2.7 with none), 1,000 of 128^3 FP32 12.8 (11.0).
#include <cmath>
#include <vector>

#include "gh_ctx.h"
#include "gh_adjoint_common.h"

namespace gh {
namespace {

__global__ __launch_bounds__(512) void adj_reduce_kernel(const double* __restrict__ part, size_t n,
                                                         const double* __restrict__ ic, double* __restrict__ out) {
    adj_reduce_body(part, n, ic, out);
}

template <typename Real>
int adjoint_t(Ctx& c, int64_t N, double T, int K, const double* lik, int stepPET, int stepTi, int use_roi,
              const double* ic, double sigma, double* loss, double* grad) {
    const size_t nc = c.ncells();
    const size_t nb = nc * sizeof(Real);
    const int ns = c.topo.nblocks();
    int rc;
    if ((rc = c.adjLam[0].ensure(nc * 8)) || (rc = c.adjLam[1].ensure(nc * 8)) ||
        (rc = c.adjPart.ensure(sizeof(double) * ADJ_PART * ns)))
        return rc;
    if ((rc = c.adjSeg.ensure(c.device, ((size_t)std::min<int64_t>(K, N) + 1) * nb, ((size_t)N + 1) * nb))) return rc;
    // segments of `len` steps, the first one shorter; the last stays on the tape
    const int64_t len = std::min<int64_t>(N, (int64_t)(c.adjSeg.buf.bytes / nb) - 1);
    const int64_t nseg = (N + len - 1) / len;
    if ((rc = c.adjCk.ensure(std::max<size_t>(1, (size_t)(nseg - 1)) * nb))) return rc;
    auto start = [&](int64_t i) { return i == 0 ? (int64_t)0 : N - (nseg - i) * len; };
    const double dt = T / (double)N;
    char* ck = (char*)c.adjCk.p;
    char* seg = (char*)c.adjSeg.buf.p;
    // two steps per launch from a clamped state (k >= 1) within a segment
    const bool pairs = c.fast_ok && c.topo.uniform_bpd > 0;
    // the two-step schedule (tile 0) leaves out the groups of blocks without
    // diffusion that u_1 leaves at zero, in both directions
    const bool skip = pairs && c.rd_bpw == 0 && c.nGrp > 0;
    // u_{k+1} (and u_{k+2}: returns 2) from u_k in `in`
    auto launch = [&](int64_t k, int64_t end, const void* in, void* one, void* mid, void* two, int* steps) -> int {
        *steps = pairs && k >= 1 && k + 2 <= end ? 2 : 1;
        if (*steps == 2) return rd_step2_buffers(c, in, two, mid, dt, skip);
        return pairs && k >= 1 ? rd_step1_buffers(c, in, one, dt, skip) : rd_step_buffers(c, in, one, dt);
    };
    // u_{k0+1} .. u_end on the tape, u_k0 at its start; u_N goes to last (if not null)
    auto run_on_tape = [&](int64_t k0, int64_t end, void* last) -> int {
        for (int64_t k = k0; k < end;) {
            char* in = seg + (size_t)(k - k0) * nb;
            auto at = [&](int64_t s) { return s == N && last ? (char*)last : seg + (size_t)(s - k0) * nb; };
            if (k == 1 && k0 == 0 && last && skip) {  // (the first sweep: the marks are not known yet)
                if ((rc = rd_mark_still(c, in, last)) || (rc = rd_zero_still(c, seg + 2 * nb, len - 1))) return rc;
            }
            int steps;
            if ((rc = launch(k, end, in, at(k + 1), at(k + 1), at(k + 2), &steps))) return rc;
            k += steps;
        }
        return GH_OK;
    };
    // forward sweep
    for (int64_t i = 0; i + 1 < nseg; ++i) {
        const int64_t end = start(i + 1);
        GH_HIP_CHECK(hipMemcpyAsync(ck + (size_t)i * nb, c.phi[c.cur].p, nb, hipMemcpyDeviceToDevice, c.stream));
        for (int64_t k = start(i); k < end;) {
            if (k == 1 && skip && ((rc = rd_mark_still(c, c.phi[c.cur].p, c.phi[1 - c.cur].p)) ||
                                   (rc = rd_zero_still(c, seg, len + 1))))
                return rc;
            void* out = c.phi[1 - c.cur].p;
            int steps;
            if ((rc = launch(k, end, c.phi[c.cur].p, out, nullptr, out, &steps))) return rc;
            k += steps;
            c.cur = 1 - c.cur;
        }
    }
    const int64_t tape0 = start(nseg - 1);
    if (tape0 == 1 && skip && ((rc = rd_mark_still(c, c.phi[c.cur].p, c.phi[1 - c.cur].p)) ||
                               (rc = rd_zero_still(c, seg, len + 1))))
        return rc;
    GH_HIP_CHECK(hipMemcpyAsync(seg, c.phi[c.cur].p, nb, hipMemcpyDeviceToDevice, c.stream));
    if ((rc = run_on_tape(tape0, N, c.phi[1 - c.cur].p))) return rc;
    c.cur = 1 - c.cur;
    // loss at u_N and its gradient as the terminal adjoint
    int64_t npet = 0;
    if ((rc = lik_eval_current(c, lik, stepPET, stepTi, use_roi, loss, &npet))) return rc;
    int lc = 0;
    if ((rc = lik_seed_gradient(c, c.phi[c.cur].p, c.adjLam[lc].as<double>(), lik, stepPET, stepTi, use_roi)))
        return rc;
    hipLaunchKernelGGL(adj_mask_kernel<Real>, dim3((unsigned)((nc + 255) / 256)), dim3(256), 0, c.stream, nc,
                       c.adjLam[lc].as<double>(), (const Real*)c.phi[c.cur].p);
    GH_HIP_CHECK(hipGetLastError());
    const bool still = skip && N > 1;  // (marked before step 1)
    if (still)  // the launches leave out the seed in the still groups: it stands in both adjoint buffers
        GH_HIP_CHECK(hipMemcpyAsync(c.adjLam[1 - lc].p, c.adjLam[lc].p, nc * 8, hipMemcpyDeviceToDevice, c.stream));
    // reverse sweep
    GH_HIP_CHECK(hipMemsetAsync(c.adjPart.p, 0, sizeof(double) * ADJ_PART * ns, c.stream));
    const double h = block_h_of(c);
    const double ih2 = 1. / (h * h);
    const UniformAdjParams prm{c.rho, ih2, dt, c.topo.uniform_bpd, bpd_magic(c.topo.uniform_bpd)};
    // blocks without diffusion take the reverse step's short path under the
    // two-step schedule (tile 0); step 0 reads the caller's state and leaves
    // nothing out
    const StepWork all = c.rd_bpw == 0 ? rd_step_work(c, false) : step_work(ns, nullptr, 0, nullptr, nullptr);
    const StepWork moving = still ? rd_step_work(c, true) : all;
    for (int64_t i = nseg - 1; i >= 0; --i) {
        const int64_t k0 = start(i), k1 = i + 1 < nseg ? start(i + 1) : N;
        if (i + 1 < nseg) {
            GH_HIP_CHECK(hipMemcpyAsync(seg, ck + (size_t)i * nb, nb, hipMemcpyDeviceToDevice, c.stream));
            if ((rc = run_on_tape(k0, k1 - 1, nullptr))) return rc;
        }
        for (int64_t k = k1 - 1; k >= k0; --k) {
            const Real* uk = (const Real*)(seg + (size_t)(k - k0) * nb);
            const int mask_out = k >= 1;
            const StepWork& wk = k >= 1 ? moving : all;
            if (c.fast_ok && k >= 1)  // u_k is a clamped state: the clamped-state records
                launch_adj_step<true, Real>(c.stream, wk, uk, mask_out, c.adjLam[lc].as<double>(),
                                            c.adjLam[1 - lc].as<double>(), c.statF.as<Stat4<Real>>(),
                                            (const Real*)nullptr, prm, c.adjPart.as<double>());
            else
                launch_adj_step<false, Real>(c.stream, wk, uk, mask_out, c.adjLam[lc].as<double>(),
                                             c.adjLam[1 - lc].as<double>(), c.statD.as<Stat4<Real>>(),
                                             c.statSig.as<Real>(), prm, c.adjPart.as<double>());
            GH_HIP_CHECK(hipGetLastError());
            lc = 1 - lc;
        }
    }
    // initial-condition gradient from lambda_0 and u_0
    if ((rc = c.likPart.ensure(sizeof(double) * 4 * 1025)) || (rc = c.pinLik.ensure_grow(ADJ_SUMS * sizeof(double))))
        return rc;
    hipLaunchKernelGGL(adj_ic_partials<Real>, dim3(ADJ_IC_GRID), dim3(256), 0, c.stream, nc, c.topo.uniform_bpd,
                       c.adjLam[lc].as<double>(), (const Real*)seg, ic[0], ic[1], ic[2], 1.0 / (sigma * sigma),
                       c.likPart.as<double>());
    GH_HIP_CHECK(hipGetLastError());
    double* const sums = c.pinLik.as<double>();
    hipLaunchKernelGGL(adj_reduce_kernel, dim3(1), dim3(512), 0, c.stream, c.adjPart.as<double>(), (size_t)ns,
                       c.likPart.as<double>(), sums);
    GH_HIP_CHECK(hipGetLastError());
    GH_HIP_CHECK(hipStreamSynchronize(c.stream));
    adj_param_grads(sums, dt, 1.0 / c.Dw, 1.0 / (double)N, c.rho, grad);
    for (int q = 0; q < 3; ++q) grad[3 + q] = sums[2 + q];
    return GH_OK;
}

}  // namespace
}  // namespace gh

using namespace gh;

extern "C" int gh_rd_adjoint(gh_ctx* ctx, int64_t nsteps, double T, int ckpt_every, const double* lik_params,
                             int stepPET, int stepTi, int use_roi, const double* ic_center, double ic_sigma,
                             double* loss, double* grad) {
    Ctx* c = as_ctx(ctx);
    if (!c || !lik_params || !ic_center || !loss || !grad) return set_error(GH_EINVAL, "null argument");
    if (!c->prepared) return set_error(GH_ESTATE, "gh_rd_adjoint: call gh_rd_prepare first");
    if (!c->lik_valid())
        return set_error(GH_ESTATE, "gh_rd_adjoint: no observations for the current grid (call gh_lik_set_data)");
    if (c->topo.uniform_bpd <= 0) return set_error(GH_ESTATE, "gh_rd_adjoint: needs a uniform grid");
    if (nsteps < 1 || ckpt_every < 1 || ckpt_every > 4096 || !(T > 0) || !(ic_sigma > 0) || !(c->Dw > 0))
        return set_error(GH_EINVAL, "gh_rd_adjoint: bad argument");
    GH_HIP_CHECK(hipSetDevice(c->device));
    if (int rc = rd_ensure_prepared(*c)) return rc;
    return c->real_kind == GH_REAL_F32
               ? adjoint_t<float>(*c, nsteps, T, ckpt_every, lik_params, stepPET, stepTi, use_roi, ic_center,
                                  ic_sigma, loss, grad)
               : adjoint_t<double>(*c, nsteps, T, ckpt_every, lik_params, stepPET, stepTi, use_roi, ic_center,
                                   ic_sigma, loss, grad);
}

extern "C" int gh_adjoint_release(gh_ctx* ctx) {
    Ctx* c = as_ctx(ctx);
    if (!c) return set_error(GH_EINVAL, "null context");
    GH_HIP_CHECK(hipSetDevice(c->device));
    GH_HIP_CHECK(hipStreamSynchronize(c->stream));
    c->adjSeg.release();
    c->adjCk.release();
    return GH_OK;
}
