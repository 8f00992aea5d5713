// gh_rd.hip -- reaction-diffusion kernels for gfx950.
//
// Reference: Glioma/Operators/ReactionDiffusionOperator.h (rhs :98-139,
// harmonic mean :148-163, no-flux BC :166-181, UpdateTumor :215-222) driven by
// Glioma/Glioma_ReactionDiffusion.cpp:176-187.
//
// Arithmetic is bit-faithful to the reference for Real = float and double:
// the same float/double promotion points, no FMA contraction (this file is
// compiled with -ffp-contract=off and the pragma below), IEEE double division
// for the harmonic mean.
//
// Split of the work:
//   constants_kernel   once per solve (Dw, Dg, anatomy fixed): the harmonic
//                      face diffusivity of each cell's +x,+y,+z face (the
//                      harmonic mean is symmetric, so each face is computed
//                      once), the threshold tau with "chf = phi+p_w+p_g < 0.1
//                      <=> phi < tau", and sigma with "p_w+p_g+phi > 0 <=>
//                      phi > sigma".  Both predicates are monotone in phi, so
//                      tau is found exactly by bisection over the ordered bit
//                      patterns of Real.
//   rd_step_kernel     every step: one workgroup per 8^3 block stages the
//                      block plus its six face halos (phi, outside flag, minus-
//                      face diffusivity) in LDS and evaluates the stencil, then
//                      either stores dphidt (two-pass API) or applies the
//                      Euler update and clamp in registers (fused step).
#include <cfloat>
#include <cmath>

#include "gh_ctx.h"
#include "gh_rd_common.h"

#pragma clang fp contract(off)

namespace gh {
namespace {

// phi += dt * dphidt, clamped: 12 B a cell, 16 B of each field a lane.  nc is a
// multiple of 512.  Each XCD takes a contiguous part, the one whose dphidt it has
// written and whose phi it reads next (rd_step_kernel), in its L2: 128^3 FP32
// 5.8 -> 5.3 us (dealt out evenly 6.4), and dphidt itself 10.4 -> 9.3 us.
template <typename Real>
struct alignas(16) Cells {
    Real v[16 / sizeof(Real)];
};
template <typename Real>
__global__ __launch_bounds__(256) void rd_update_kernel(size_t nc, unsigned per_xcd, Cells<Real>* __restrict__ phi,
                                                        const Cells<Real>* __restrict__ dphidt, double dt) {
    constexpr int N = 16 / sizeof(Real);
    const size_t i = (size_t)(blockIdx.x % 8 * per_xcd + blockIdx.x / 8) * 256 + threadIdx.x;
    if (i * N >= nc) return;
    Cells<Real> p = phi[i];
    const Cells<Real> d = dphidt[i];
#pragma unroll
    for (int k = 0; k < N; ++k) p.v[k] = rd_update(p.v[k], d.v[k], dt);
    phi[i] = p;
}

constexpr int64_t kStillMinSteps = 9;  // shortest call that marks the still groups

inline double block_h(const Ctx& c) {
    // info.h[0] = 2^-level / 8 as Real (MRAGrid.inl:200-206); exact in float
    return std::ldexp(1.0, -c.topo.blocks[0].level) / BS;
}

// The per-solve constants (constants_kernel) and, from its flags, the work list
// of the two-step and reverse-step kernels (StepWork).
template <typename Real>
int prepare_t(Ctx& c, double Dw, double Dg, double rho) {
    const int ns = c.topo.nblocks();
    const size_t nc = c.ncells();
    int rc;
    if ((rc = c.statF.ensure_grow(std::max<size_t>(1, nc) * sizeof(Stat4<Real>))) ||
        (rc = c.zeroFlux.ensure_grow((size_t)ns + 3)) || (rc = clear_stat_flags(c.stream, c.flag)))
        return rc;
    const int bpd = c.topo.uniform_bpd;
    const UniformAnatomy<Real> src{c.pw.as<Real>(), c.pg.as<Real>(), (Real)Dw, (Real)Dg, bpd, bpd_magic(bpd)};
    hipLaunchKernelGGL((constants_kernel<Real, UniformAnatomy<Real>>), dim3(ns), dim3(512), 0, c.stream, src,
                       c.statD.as<Stat4<Real>>(), c.statSig.as<Real>(), c.statF.as<Stat4<Real>>(),
                       c.zeroFlux.as<unsigned char>(), c.flag.as<unsigned int>());
    GH_HIP_CHECK(hipGetLastError());
    std::vector<unsigned char> z(ns);
    unsigned int flags[2] = {1, 1};
    GH_HIP_CHECK(hipMemcpyAsync(flags, c.flag.p, sizeof(flags), hipMemcpyDeviceToHost, c.stream));
    GH_HIP_CHECK(hipMemcpyAsync(z.data(), c.zeroFlux.p, ns, hipMemcpyDeviceToHost, c.stream));
    GH_HIP_CHECK(hipStreamSynchronize(c.stream));
    c.fast_ok = flags[0] == 0;
    c.plain_dom = flags[1] == 0;
    c.nZeroFlux = 0;
    c.nFull = ns;
    c.nGrp = 0;
    std::vector<int32_t> full;
    std::vector<int2> grp;
    if (c.fast_ok) build_step_work(z.data(), {(size_t)ns}, full, grp, nullptr, nullptr);
    for (const int2& g : grp) c.nZeroFlux += g.y;
    if (!grp.empty()) {  // (without: item i is slot i)
        if ((rc = c.fullList.ensure_grow(std::max<size_t>(1, full.size()) * sizeof(int32_t))) ||
            (rc = c.grpList.ensure_grow(grp.size() * sizeof(int2))) || (rc = c.stillGrp.ensure_grow(grp.size())))
            return rc;
        if (!full.empty())
            GH_HIP_CHECK(hipMemcpyAsync(c.fullList.p, full.data(), full.size() * sizeof(int32_t),
                                        hipMemcpyHostToDevice, c.stream));
        GH_HIP_CHECK(hipMemcpyAsync(c.grpList.p, grp.data(), grp.size() * sizeof(int2), hipMemcpyHostToDevice,
                                    c.stream));
        GH_HIP_CHECK(hipStreamSynchronize(c.stream));
        c.nFull = (int)full.size();
        c.nGrp = (int)grp.size();
    }
    c.Dw = Dw;
    c.Dg = Dg;
    c.rho = rho;
    c.prepared = true;
    c.constants_stale = false;
    return GH_OK;
}

// marks the still groups from the state in `in` (clamped: written by the fused
// update) and writes their zeros into `out`
template <typename Real>
int mark_still(Ctx& c, const Real* in, Real* out) {
    if (c.nGrp == 0) return GH_OK;
    hipLaunchKernelGGL(still_kernel<Real>, dim3(c.nGrp), dim3(256), 0, c.stream, c.nGrp, c.grpList.as<int2>(),
                       c.zeroFlux.as<unsigned char>(), in, out, c.stillGrp.as<unsigned char>());
    GH_HIP_CHECK(hipGetLastError());
    return GH_OK;
}

template <typename Real, bool FUSED, int BPW>
void launch_step(Ctx& c, const Real* in, Real* out, double dt) {
    const double h = block_h(c);
    const double ih2 = 1. / (h * h);
    const UniformStepParams<Real> prm{(Real)c.rho, ih2, dt, c.topo.uniform_bpd, bpd_magic(c.topo.uniform_bpd)};
    launch_step_kernel<Real, FUSED, BPW>(c.stream, c.topo.nblocks(), c.zeroFlux, in, out, c.statD.as<Stat4<Real>>(),
                                         c.statSig.as<Real>(), prm);
}

// two fused steps per launch (rd_step2_kernel), one block per workgroup
template <typename Real>
int launch_step2(Ctx& c, const Real* in, Real* out, double dt) {
    const int ns = c.topo.nblocks();
    const int per_xcd = (ns + 7) / 8;
    const double h = block_h(c);
    const double ih2 = 1. / (h * h);
    const UniformStepParams<Real> prm{(Real)c.rho, ih2, dt, c.topo.uniform_bpd, bpd_magic(c.topo.uniform_bpd)};
    hipLaunchKernelGGL((rd_step2_kernel<Real, UniformStepParams<Real>>), dim3(8 * per_xcd), dim3(512), 0, c.stream,
                       ns, per_xcd, in, out, c.statD.as<Stat4<Real>>(), c.statSig.as<Real>(), prm);
    GH_HIP_CHECK(hipGetLastError());
    return GH_OK;
}

// two fused steps (or one) per launch on a clamped state (rd_step2f_kernel);
// mid, when not null, receives the state after the first of two; skip_still:
// the still groups are marked and their zeros stand in out (and mid)
template <typename Real>
int launch_step2f(Ctx& c, const Real* in, Real* out, double dt, bool two, bool skip_still, Real* mid = nullptr) {
    const double h = block_h(c);
    const double ih2 = 1. / (h * h);
    const UniformStepParams<Real> prm{(Real)c.rho, ih2, dt, c.topo.uniform_bpd, bpd_magic(c.topo.uniform_bpd)};
    const StepWork wk = rd_step_work(c, skip_still);
    launch_step2f_kernel<Real>(c.stream, wk, c.plain_dom, two, in, out, mid, c.statF.as<Stat4<Real>>(), prm);
    GH_HIP_CHECK(hipGetLastError());
    return GH_OK;
}

template <typename Real, bool FUSED>
int step_t(Ctx& c, const Real* in, Real* out, double dt) {
    switch (c.rd_bpw) {
        case 1: launch_step<Real, FUSED, 1>(c, in, out, dt); break;
        case 4: launch_step<Real, FUSED, 4>(c, in, out, dt); break;
        default: launch_step<Real, FUSED, 2>(c, in, out, dt); break;
    }
    GH_HIP_CHECK(hipGetLastError());
    return GH_OK;
}

template <typename Real, bool FUSED>
int step_t(Ctx& c, Real* out) {
    return step_t<Real, FUSED>(c, c.phi[c.cur].as<Real>(), out, c.dt_last);
}

}  // namespace

int rd_ensure_prepared(Ctx& c) {
    if (!c.prepared || !c.constants_stale) return GH_OK;
    return rd_prepare(c, c.Dw, c.Dg, c.rho);
}

int rd_prepare(Ctx& c, double Dw, double Dg, double rho) {
    if (c.topo.uniform_bpd <= 0) {  // blocks on several levels: ghosts across level jumps
        int rc = rd_prepare_ghosted(c, Dw, Dg);
        if (rc) return rc;
        c.Dw = Dw;
        c.Dg = Dg;
        c.rho = rho;
        c.prepared = true;
        c.constants_stale = false;
        return GH_OK;
    }
    return c.real_kind == GH_REAL_F32 ? prepare_t<float>(c, Dw, Dg, rho) : prepare_t<double>(c, Dw, Dg, rho);
}

int rd_rhs(Ctx& c) {
    if (c.topo.uniform_bpd <= 0) return rd_step_ghosted(c, c.phi[c.cur].p, c.dphidt.p, 0.0, false);
    return c.real_kind == GH_REAL_F32 ? step_t<float, false>(c, c.dphidt.as<float>())
                                      : step_t<double, false>(c, c.dphidt.as<double>());
}

int rd_update(Ctx& c, double dt) {
    const size_t nc = c.ncells();
    const unsigned per_xcd = (unsigned)((nc * c.real_size / 16 + 2047) / 2048);
    const dim3 grid(8 * per_xcd);
    if (c.real_kind == GH_REAL_F32)
        hipLaunchKernelGGL(rd_update_kernel<float>, grid, dim3(256), 0, c.stream, nc, per_xcd,
                           c.phi[c.cur].as<Cells<float>>(),
                           c.dphidt.as<Cells<float>>(), dt);
    else
        hipLaunchKernelGGL(rd_update_kernel<double>, grid, dim3(256), 0, c.stream, nc, per_xcd,
                           c.phi[c.cur].as<Cells<double>>(), c.dphidt.as<Cells<double>>(), dt);
    GH_HIP_CHECK(hipGetLastError());
    return GH_OK;
}

// Times trial steps of each blocks-per-workgroup tile on the current state
// (saved in the dphidt scratch and restored after every trial) and keeps the
// fastest.
int rd_autotune(Ctx& c, double dt, int trial_steps, int* best_out) {
    static const int cand[4] = {1, 2, 4, 0};
    if (c.topo.uniform_bpd <= 0) {  // the multi-level kernel has a single tile
        if (best_out) *best_out = c.rd_bpw;
        return GH_OK;
    }
    const size_t nb = c.ncells() * c.real_size;
    GH_HIP_CHECK(hipMemcpyAsync(c.dphidt.p, c.phi[c.cur].p, nb, hipMemcpyDeviceToDevice, c.stream));
    const int cur0 = c.cur;
    float best_ms = 1e30f;
    int best = c.rd_bpw;
    for (int k = 0; k < 4; ++k) {
        c.rd_bpw = cand[k];
        int rc = rd_steps(c, cand[k] == 0 ? kStillMinSteps : 2, dt);  // warm: every kernel of the trial
        if (rc) return rc;
        GH_HIP_CHECK(hipEventRecord(c.ev0, c.stream));
        if ((rc = rd_steps(c, trial_steps, dt))) return rc;
        GH_HIP_CHECK(hipEventRecord(c.ev1, c.stream));
        GH_HIP_CHECK(hipEventSynchronize(c.ev1));
        float ms = 0;
        GH_HIP_CHECK(hipEventElapsedTime(&ms, c.ev0, c.ev1));
        if (ms < best_ms) { best_ms = ms; best = cand[k]; }
        c.cur = cur0;
        GH_HIP_CHECK(hipMemcpyAsync(c.phi[c.cur].p, c.dphidt.p, nb, hipMemcpyDeviceToDevice, c.stream));
    }
    c.rd_bpw = best;
    GH_HIP_CHECK(hipStreamSynchronize(c.stream));
    if (best_out) *best_out = best;
    return GH_OK;
}

double block_h_of(const Ctx& c) { return block_h(c); }

StepWork rd_step_work(const Ctx& c, bool skip_still) {
    if (c.nGrp == 0) return step_work(c.nFull, nullptr, 0, nullptr, nullptr);
    return step_work(c.nFull, c.fullList.as<int32_t>(), c.nGrp, c.grpList.as<int2>(),
                     skip_still ? c.stillGrp.as<unsigned char>() : nullptr);
}

int clear_stat_flags(hipStream_t stream, DevBuf& flag) {
    if (int rc = flag.ensure(2 * sizeof(unsigned int))) return rc;
    GH_HIP_CHECK(hipMemsetAsync(flag.p, 0, 2 * sizeof(unsigned int), stream));
    return GH_OK;
}

int rd_mark_still(Ctx& c, const void* in, void* out) {
    return c.real_kind == GH_REAL_F32 ? mark_still<float>(c, (const float*)in, (float*)out)
                                      : mark_still<double>(c, (const double*)in, (double*)out);
}

template <typename Real>
static int zero_still(Ctx& c, Real* states, int64_t n) {
    const int bpd = c.topo.uniform_bpd;
    const UniformStepParams<Real> prm{0, 0, 0, bpd, bpd_magic(bpd)};  // (its pos)
    launch_still_zero<Real>(c.stream, c.nGrp, c.grpList, c.stillGrp, c.zeroFlux, prm, states, c.ncells(), n);
    GH_HIP_CHECK(hipGetLastError());
    return GH_OK;
}
int rd_zero_still(Ctx& c, void* states, int64_t n) {
    if (c.nGrp == 0 || n <= 0) return GH_OK;
    return c.real_kind == GH_REAL_F32 ? zero_still(c, (float*)states, n) : zero_still(c, (double*)states, n);
}

static int step2f_buffers(Ctx& c, const void* in, void* out, void* mid, double dt, bool two, bool skip_still) {
    if (!c.fast_ok || c.topo.uniform_bpd <= 0)
        return set_error(GH_ESTATE, "two-step launch: needs a uniform grid with p_w + p_g >= 0");
    return c.real_kind == GH_REAL_F32
               ? launch_step2f<float>(c, (const float*)in, (float*)out, dt, two, skip_still, (float*)mid)
               : launch_step2f<double>(c, (const double*)in, (double*)out, dt, two, skip_still, (double*)mid);
}

int rd_step2_buffers(Ctx& c, const void* in, void* out, void* mid, double dt, bool skip_still) {
    return step2f_buffers(c, in, out, mid, dt, true, skip_still);
}

int rd_step1_buffers(Ctx& c, const void* in, void* out, double dt, bool skip_still) {
    return step2f_buffers(c, in, out, nullptr, dt, false, skip_still);
}

int rd_step_buffers(Ctx& c, const void* in, void* out, double dt) {
    return c.real_kind == GH_REAL_F32 ? step_t<float, true>(c, (const float*)in, (float*)out, dt)
                                      : step_t<double, true>(c, (const double*)in, (double*)out, dt);
}

// Tile 0 takes two steps per launch.  A state written by the fused update is
// clamped, so after one single step from whatever state the call starts with,
// the pairs run rd_step2f_kernel when the anatomy allows it (fast_ok).  The
// still groups are marked after that step: one launch of 4-6 us, worth it from
// a few pairs on.
int rd_steps(Ctx& c, int64_t nsteps, double dt) {
    c.dt_last = dt;
    const bool ghosted = c.topo.uniform_bpd <= 0;
    const bool f32 = c.real_kind == GH_REAL_F32;
    int64_t k = 0;
    if (!ghosted && c.rd_bpw == 0) {
        const bool fast = c.fast_ok && nsteps >= 3;
        if (fast) {
            int rc = f32 ? step_t<float, true>(c, c.phi[1 - c.cur].as<float>())
                         : step_t<double, true>(c, c.phi[1 - c.cur].as<double>());
            if (rc) return rc;
            c.cur = 1 - c.cur;
            k = 1;
        }
        const bool skip = fast && c.nGrp > 0 && nsteps >= kStillMinSteps;
        if (skip)
            if (int rc = rd_mark_still(c, c.phi[c.cur].p, c.phi[1 - c.cur].p)) return rc;
        for (; k + 1 < nsteps; k += 2) {
            const int cur = c.cur;
            int rc = fast ? step2f_buffers(c, c.phi[cur].p, c.phi[1 - cur].p, nullptr, dt, true, skip)
                          : (f32 ? launch_step2<float>(c, c.phi[cur].as<float>(), c.phi[1 - cur].as<float>(), dt)
                                 : launch_step2<double>(c, c.phi[cur].as<double>(), c.phi[1 - cur].as<double>(), dt));
            if (rc) return rc;
            c.cur = 1 - c.cur;
        }
        if (fast && k < nsteps) {  // the odd step
            if (int rc = rd_step1_buffers(c, c.phi[c.cur].p, c.phi[1 - c.cur].p, dt, skip)) return rc;
            c.cur = 1 - c.cur;
            ++k;
        }
    }
    for (; k < nsteps; ++k) {
        int rc = ghosted ? rd_step_ghosted(c, c.phi[c.cur].p, c.phi[1 - c.cur].p, dt, true)
                 : c.real_kind == GH_REAL_F32 ? step_t<float, true>(c, c.phi[1 - c.cur].as<float>())
                                              : step_t<double, true>(c, c.phi[1 - c.cur].as<double>());
        if (rc) return rc;
        c.cur = 1 - c.cur;
    }
    return GH_OK;
}

template <typename Real>
static void thresholds_host(int64_t n, const Real* pw, const Real* pg, Real* tau, Real* sig) {
    for (int64_t i = 0; i < n; ++i) {
        tau[i] = chf_threshold(pw[i], pg[i]);
        sig[i] = domain_threshold(pw[i], pg[i]);
    }
}

}  // namespace gh

extern "C" int gh_rd_thresholds(int real_kind, int64_t n, const void* p_w, const void* p_g, void* tau, void* sigma) {
    if (n < 0 || (n > 0 && (!p_w || !p_g || !tau || !sigma)))
        return gh::set_error(GH_EINVAL, "gh_rd_thresholds: bad argument");
    if (real_kind == GH_REAL_F32)
        gh::thresholds_host(n, (const float*)p_w, (const float*)p_g, (float*)tau, (float*)sigma);
    else if (real_kind == GH_REAL_F64)
        gh::thresholds_host(n, (const double*)p_w, (const double*)p_g, (double*)tau, (double*)sigma);
    else
        return gh::set_error(GH_EINVAL, "gh_rd_thresholds: bad real_kind");
    return GH_OK;
}
