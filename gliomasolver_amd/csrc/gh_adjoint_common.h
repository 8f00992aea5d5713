// gh_adjoint_common.h -- reverse-step kernels of the discrete adjoint, shared
// by the single-solve adjoint (gh_adjoint.hip) and the batched one
// (gh_batch.hip).  The model and the per-cell formulas are documented at the
// top of gh_adjoint.hip.
#pragma once
#include "gh_rd_common.h"

#pragma clang fp contract(off)

namespace gh {

// LDS tiles of the reverse step: states and flags Q on [-2,10)^3, weights W on
// [-1,9)^3, with rows padded so that the 8 x 8 lanes of a wave meet few bank
// conflicts; 40.2 KB in FP32, four workgroups a CU, and shorter rows in FP64.
template <typename Real>
struct AdjTile {
    static constexpr int RQ = sizeof(Real) == 4 ? 24 : 12, PQ = sizeof(Real) == 4 ? 293 : 148;
    static constexpr int RW = sizeof(Real) == 4 ? 24 : 12, PW = 10 * RW;
    static constexpr int NQ = 12 * PQ, NW = 10 * PW;
    __device__ static inline int Q(int x, int y, int z) { return (z + 2) * PQ + (y + 2) * RQ + (x + 2); }
    __device__ static inline int W(int x, int y, int z) { return (z + 1) * PW + (y + 1) * RW + (x + 1); }
};

// Doubles of parameter-gradient partials per slot: per wave of the 512-lane
// workgroup the two sums A = sum w_c Rdiff_c and B = sum w_c u_c (1 - u_c)
// (Rdiff including ih2); the parameter gradients are linear in them
// (adj_param_grads).
constexpr int ADJ_PART = 2 * 8;

// dJ/dDw = dt A / Dw, dJ/drho = dt B, dJ/dT = sum w_c R_c / N = (A + rho B) / N
inline void adj_param_grads(const double ab[2], double dt, double invDw, double invN, double rho, double out[3]) {
    out[0] = dt * ab[0] * invDw;
    out[1] = dt * ab[1];
    out[2] = (ab[0] + rho * ab[1]) * invN;
}

__device__ inline double block_sum(double v, double* red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const int w = threadIdx.x / 64, lane = threadIdx.x % 64;
    __syncthreads();
    if (lane == 0) red[w] = v;
    __syncthreads();
    double s = 0;
    if (threadIdx.x == 0)
        for (int k = 0; k < (int)(blockDim.x / 64); ++k) s += red[k];
    return s;  // valid in thread 0
}

// adj_step_kernel's parameters as plain arguments (StepArgs)
struct AdjArgs {
    double rho, ih2, dt;
    int bpd;
    uint32_t magic;
    const int4* slots;
    const void* range;
};

// Per-slot parameters of the reverse step: one solve, or packed solves.
struct UniformAdjParams {
    double rho, ih2, dt;
    int bpd;
    uint32_t magic;  // bpd_magic(bpd)
    __host__ __device__ static inline UniformAdjParams make(double r, double i, double d, int b, uint32_t m, const int4*,
                                                            const void*) {
        return {r, i, d, b, m};
    }
    AdjArgs args() const { return {rho, ih2, dt, bpd, magic, nullptr, nullptr}; }
    using Item = int;
    __device__ static inline Item item(const int32_t* full, int i) { return full ? full[i] : i; }
    __device__ static inline Item item_of(int s) { return s; }
    __device__ static inline int slot(Item it) { return it; }
    __device__ inline void get(int, double& r, double& i, double& d) const {
        r = rho;
        i = ih2;
        d = dt;
    }
    __device__ inline BlockPos pos(int s) const { return block_pos(s, 0, bpd, magic); }
};

// Domain test and outside flag of a cell with state u and record r.  Generic
// records (CLAMPED false) carry tau, with the domain threshold in sig.  Clamped
// records (constants_kernel: every threshold <= 0, state u >= +0, i.e. any step
// k >= 1) carry +-max(tau, 0) with the sign set where the threshold is < 0:
// then u > sig holds there, and elsewhere it is u > 0; u < tau is
// u < max(tau, 0).
template <bool CLAMPED, typename Real>
__device__ inline bool adj_in_domain(Real u, const Stat4<Real>& r, const Real* sig, size_t g) {
    if (CLAMPED) return sign_of(r.tau) || u > (Real)0;
    return u > sig[g];
}

// Face halo cell (a, b) of face f at depth d (1 or 2): the cell index in the
// neighbour block across the face and the tile indices q (state, flags) and,
// at depth 1, p (w), each base + a * step_a + b * step_b with wave-uniform
// bases and steps (selects: no branch for a uniform f).
struct AdjHalo {
    int src, sa, sb, q, qa, qb, p, pa, pb;
};
template <typename Real>
__device__ inline AdjHalo adj_halo(int f, int d) {
    using T = AdjTile<Real>;
    const bool ax = f < 2, az = f >= 4;
    const int out = f & 1 ? 7 + d : -d, in = f & 1 ? d - 1 : 8 - d;
    return {(ax ? 1 : (az ? 64 : 8)) * in, ax ? 8 : 1, az ? 8 : 64,
            T::Q(0, 0, 0) + (ax ? 1 : (az ? T::PQ : T::RQ)) * out, ax ? T::RQ : 1, az ? T::RQ : T::PQ,
            T::W(0, 0, 0) + (ax ? 1 : (az ? T::PW : T::RW)) * out, ax ? T::RW : 1, az ? T::RW : T::PW};
}

// One cell of one reverse step: lambda_k (lk) and ih2 sum_i d'_i (u_i - u_c)
// (rdiff) from the face coefficients (-x, +x, -y, +y, -z, +z), per face i the
// outside flags of the opposite neighbour (that of face i ^ 1) and of the cell
// two steps out, the neighbour state and weight, and the cell's state u0,
// masked adjoint l1 and domain test.  axis(a) gives both faces of axis a; its
// data are read axis by axis (64 registers: eight waves a SIMD).
template <typename Real>
struct AdjAxis {
    Real dm, dp;      // face coefficients towards - and +
    Real um, up;      // neighbour states
    int om, op;       // their outside flags
    int om2, op2;     // the flags of the cells two steps out
    double wm, wp;    // neighbour weights
};
template <typename Axis>
__device__ inline void adj_cell(Axis axis, double u0, double l1, bool dom, double rho, double ih2, double dt,
                                double& lk, double& rdiff) {
    double sdu = 0, sumd = 0, acc = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const auto f = axis(a);
        // face coefficients doubled (exactly: ldexp by the 0/1 flag) where the
        // opposite neighbour of c, or of the neighbour, is outside
        auto face = [&](double d, int oo, int of, double un, double wn) {
            const double dd = ldexp(d, oo);
            sdu = fma(dd, un, sdu);
            sumd += dd;
            acc = fma(wn, ldexp(d, of), acc);
        };
        face((double)f.dm, f.op, f.om2, (double)f.um, f.wm);
        face((double)f.dp, f.om, f.op2, (double)f.up, f.wp);
        asm volatile("" : "+v"(sdu), "+v"(sumd), "+v"(acc));  // (the sums are formed here, not after the last axis)
    }
    rdiff = fma(-sumd, u0, sdu) * ih2;  // ih2 sum_i d'_i (u_i - u_c)
    const double self = dom ? l1 * (1. + dt * (-ih2 * sumd + rho * (1. - 2. * u0))) : l1;
    lk = self + dt * ih2 * acc;
}

// adds the wave's sums of a and b to its two words of block s
__device__ inline void adj_accumulate(double* __restrict__ partial, int s, double a, double b) {
    const double v = wave_sum2(a, b);
    const int t = threadIdx.x;
    if ((t & 31) == 0) partial[ADJ_PART * (size_t)s + 2 * (t >> 6) + ((t >> 5) & 1)] += v;
}

// lambda[c] = 0 where u[c] >= 1 (the upper clamp of the step that produced u
// is active): the masked adjoint the reverse step reads.
template <typename Real>
__device__ inline void adj_mask_cell(size_t c, double* __restrict__ lam, const Real* __restrict__ u) {
    if (!(u[c] < (Real)1)) lam[c] = 0.0;
}
template <typename Real>
__global__ __launch_bounds__(256) void adj_mask_kernel(size_t n, double* __restrict__ lam,
                                                       const Real* __restrict__ u) {
    const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c < n) adj_mask_cell(c, lam, u);
}

// One reverse step; one workgroup per block (XCD-aware order).  lam1 holds
// m lambda_{k+1} with m = [u_{k+1} < 1] (the seed masked by adj_mask_kernel,
// later steps by the previous launch); lam0 receives lambda_k, masked by
// [u_k < 1] when mask_out (k >= 1: the next reverse step reads it), plain
// at k = 0 (the initial-condition gradient reads it).
// partial[ADJ_PART s + 2 w + q] accumulates wave w's sums A (q = 0) and B
// (q = 1) of block s, step after step.  CLAMPED: st holds the clamped-state records and
// sig is not read (steps k >= 1 when every threshold is <= 0).
// Blocks without diffusion (constants_kernel; wk's groups): every face
// coefficient their cells use is +0, so each of adj_cell's face terms is a
// signed zero whatever the neighbour's state, flag or weight (finite values),
// the sums come out +0, and the cell's update is adj_cell with zero neighbour
// data -- the same bits with no halo and no LDS.  A still group (still_kernel)
// needs nothing at all for k >= 1: its adjoint stays what the seed put into
// both buffers, and its sums are zeros.
// Every load of a wave -- its cells' and its halo roles' -- is issued before the
// first wait, the sums of the previous steps with them, and halo and interior
// results keep registers of their own; with the interior stored to LDS before
// the halos were loaded the kernel waited for memory three times (128^3 FP32
// 7.6 -> 7.0 us with the tissue blocks only, 64^3 FP64 5.1 -> 4.4 us, a mixed
// population 24.3 -> 21.7 us).  On clamped states a neighbour's outside flag travels in
// the sign bit of its LDS copy (rd_step2f_kernel).
template <typename Real, typename Params, bool CLAMPED = false>
__global__ __launch_bounds__(512) void adj_step_kernel(
    int nfull, int fper, const int32_t* __restrict__ full, const Real* __restrict__ uk,
    const Stat4<Real>* __restrict__ st, int bpd, uint32_t magic, const int4* __restrict__ slots,
    const void* __restrict__ range, const double* __restrict__ lam1, double* __restrict__ lam0,
    const Real* __restrict__ sig, double* __restrict__ partial, int mask_out, double rho_, double ih2_, double dt_,
    int ngrp, int gper, const int2* __restrict__ grp, const unsigned char* __restrict__ still) {
    const StepWork wk{nfull, fper, ngrp, gper, full, grp, still};
    const Params prm = Params::make(rho_, ih2_, dt_, bpd, magic, slots, range);
    int nzf;
    typename Params::Item it;
    const int s = wk.item(prm, &nzf, it);
    if (s < 0) return;
    double rho, ih2, dt;
    prm.get(it, rho, ih2, dt);  // a group's blocks belong to one solve
    const int t = threadIdx.x;
    for (int b = 0; b < nzf; ++b) {  // uniform per workgroup
        const size_t g = (size_t)(s + b) * BCELLS + t;
        const Real uc = uk[g];
        const Stat4<Real> sv = st[g];
        const bool domc = adj_in_domain<CLAMPED>(uc, sv, sig, g);
        const double l1c = lam1[g];
        const double u0 = (double)uc;
        double lk, rdiff;
        adj_cell([](int) { return AdjAxis<Real>{0, 0, 0, 0, 0, 0, 0, 0, 0., 0.}; }, u0, l1c, domc, rho, ih2, dt, lk,
                 rdiff);
        lam0[g] = (mask_out && !(uc < (Real)1)) ? 0.0 : lk;
        const double wc = domc ? l1c : 0.0;
        adj_accumulate(partial, s + b, wc * rdiff, wc * (u0 * (1. - u0)));
    }
    if (nzf > 0) return;
    using T = AdjTile<Real>;
    __shared__ Real s_u[T::NQ];
    __shared__ unsigned char s_o[CLAMPED ? 1 : T::NQ];
    __shared__ double s_w[T::NW];
    __shared__ Real s_Dx[576], s_Dy[576], s_Dz[576];

    const int x = t & 7, y = (t >> 3) & 7, z = t >> 6;
    const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const size_t base = (size_t)s * BCELLS;
    const unsigned ut = (unsigned)t;
    const BlockPos bp = prm.pos(it);
    // halo roles: waves 0-5 the depth-1 cells of face wv (state, flags, w,
    // minus-face D), waves 6, 7 and 0-3 the depth-2 cells of faces 0-5 (state,
    // flags)
    const int f2 = wv >= 6 ? wv - 6 : wv + 2;
    const bool deep = wv >= 6 || wv < 4;
    Real u_1, u_2, tau_2;  // no defaults: merging them with loaded values would wait for the loads
    Stat4<Real> st_1;
    double l_1;
    int q1 = 0, p1 = 0, q2 = 0;
    bool dom_1 = false;
    size_t g1 = 0;
    if (wv < 6) {
        const AdjHalo m = adj_halo<Real>(wv, 1);
        const size_t nb = (size_t)face_nb(bp, wv) * BCELLS;
        const unsigned l = (unsigned)mad24(y, m.sb, mad24(x, m.sa, m.src)) & (BCELLS - 1);
        u_1 = (uk + nb)[l];
        st_1 = (st + nb)[l];
        l_1 = (lam1 + nb)[l];
        g1 = nb + l;
        q1 = mad24(y, m.qb, mad24(x, m.qa, m.q));
        p1 = mad24(y, m.pb, mad24(x, m.pa, m.p));
    }
    if (deep) {
        const AdjHalo m = adj_halo<Real>(f2, 2);
        const size_t nb = (size_t)face_nb(bp, f2) * BCELLS;
        const unsigned l = (unsigned)mad24(y, m.sb, mad24(x, m.sa, m.src)) & (BCELLS - 1);
        u_2 = (uk + nb)[l];
        tau_2 = (st + nb)[l].tau;
        q2 = mad24(y, m.qb, mad24(x, m.qa, m.q));
    }
    const Real uc = (uk + base)[ut];
    const Stat4<Real> sv = (st + base)[ut];
    const double l1c = (lam1 + base)[ut];
    double* pw = partial + ADJ_PART * (size_t)s + 2 * wv + ((t >> 5) & 1);
    const double sum0 = *pw;  // the sums of the steps before
    const bool domc = adj_in_domain<CLAMPED>(uc, sv, sig, base + ut);
    if (wv < 6) dom_1 = adj_in_domain<CLAMPED>(u_1, st_1, sig, g1);

    auto put = [&](int q, Real u, Real tau) {  // a state and its outside flag
        if constexpr (CLAMPED) {
            s_u[q] = flag_in_sign(u, std::fabs(tau));
        } else {
            s_u[q] = u;
            s_o[q] = u < tau;
        }
    };
    put(T::Q(x, y, z), uc, sv.tau);
    s_w[T::W(x, y, z)] = domc ? l1c : 0.0;
    s_Dx[z * 72 + y * 9 + x + 1] = sv.dx;
    s_Dy[z * 72 + (y + 1) * 8 + x] = sv.dy;
    s_Dz[(z + 1) * 64 + y * 8 + x] = sv.dz;
    if (wv < 6) {
        put(q1, u_1, st_1.tau);
        s_w[p1] = dom_1 ? l_1 : 0.0;
        if (wv == FXM) s_Dx[y * 72 + x * 9] = st_1.dx;
        else if (wv == FYM) s_Dy[y * 72 + x] = st_1.dy;
        else if (wv == FZM) s_Dz[y * 8 + x] = st_1.dz;
    }
    if (deep) put(q2, u_2, tau_2);
    __syncthreads();

    const double u0 = (double)uc;
    const int q0 = T::Q(x, y, z), w0 = T::W(x, y, z);
    double lk, rdiff;
    adj_cell(
        [&](int a) {
            const int dq = a == 0 ? 1 : (a == 1 ? T::RQ : T::PQ), dw = a == 0 ? 1 : (a == 1 ? T::RW : T::PW);
            AdjAxis<Real> f;
            f.dm = a == 0 ? s_Dx[z * 72 + y * 9 + x] : (a == 1 ? s_Dy[z * 72 + y * 8 + x] : s_Dz[z * 64 + y * 8 + x]);
            f.dp = a == 0 ? sv.dx : (a == 1 ? sv.dy : sv.dz);
            const Real em = s_u[q0 - dq], ep = s_u[q0 + dq];
            if constexpr (CLAMPED) {
                f.um = std::fabs(em);
                f.up = std::fabs(ep);
                f.om = (int)sign_of(em);
                f.op = (int)sign_of(ep);
                f.om2 = (int)sign_of(s_u[q0 - 2 * dq]);
                f.op2 = (int)sign_of(s_u[q0 + 2 * dq]);
            } else {
                f.um = em;
                f.up = ep;
                f.om = s_o[q0 - dq];
                f.op = s_o[q0 + dq];
                f.om2 = s_o[q0 - 2 * dq];
                f.op2 = s_o[q0 + 2 * dq];
            }
            f.wm = s_w[w0 - dw];
            f.wp = s_w[w0 + dw];
            return f;
        },
        u0, l1c, domc, rho, ih2, dt, lk, rdiff);
    (lam0 + base)[ut] = (mask_out && !(uc < (Real)1)) ? 0.0 : lk;
    const double wc = domc ? l1c : 0.0;
    const double v = sum0 + wave_sum2(wc * rdiff, wc * (u0 * (1. - u0)));
    if ((t & 31) == 0) *pw = v;
}

template <bool CLAMPED, typename Real, typename Params>
inline void launch_adj_step(hipStream_t stream, const StepWork& wk, const Real* uk, int mask_out, const double* lam1,
                            double* lam0, const Stat4<Real>* st, const Real* sig, const Params& prm, double* partial) {
    const AdjArgs q = prm.args();
    hipLaunchKernelGGL((adj_step_kernel<Real, Params, CLAMPED>), dim3(wk.grid()), dim3(512), 0, stream, wk.nfull,
                       wk.fper, wk.full, uk, st, q.bpd, q.magic, q.slots, q.range, lam1, lam0, sig, partial,
                       mask_out, q.rho, q.ih2, q.dt, wk.ngrp, wk.gper, wk.grp, wk.still);
}

// sum over cells of lam0 * u0 * (X - x0) / sigma^2 for X = ix, iy, iz, by
// workgroup wg of nwg (256 lanes): partial[3 wg + q]
template <typename Real>
__device__ inline void adj_ic_body(int wg, int nwg, size_t nc, int bpd, const double* __restrict__ lam,
                                   const Real* __restrict__ u0, double x0, double y0, double z0, double is2,
                                   double* __restrict__ partial) {
    double a[3] = {0, 0, 0};
    for (size_t c = (size_t)wg * 256 + threadIdx.x; c < nc; c += (size_t)nwg * 256) {
        const int s = (int)(c / BCELLS), l = (int)(c % BCELLS);
        const double ix = (s % bpd) * BS + (l & 7), iy = ((s / bpd) % bpd) * BS + ((l >> 3) & 7),
                     iz = (s / (bpd * bpd)) * BS + (l >> 6);
        const double v = lam[c] * (double)u0[c] * is2;
        a[0] += v * (ix - x0);
        a[1] += v * (iy - y0);
        a[2] += v * (iz - z0);
    }
    __shared__ double red[8];
    for (int q = 0; q < 3; ++q) {
        const double sq = block_sum(a[q], red);
        if (threadIdx.x == 0) partial[3 * wg + q] = sq;
    }
}

template <typename Real>
__global__ __launch_bounds__(256) void adj_ic_partials(size_t nc, int bpd, const double* __restrict__ lam,
                                                       const Real* __restrict__ u0, double x0, double y0, double z0,
                                                       double is2, double* __restrict__ partial) {
    adj_ic_body<Real>((int)blockIdx.x, (int)gridDim.x, nc, bpd, lam, u0, x0, y0, z0, is2, partial);
}

// A solve's sums A, B over its n slots and the three initial-condition sums over
// ADJ_IC_GRID partials, by one workgroup of 512 lanes in a fixed order.  (The
// partials of twelve mixed samples were 3 MB copied to pageable memory and added
// one after another on the host: 0.4 of 20.7 ms; of 64^3 FP64 0.1 of 2.7 ms.)
constexpr int ADJ_IC_GRID = 512;
constexpr int ADJ_SUMS = 5;
__device__ inline void adj_reduce_body(const double* __restrict__ part, size_t n, const double* __restrict__ ic,
                                       double* __restrict__ out) {
    static_assert(ADJ_PART % 2 == 0 && ADJ_IC_GRID == 512, "even words are A's, odd ones B's; a lane per partial");
    __shared__ double red[ADJ_SUMS][8];
    const int t = threadIdx.x;
    double a[4] = {0, 0, 0, 0};
    const size_t m = n * ADJ_PART;  // a multiple of 16
    size_t i = t;
    for (; i + 3 * 512 < m; i += 4 * 512)
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] += part[i + 512 * k];
    for (int k = 0; i < m; i += 512, ++k) a[k] += part[i];
    double v = (a[0] + a[1]) + (a[2] + a[3]), g[3];
    for (int q = 0; q < 3; ++q) g[q] = ic[3 * t + q];
    for (int o = 32; o > 1; o >>= 1) v += __shfl_xor(v, o, 64);  // lane 0: A's, lane 1: B's
    for (int o = 32; o > 0; o >>= 1)
        for (int q = 0; q < 3; ++q) g[q] += __shfl_xor(g[q], o, 64);
    const int w = t >> 6, lane = t & 63;
    if (lane < 2) red[lane][w] = v;
    if (lane == 0)
        for (int q = 0; q < 3; ++q) red[2 + q][w] = g[q];
    __syncthreads();
    if (t < ADJ_SUMS) {
        double s = 0;
        for (int k = 0; k < 8; ++k) s += red[t][k];
        out[t] = s;
    }
}

}  // namespace gh
