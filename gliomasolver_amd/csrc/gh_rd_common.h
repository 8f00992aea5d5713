// gh_rd_common.h -- per-cell arithmetic of the RD operator shared by the HIP
// kernels and host-side utilities (__host__ __device__).
//
// Reference: Glioma/Operators/ReactionDiffusionOperator.h.  Every expression
// keeps the reference's rounding points for Real = float and Real = double;
// translation units including this header are compiled with
// -ffp-contract=off.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <limits>
#include <vector>

#include "gh_internal.h"

#pragma clang fp contract(off)

namespace gh {

// Per-cell constants of one solve, one 4-Real record per cell so a lane
// fetches them with one vector load: harmonic diffusivity of the cell's +x,
// +y, +z faces and the outside threshold tau.
template <typename Real>
struct alignas(4 * sizeof(Real)) Stat4 {
    Real dx, dy, dz, tau;
};

// ordered integer keys: okey(a) < okey(b) iff a < b for non-NaN a, b
// (except -0 < +0, harmless: the predicates below agree on both zeros)
__host__ __device__ inline int64_t okey(float x) {
    const int32_t b = __builtin_bit_cast(int32_t, x);
    return b >= 0 ? (int64_t)b : (int64_t)(b ^ 0x7fffffff);
}
__host__ __device__ inline float okey_inv(int64_t k, float) {
    const int32_t kk = (int32_t)k;
    return __builtin_bit_cast(float, kk >= 0 ? kk : (kk ^ 0x7fffffff));
}
__host__ __device__ inline int64_t okey(double x) {
    const int64_t b = __builtin_bit_cast(int64_t, x);
    return b >= 0 ? b : (b ^ 0x7fffffffffffffffLL);
}
__host__ __device__ inline double okey_inv(int64_t k, double) {
    return __builtin_bit_cast(double, k >= 0 ? k : (k ^ 0x7fffffffffffffffLL));
}
template <typename Real> __host__ __device__ inline Real real_max();
template <> __host__ __device__ inline float real_max<float>() { return FLT_MAX; }
template <> __host__ __device__ inline double real_max<double>() { return DBL_MAX; }

// df = p_w*Dw + p_g*Dg in Real (ReactionDiffusionOperator.h:105-111)
template <typename Real>
__host__ __device__ inline Real diffusivity(Real pw, Real pg, Real Dw, Real Dg) {
    const Real a = pw * Dw;
    const Real b = pg * Dg;
    return a + b;
}

// _harmonic_mean (ReactionDiffusionOperator.h:148-163) seen from a cell with
// df_loc = dc and neighbour dn: (dn+dc < 1e-8) ? 0 : 2.*dn*dc/(dn+dc), the
// quotient in double, the sum in Real.  (2*dn)*dc and (2*dc)*dn are the same
// double and dn+dc commutes, so both cells of a face get the same value.
template <typename Real>
__host__ __device__ inline Real harmonic(Real dn, Real dc) {
    const Real s = dn + dc;
    if (s < (Real)1.0e-08) return (Real)0.;
    return (Real)(((2. * (double)dn) * (double)dc) / (double)s);
}

// chf = phi + p_w + p_g (Real, left to right) < 0.1 marks an outside neighbour
// (ReactionDiffusionOperator.h:115-120, 166-171).  The predicate is monotone
// in phi, so it equals "phi < tau" with tau the smallest Real for which it is
// false; tau is found by bisection over the ordered bit patterns.  It lies a
// few roundings from 0.1 - (p_w + p_g): where the predicate holds just below
// that neighbourhood and not just above it, the bisection starts from there
// (about 5 steps instead of 32 in FP32 and 63 in FP64).
template <typename Real>
__host__ __device__ inline bool chf_outside(Real phi, Real pw, Real pg) {
    Real t = phi + pw;
    t = t + pg;
    return t < (Real)0.1;
}

template <typename Real>
__host__ __device__ inline Real chf_threshold(Real pw, Real pg) {
    const Real M = real_max<Real>();
    const Real g = (Real)0.1 - (pw + pg);
    const Real e = 4 * std::numeric_limits<Real>::epsilon() * (std::fabs(pw) + std::fabs(pg) + (Real)0.1);
    int64_t lo, hi;  // outside at lo, not outside at hi
    if (std::fabs(g) + e < M && chf_outside(g - e, pw, pg) && !chf_outside(g + e, pw, pg)) {
        lo = okey(g - e);
        hi = okey(g + e);
    } else {
        if (!chf_outside(-M, pw, pg)) return -(Real)INFINITY;
        if (chf_outside(M, pw, pg)) return (Real)INFINITY;
        lo = okey(-M);
        hi = okey(M);
    }
    while ((uint64_t)hi - (uint64_t)lo > 1) {
        const int64_t mid = lo + (int64_t)(((uint64_t)hi - (uint64_t)lo) >> 1);
        if (chf_outside(okey_inv(mid, (Real)0), pw, pg)) lo = mid;
        else hi = mid;
    }
    return okey_inv(hi, (Real)0);
}

// p_w + p_g + phi > 0 (ReactionDiffusionOperator.h:103) <=> phi > -(p_w+p_g):
// an exact sum of two Reals is > 0 iff its rounding is > 0.
template <typename Real>
__host__ __device__ inline Real domain_threshold(Real pw, Real pg) {
    const Real s = pw + pg;
    return -s;
}

// p_w + p_g = 0 with p_w = -p_g != 0: a cell outside the domain (at phi = 0)
// whose face coefficients need not be zeros
template <typename Real>
__host__ __device__ inline bool cancels(Real pw, Real pg) {
    return pw != (Real)0 && pw + pg == (Real)0;
}

// LDS index of cell (x, y, z) in a 10^3 block tile with a one-cell halo
__device__ inline int P(int x, int y, int z) { return (z + 1) * 100 + (y + 1) * 10 + (x + 1); }

// dphidt of one cell (ReactionDiffusionOperator.h:103-138) from its six face
// coefficients d0..d5 (-x,+x,-y,+y,-z,+z) after the no-flux rule, the
// neighbour values p0..p5, its own value pc and whether it lies in the brain
// domain.
template <typename Real>
__device__ inline Real rd_rhs_core(Real d0, Real d1, Real d2, Real d3, Real d4, Real d5, Real p0, Real p1, Real p2,
                                   Real p3, Real p4, Real p5, Real pc, bool dom, Real rho, double ih2) {
    // diffusionFluxIn = ih2 * (Real sum of df_i*phi_i, left to right)
    Real sin_ = d0 * p0;
    sin_ = sin_ + d1 * p1;
    sin_ = sin_ + d2 * p2;
    sin_ = sin_ + d3 * p3;
    sin_ = sin_ + d4 * p4;
    sin_ = sin_ + d5 * p5;
    const double fin = ih2 * (double)sin_;
    // diffusionFluxOut = -((Real sum of df_i) * phi * ih2)
    Real sdf = d0 + d1;
    sdf = sdf + d2;
    sdf = sdf + d3;
    sdf = sdf + d4;
    sdf = sdf + d5;
    const Real sdp = sdf * pc;
    const double fout = -((double)sdp * ih2);
    // reactionFlux = (Real)(rho*phi) * (1. - phi)
    const Real rp = rho * pc;
    const double react = (double)rp * (1. - (double)pc);
    const Real dphidt = (Real)((fout + fin) + react);
    return dom ? dphidt : (Real)0.;  // outside the brain domain (:103, :137-138)
}

// dphidt of one cell from its face coefficients d0..d5 before the no-flux
// rule, the neighbour values p0..p5 with their outside flags o0..o5, its own
// value pc and domain threshold sc.
template <typename Real>
__device__ inline Real rd_cell_rhs(Real d0, Real d1, Real d2, Real d3, Real d4, Real d5, Real p0, Real p1, Real p2,
                                   Real p3, Real p4, Real p5, bool o0, bool o1, bool o2, bool o3, bool o4, bool o5,
                                   Real pc, Real sc, Real rho, double ih2) {
    // _applyNoFluxBC: an outside neighbour doubles the opposite face (exact)
    if (o0) d1 = (Real)((double)d1 * 2.0);
    if (o1) d0 = (Real)((double)d0 * 2.0);
    if (o2) d3 = (Real)((double)d3 * 2.0);
    if (o3) d2 = (Real)((double)d2 * 2.0);
    if (o4) d5 = (Real)((double)d5 * 2.0);
    if (o5) d4 = (Real)((double)d4 * 2.0);
    return rd_rhs_core<Real>(d0, d1, d2, d3, d4, d5, p0, p1, p2, p3, p4, p5, pc, pc > sc, rho, ih2);
}

// UpdateTumor (ReactionDiffusionOperator.h:219-221): phi += dt*dphidt in
// double, then std::max((Real)0, .), std::min((Real)1, .)
template <typename Real>
__device__ inline Real rd_update(Real pc, Real dphidt, double dt) {
    Real p = (Real)((double)pc + dt * (double)dphidt);
    p = ((Real)0. < p) ? p : (Real)0.;
    return (p < (Real)1.) ? p : (Real)1.;
}

// Position of a block in a uniform periodic grid of bpd^3 blocks whose slots
// start at slot0 (slot = slot0 + bx + bpd*(by + bpd*bz)): the step kernels
// find neighbour blocks by arithmetic on the workgroup-uniform block index,
// so no halo load waits on a table load.
struct BlockPos {
    int slot0, bpd, bx, by, bz;
    __device__ inline int nb(int dx, int dy, int dz) const {
        int x = bx + dx, y = by + dy, z = bz + dz;
        x += x < 0 ? bpd : 0;
        x -= x >= bpd ? bpd : 0;
        y += y < 0 ? bpd : 0;
        y -= y >= bpd ? bpd : 0;
        z += z < 0 ? bpd : 0;
        z -= z >= bpd ? bpd : 0;
        return slot0 + x + bpd * (y + bpd * z);
    }
};
// magic multiplier of the division by bpd in block_pos: m = ceil(2^32 / bpd),
// m * bpd = 2^32 + r with 0 <= r < bpd.  floor(l * m / 2^32) = floor(l / bpd)
// whenever l * r < 2^32: always for a power of two (r = 0), and for l < bpd^3
// with bpd <= 64 otherwise (bpd = 1 has l = 0 only).
__host__ __device__ inline uint32_t bpd_magic(int bpd) {
    return bpd <= 1 ? 0xffffffffu : (uint32_t)((0x100000000ull + (uint64_t)bpd - 1) / (uint64_t)bpd);
}
__device__ inline BlockPos block_pos(int s, int slot0, int bpd, uint32_t magic) {
    const uint32_t l = (uint32_t)(s - slot0);
    const uint32_t q = __umulhi(l, magic);  // l / bpd
    const uint32_t z = __umulhi(q, magic);  // l / bpd^2
    return BlockPos{slot0, bpd, (int)(l - q * (uint32_t)bpd), (int)(q - z * (uint32_t)bpd), (int)z};
}
// unit offset of face f (FXM, FXP, FYM, FYP, FZM, FZP)
__device__ inline int face_dx(int f) { return f == FXM ? -1 : (f == FXP ? 1 : 0); }
__device__ inline int face_dy(int f) { return f == FYM ? -1 : (f == FYP ? 1 : 0); }
__device__ inline int face_dz(int f) { return f == FZM ? -1 : (f == FZP ? 1 : 0); }
__device__ inline int face_nb(const BlockPos& p, int f) { return p.nb(face_dx(f), face_dy(f), face_dz(f)); }

// v moved across lanes by the DPP pattern CTRL (both 32-bit halves)
template <int CTRL>
__device__ inline double dpp_move(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)b, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ inline double double_of(unsigned lo, unsigned hi) {
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ inline unsigned lo_of(double v) { return (unsigned)(unsigned long long)__double_as_longlong(v); }
__device__ inline unsigned hi_of(double v) { return (unsigned)((unsigned long long)__double_as_longlong(v) >> 32); }
// Sums of a and of b over the 64 lanes of a wave (all lanes active): a's in
// lanes 0-31, b's in lanes 32-63.  The halves of the wave are exchanged so that
// one addition leaves a's 32 partial sums in the lower and b's in the upper
// half, then the rows of 16 lanes, then butterflies within a row (lane pairs,
// quad halves, row half mirror, row mirror: floating-point addition commutes,
// so every lane of a row ends with the same sum).  Fixed order, no LDS, no
// barrier; 21 operations for both sums (42 with one reduction each).
__device__ inline double wave_sum2(double a, double b) {
    auto lo = __builtin_amdgcn_permlane32_swap(lo_of(a), lo_of(b), false, false);
    auto hi = __builtin_amdgcn_permlane32_swap(hi_of(a), hi_of(b), false, false);
    double v = double_of(lo[0], hi[0]) + double_of(lo[1], hi[1]);
    lo = __builtin_amdgcn_permlane16_swap(lo_of(v), lo_of(v), false, false);
    hi = __builtin_amdgcn_permlane16_swap(hi_of(v), hi_of(v), false, false);
    v = double_of(lo[0], hi[0]) + double_of(lo[1], hi[1]);
    v += dpp_move<0xB1>(v);   // quad_perm [1,0,3,2]
    v += dpp_move<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp_move<0x141>(v);  // row_half_mirror
    v += dpp_move<0x140>(v);  // row_mirror
    return v;
}

// rd_step2f_kernel's parameters as plain arguments: the scalars that its first
// loads depend on lie in front, where they are in registers when a wave starts
// (build.py: kernarg preload), 0.4 us of a 6.1 us pair of steps at 128^3.
template <typename Real>
struct StepArgs {
    Real rho;
    double ih2, dt;
    int bpd;
    uint32_t magic;
    const int4* slots;  // packed solves: where a slot lies, and its solve's SlotRange
    const void* range;
};

// Step parameters of a slot: one solve (the same rho, 1/h^2, dt for every
// slot) or many independent solves packed slot range after slot range.
template <typename Real>
struct UniformStepParams {
    Real rho;
    double ih2, dt;
    int bpd;
    uint32_t magic;  // bpd_magic(bpd)
    static constexpr bool kPow2 = true;  // h = 2^-level / 8
    __host__ __device__ static inline UniformStepParams make(Real r, double i, double d, int b, uint32_t m,
                                                             const int4*, const void*) {
        return {r, i, d, b, m};
    }
    StepArgs<Real> args() const { return {rho, ih2, dt, bpd, magic, nullptr, nullptr}; }
    // what a work list's entry, or a slot alone, tells of a block
    using Item = int;
    __device__ static inline Item item(const int32_t* full, int i) { return full ? full[i] : i; }
    __device__ static inline Item item_of(int s) { return s; }
    __device__ static inline int slot(Item it) { return it; }
    __device__ inline void get(int, Real& r, double& i, double& d) const {
        r = rho;
        i = ih2;
        d = dt;
    }
    __device__ inline BlockPos pos(int s) const { return block_pos(s, 0, bpd, magic); }
};
// Packed solves: {slot, the solve's first slot, blocks per side | x << 8 | y << 16 |
// z << 24, the solve}, 16 B in one scalar load.  (The slot, its solve, the solve's
// first slot and a division were three loads in a row before a workgroup's first
// load of a cell: 24 samples of 96^3, a pair of steps 21.1 -> 20.5 us.)
struct PackedItems {
    using Item = int4;
    const int4* __restrict__ slots;
    __device__ inline Item item(const int32_t* full, int i) const {
        return (full ? reinterpret_cast<const int4*>(full) : slots)[i];
    }
    __device__ inline Item item_of(int s) const { return slots[s]; }
    __device__ static inline int slot(const Item& it) { return it.x; }
    __device__ static inline BlockPos pos(const Item& it) {
        return BlockPos{it.y, it.z & 0xff, (it.z >> 8) & 0xff, (it.z >> 16) & 0xff, (it.z >> 24) & 0xff};
    }
    __device__ inline BlockPos pos(int s) const { return pos(slots[s]); }
};

// Two fused Euler steps per launch (temporal blocking): one workgroup per 8^3
// block.  Step 1 is evaluated on the block and its six depth-1 face halos
// (the cells step 2 reads), from the state on the block, the depth-1 and
// depth-2 face halos and the twelve edge rows next to the depth-1 halos; step
// 2 then runs on the block from the step-1 values in LDS.  A halo cell's
// step-1 value is computed with exactly the inputs and arithmetic its own
// block uses, so two launches of rd_step_kernel and one of this kernel give
// the same bits.  Per two steps a block reads 1,376 states and constant
// records (512 + 864 halo) instead of 2 x 896.
__device__ inline int T12(int x, int y, int z) { return (z + 2) * 144 + (y + 2) * 12 + (x + 2); }  // [-2,10)^3

template <typename Real, typename Params>
__global__ __launch_bounds__(512) void rd_step2_kernel(int nslots, int per_xcd,
                                                       const Real* __restrict__ phi, Real* __restrict__ out,
                                                       const Stat4<Real>* __restrict__ st,
                                                       const Real* __restrict__ sig, Params prm) {
    const int s = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (s >= nslots) return;
    __shared__ Real s_u0[1728], s_tau[1728], s_dx[1728], s_dy[1728], s_dz[1728];
    __shared__ Real s_u1[1000];

    const int t = threadIdx.x;
    const int x = t & 7, y = (t >> 3) & 7, z = t >> 6;
    const size_t g = (size_t)s * BCELLS + t;
    const Real pc0 = phi[g];
    const Stat4<Real> sv = st[g];
    const Real sc = sig[g];
    const BlockPos bp = prm.pos(s);
    // halo cells: [0,384) depth-1 faces, [384,768) depth-2 faces, [768,864) edge rows
    Real hsig = 0;         // sigma of this lane's depth-1 face cell (lanes < 384)
    int fx = 0, fy = 0, fz = 0;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const int h = t + 512 * it;
        if (h >= 864) break;
        int src_slot, lx, ly, lz, tx, ty, tz;
        if (h < 768) {
            const int d = h < 384 ? 1 : 2;
            const int r = h % 384, f = r >> 6, a = r & 7, b = (r >> 3) & 7;
            src_slot = face_nb(bp, f);
            switch (f) {
                case FXM: tx = -d; ty = a; tz = b; lx = 8 - d; ly = a; lz = b; break;
                case FXP: tx = 7 + d; ty = a; tz = b; lx = d - 1; ly = a; lz = b; break;
                case FYM: tx = a; ty = -d; tz = b; lx = a; ly = 8 - d; lz = b; break;
                case FYP: tx = a; ty = 7 + d; tz = b; lx = a; ly = d - 1; lz = b; break;
                case FZM: tx = a; ty = b; tz = -d; lx = a; ly = b; lz = 8 - d; break;
                default:  tx = a; ty = b; tz = 7 + d; lx = a; ly = b; lz = d - 1; break;
            }
        } else {
            const int e = (h - 768) >> 3, i = (h - 768) & 7;
            const int pair = e >> 2, s1 = e & 1, s2 = (e >> 1) & 1;
            const int c1 = s1 ? 8 : -1, c2 = s2 ? 8 : -1;  // tile coordinate on the two crossed axes
            const int l1 = s1 ? 0 : 7, l2 = s2 ? 0 : 7;    // local coordinate in the diagonal block
            int f1, f2;
            if (pair == 0) {         // x and y crossed, z free
                f1 = s1 ? FXP : FXM; f2 = s2 ? FYP : FYM;
                tx = c1; ty = c2; tz = i; lx = l1; ly = l2; lz = i;
            } else if (pair == 1) {  // x and z crossed, y free
                f1 = s1 ? FXP : FXM; f2 = s2 ? FZP : FZM;
                tx = c1; ty = i; tz = c2; lx = l1; ly = i; lz = l2;
            } else {                 // y and z crossed, x free
                f1 = s1 ? FYP : FYM; f2 = s2 ? FZP : FZM;
                tx = i; ty = c1; tz = c2; lx = i; ly = l1; lz = l2;
            }
            src_slot = bp.nb(face_dx(f1) + face_dx(f2), face_dy(f1) + face_dy(f2), face_dz(f1) + face_dz(f2));
        }
        const size_t gs = (size_t)src_slot * BCELLS + lx + 8 * ly + 64 * lz;
        const int q = T12(tx, ty, tz);
        const Stat4<Real> hs = st[gs];
        s_u0[q] = phi[gs];
        s_tau[q] = hs.tau;
        s_dx[q] = hs.dx;
        s_dy[q] = hs.dy;
        s_dz[q] = hs.dz;
        if (h < 384) {
            hsig = sig[gs];
            fx = tx; fy = ty; fz = tz;
        }
    }
    {
        const int q = T12(x, y, z);
        s_u0[q] = pc0;
        s_tau[q] = sv.tau;
        s_dx[q] = sv.dx;
        s_dy[q] = sv.dy;
        s_dz[q] = sv.dz;
    }
    Real rho;
    double ih2, dt;
    prm.get(s, rho, ih2, dt);
    __syncthreads();

    // step 1 on the block cell of this lane and (lanes < 384) one depth-1 face cell
    auto step1 = [&](int cx, int cy, int cz, Real sc1) {
        const int q = T12(cx, cy, cz);
        const int n0 = T12(cx - 1, cy, cz), n1 = T12(cx + 1, cy, cz), n2 = T12(cx, cy - 1, cz),
                  n3 = T12(cx, cy + 1, cz), n4 = T12(cx, cy, cz - 1), n5 = T12(cx, cy, cz + 1);
        const Real p0 = s_u0[n0], p1 = s_u0[n1], p2 = s_u0[n2], p3 = s_u0[n3], p4 = s_u0[n4], p5 = s_u0[n5];
        const Real pc = s_u0[q];
        const Real d = rd_cell_rhs<Real>(s_dx[n0], s_dx[q], s_dy[n2], s_dy[q], s_dz[n4], s_dz[q], p0, p1, p2, p3, p4,
                                         p5, p0 < s_tau[n0], p1 < s_tau[n1], p2 < s_tau[n2], p3 < s_tau[n3],
                                         p4 < s_tau[n4], p5 < s_tau[n5], pc, sc1, rho, ih2);
        s_u1[P(cx, cy, cz)] = rd_update(pc, d, dt);
    };
    step1(x, y, z, sc);
    if (t < 384) step1(fx, fy, fz, hsig);
    __syncthreads();

    // step 2 on the block
    {
        const int q = T12(x, y, z);
        const int n0 = T12(x - 1, y, z), n1 = T12(x + 1, y, z), n2 = T12(x, y - 1, z), n3 = T12(x, y + 1, z),
                  n4 = T12(x, y, z - 1), n5 = T12(x, y, z + 1);
        const Real p0 = s_u1[P(x - 1, y, z)], p1 = s_u1[P(x + 1, y, z)], p2 = s_u1[P(x, y - 1, z)],
                   p3 = s_u1[P(x, y + 1, z)], p4 = s_u1[P(x, y, z - 1)], p5 = s_u1[P(x, y, z + 1)];
        const Real pc = s_u1[P(x, y, z)];
        const Real d = rd_cell_rhs<Real>(s_dx[n0], s_dx[q], s_dy[n2], s_dy[q], s_dz[n4], s_dz[q], p0, p1, p2, p3, p4,
                                         p5, p0 < s_tau[n0], p1 < s_tau[n1], p2 < s_tau[n2], p3 < s_tau[n3],
                                         p4 < s_tau[n4], p5 < s_tau[n5], pc, sc, rho, ih2);
        out[g] = rd_update(pc, d, dt);
    }
}

// ---------------------------------------------------------------------------
// Two fused steps per launch on clamped states (rd_step2f_kernel).
//
// Preconditions, checked by the callers: every state value has a clear sign
// bit (true of any state written by the fused update, whose clamp returns +0
// for p <= 0 and for NaN), and every cell has p_w + p_g >= 0.  Then
//   * "phi < tau" equals "phi < max(tau, +0)" and "phi > sigma" equals
//     "sigma < 0 or phi > 0", so one record {D+x, D+y, D+z, tau_enc} per cell
//     (tau_enc = max(tau, +0), negated for cells with sigma < 0) carries all
//     per-solve constants (StatFast);
//   * a neighbour's outside flag travels in the sign bit of its value in LDS
//     (-phi when phi < tau), so a stencil reads six values instead of six
//     values and six thresholds, and the flag doubles a face by ldexp.
// The arithmetic after the no-flux doubling has rd_rhs_core's results, and
// doubling is exact, so the results are those of rd_step2_kernel bit for bit.
//
// LDS: s_uu holds the encoded step-0 state on [-2,10)^3 and, in the second
// half of each 24-value row, the encoded step-1 state on [-1,9)^3; rows of 24
// and planes of 293 values make the 8x8 lane patterns of a wave conflict-free
// for the block interior.  s_dmx/y/z[c] = D+x(c-x), D+y(c-y), D+z(c-z): the
// minus face coefficients of every cell evaluated in step 1.
// ---------------------------------------------------------------------------
__device__ inline int UU(int x, int y, int z) { return (x + 2) + 24 * (y + 2) + 293 * (z + 2); }  // [-2,10)^3
constexpr int UU1 = 12;  // offset of the step-1 state in a row
constexpr int UU_SIZE = 3516;
__device__ inline int DMI(int x, int y, int z) { return (x + 1) + 10 * (y + 1) + 100 * (z + 1); }  // [-1,9)^3

__device__ inline uint32_t sign_of(float v) { return __builtin_bit_cast(uint32_t, v) >> 31; }
__device__ inline uint32_t sign_of(double v) { return (uint32_t)(__builtin_bit_cast(uint64_t, v) >> 63); }
__device__ inline float twice_if(float d, uint32_t o) { return __builtin_amdgcn_ldexpf(d, (int)o); }
__device__ inline double twice_if(double d, uint32_t o) { return __builtin_amdgcn_ldexp(d, (int)o); }
// value with the outside flag in its sign bit (value >= +0)
template <typename Real>
__device__ inline Real flag_in_sign(Real u, Real tau) { return u < tau ? -u : u; }

// rd_rhs_core where 1/h^2 is a power of two: the scalings of both fluxes are
// exact, so ih2*in - ih2*out = ih2*(in - out), and the sum with the reaction is
// one fused multiply-add of an exact product.  The same bits.
template <typename Real>
__device__ inline Real rd_rhs_pow2(Real d0, Real d1, Real d2, Real d3, Real d4, Real d5, Real p0, Real p1, Real p2,
                                   Real p3, Real p4, Real p5, Real pc, bool dom, Real rho, double ih2) {
    Real sin_ = d0 * p0;
    sin_ = sin_ + d1 * p1;
    sin_ = sin_ + d2 * p2;
    sin_ = sin_ + d3 * p3;
    sin_ = sin_ + d4 * p4;
    sin_ = sin_ + d5 * p5;
    Real sdf = d0 + d1;
    sdf = sdf + d2;
    sdf = sdf + d3;
    sdf = sdf + d4;
    sdf = sdf + d5;
    const Real sdp = sdf * pc;
    const Real rp = rho * pc;
    const double react = (double)rp * (1. - (double)pc);
    const Real dphidt = (Real)__builtin_fma((double)sin_ - (double)sdp, ih2, react);
    return dom ? dphidt : (Real)0.;
}

// The state after one step from encoded neighbours e0..e5 (-x,+x,-y,+y,-z,+z)
// and the face coefficients d0..d5 before the no-flux rule.  DOM = false (every
// cell has p_w + p_g != 0 or p_w = p_g = 0): a cell out of the domain has six
// zero face coefficients and the state 0, so its dphidt comes out +0 without the
// test.  POW2: rd_rhs_pow2.
template <bool DOM, bool POW2, typename Real>
__device__ inline Real rd_step_enc(Real d0, Real d1, Real d2, Real d3, Real d4, Real d5, Real e0, Real e1, Real e2,
                                   Real e3, Real e4, Real e5, Real pc, bool inside, Real rho, double ih2, double dt) {
    d1 = twice_if(d1, sign_of(e0));
    d0 = twice_if(d0, sign_of(e1));
    d3 = twice_if(d3, sign_of(e2));
    d2 = twice_if(d2, sign_of(e3));
    d5 = twice_if(d5, sign_of(e4));
    d4 = twice_if(d4, sign_of(e5));
    const bool dom = !DOM || inside || pc > (Real)0.;
    const Real p0 = std::fabs(e0), p1 = std::fabs(e1), p2 = std::fabs(e2), p3 = std::fabs(e3), p4 = std::fabs(e4),
               p5 = std::fabs(e5);
    return rd_update(pc,
                     POW2 ? rd_rhs_pow2<Real>(d0, d1, d2, d3, d4, d5, p0, p1, p2, p3, p4, p5, pc, dom, rho, ih2)
                          : rd_rhs_core<Real>(d0, d1, d2, d3, d4, d5, p0, p1, p2, p3, p4, p5, pc, dom, rho, ih2),
                     dt);
}

// Blocks without diffusion.  When every face coefficient a block's cells use
// is +0 -- no tissue in the block, p_w*Dw + p_g*Dg == 0 in every cell, makes
// each harmonic mean with such a cell +0 -- the operator's flux sums are exact
// zeros: sum df_i*phi_i = +0, fin = ih2*(+0) = +0, fout = -(+0*ih2) = -0 and
// fout + fin = +0 (ReactionDiffusionOperator.h:125-135), so dphidt reduces to
// (Real)(+0 + reaction) in the domain and 0 outside it.
//
// The per-solve constants of a uniform grid, one workgroup per block, one pass
// over p_w and p_g (three kernels read each other's 16 B records before: 24
// samples of 96^3 540 -> 205 us): the records {D+, tau} and sigma, the records
// of rd_step2f_kernel, and
//   zflux[s]: 0 a block with diffusion, 1 without -- the plus-face coefficients
//     of its 512 cells and the minus-face ones across its -x, -y, -z faces are
//     all +0 --, 2 without and with no cell that is in the domain at phi = 0
//     (p_w + p_g = 0 in every cell): still_kernel;
//   flags[0] |= 1: a cell with p_w + p_g < 0; flags[1] |= 1: a cell cancels.
// Src gives a slot's anatomy (cells of slot q at [(q - slot0) * 512, ...)), its
// Dw and Dg and its position.
template <typename Real, typename Src>
__global__ __launch_bounds__(512) void constants_kernel(Src src, Stat4<Real>* __restrict__ st, Real* __restrict__ sig,
                                                        Stat4<Real>* __restrict__ stf,
                                                        unsigned char* __restrict__ zflux,
                                                        unsigned int* __restrict__ flags) {
    __shared__ Real s_df[1000];
    __shared__ unsigned int s_bits;
    const int s = blockIdx.x, t = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int u = t & 7, v = (t >> 3) & 7;
    const Real *pw, *pg;
    Real Dw, Dg;
    src.anatomy(s, pw, pg, Dw, Dg);
    const BlockPos bp = src.pos(s);
    const size_t base = (size_t)(s - bp.slot0) * BCELLS;
    if (t == 0) s_bits = 0;
    Real dh = 0;
    int in = 0;  // the cell next to the halo cell
    if (w < 6) {
        const int l0 = w & 1 ? 0 : 7, l1 = 7 - l0, o = w & 1 ? 8 : -1;
        const unsigned l = (unsigned)(w < 2 ? l0 + 8 * u + 64 * v : (w < 4 ? u + 8 * l0 + 64 * v : u + 8 * v + 64 * l0));
        const size_t c = (size_t)(face_nb(bp, w) - bp.slot0) * BCELLS + l;
        dh = diffusivity(pw[c], pg[c], Dw, Dg);
        s_df[w < 2 ? P(o, u, v) : (w < 4 ? P(u, o, v) : P(u, v, o))] = dh;
        in = w < 2 ? P(l1, u, v) : (w < 4 ? P(u, l1, v) : P(u, v, l1));
    }
    const Real pwc = pw[base + t], pgc = pg[base + t];
    const Real dc = diffusivity(pwc, pgc, Dw, Dg);
    const int q = P(u, v, w);
    s_df[q] = dc;
    __syncthreads();
    Stat4<Real> r;
    r.dx = harmonic(s_df[q + 1], dc);
    r.dy = harmonic(s_df[q + 10], dc);
    r.dz = harmonic(s_df[q + 100], dc);
    r.tau = chf_threshold(pwc, pgc);
    const Real sg = domain_threshold(pwc, pgc);
    auto not_zero = [](Real d) { return d != (Real)0 || sign_of(d) != 0; };
    bool nz = not_zero(r.dx) || not_zero(r.dy) || not_zero(r.dz);
    if (w < 6 && !(w & 1)) nz |= not_zero(harmonic(s_df[in], dh));
    const size_t g = (size_t)s * BCELLS + t;
    st[g] = r;
    sig[g] = sg;
    const Real tp = r.tau > (Real)0. ? r.tau : (Real)0.;
    r.tau = sg < (Real)0. ? -tp : tp;
    stf[g] = r;
    const unsigned int bits = (__any(nz) ? 1u : 0u) | (__any(sign_of(r.tau) != 0) ? 2u : 0u) |
                              (__any(!(sg <= (Real)0.)) ? 4u : 0u) | (__any(cancels(pwc, pgc)) ? 8u : 0u);
    if ((t & 63) == 0 && bits) atomicOr(&s_bits, bits);
    __syncthreads();
    if (t == 0) {
        zflux[s] = s_bits & 1u ? 0 : (s_bits & 2u ? 1 : 2);
        if (s_bits & 4u) atomicOr(flags, 1u);
        if (s_bits & 8u) atomicOr(flags + 1, 1u);
    }
}
// one solve: the fields of a context
template <typename Real>
struct UniformAnatomy {
    const Real* __restrict__ pw;
    const Real* __restrict__ pg;
    Real Dw, Dg;
    int bpd;
    uint32_t magic;
    __device__ inline void anatomy(int, const Real*& w, const Real*& g, Real& dw, Real& dg) const {
        w = pw;
        g = pg;
        dw = Dw;
        dg = Dg;
    }
    __device__ inline BlockPos pos(int s) const { return block_pos(s, 0, bpd, magic); }
};

// dphidt of a cell of a block without diffusion (see constants_kernel)
template <typename Real>
__device__ inline Real rd_rhs_reaction_only(Real pc, bool dom, Real rho) {
    const Real rp = rho * pc;
    const double react = (double)rp * (1. - (double)pc);
    const Real dphidt = (Real)(0.0 + react);
    return dom ? dphidt : (Real)0.;
}

// Work list of the two-step and the reverse-step kernels.  Blocks with
// diffusion are one item each (full: their items, ascending -- slots, or the
// int4 of packed solves; null: item i is slot i), runs of up to ZF_GROUP consecutive blocks without diffusion one item
// of grp {slot, blocks}.  Workgroup w runs on XCD w % 8 and takes item w / 8 of
// that XCD's contiguous share of full (fper items) -- neighbours' halos stay in
// one L2 -- and after these its share of grp (gper), which fill the tail.
// still (may be null) marks the grp items that need nothing (still_kernel).
struct StepWork {
    int nfull, fper, ngrp, gper;
    const int32_t* __restrict__ full;
    const int2* __restrict__ grp;
    const unsigned char* __restrict__ still;
    // this workgroup's item and its first slot, *nzf = 0 for a block with
    // diffusion, else the blocks without diffusion; -1: nothing to do
    template <typename Params>
    __device__ inline int item(const Params& prm, int* nzf, typename Params::Item& it) const {
        const int x = (int)(blockIdx.x % 8), j = (int)(blockIdx.x / 8);
        *nzf = 0;
        if (j < fper) {
            const int i = x * fper + j;
            if (i >= nfull) return -1;
            it = prm.item(full, i);
            return prm.slot(it);
        }
        const int i = x * gper + j - fper;
        if (i >= ngrp || (still && still[i])) return -1;
        const int2 v = grp[i];
        *nzf = v.y;
        it = prm.item_of(v.x);
        return v.x;
    }
    unsigned grid() const { return 8u * (unsigned)(fper + gper); }
};
constexpr int ZF_GROUP = 8;  // blocks without diffusion per workgroup
// the first nfull blocks and ngrp groups of a list
inline StepWork step_work(int nfull, const int32_t* full, int ngrp, const int2* grp, const unsigned char* still) {
    return StepWork{nfull, (nfull + 7) / 8, ngrp, (ngrp + 7) / 8, full, grp, still};
}

// One step, or dphidt, of any state.  BPW blocks per workgroup of 512 lanes; lane =
// cell (x fastest) of each block.  All loads of a lane -- wave w < 6 the halo of
// face w, one vector load of constants per cell -- are issued before the first
// wait.  A block without diffusion (zflux[s] != 0, constants_kernel) has +0 in
// every face coefficient: its records are not read, 16 of 28 B a cell.  Group
// mapping is XCD-aware: consecutive workgroups land on different XCDs, so
// workgroup w serves group (w % 8) * per_xcd + w / 8 and each XCD sweeps a
// contiguous range of blocks, whose halos -- and, from launch to launch, states --
// stay in its own L2.  (The work list of the two-step kernel, which deals the two
// kinds of blocks out evenly, gives an XCD other blocks' states than the kernels
// around it do: dphidt 15.1 us, and rd_update 7.4 instead of 5.1.)  dphidt of
// 128^3 FP32, 62 % of the blocks without diffusion: 13.7 -> 9.3 us; a step of 24
// samples of 96^3 148 -> 105 us.
template <typename Real, bool FUSED, int BPW, typename Params>
__global__ __launch_bounds__(512) void rd_step_kernel(int nslots, int per_xcd, const uint32_t* __restrict__ zflux,
                                                      const Real* __restrict__ phi, Real* __restrict__ out,
                                                      const Stat4<Real>* __restrict__ st,
                                                      const Real* __restrict__ sig, Params prm) {
    const int s0 = ((int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8)) * BPW;
    if (s0 >= nslots) return;
    __shared__ Real s_phi[BPW][1000];
    __shared__ unsigned char s_out[BPW][1000];
    __shared__ Real s_Dx[BPW][576], s_Dy[BPW][576], s_Dz[BPW][576];

    const int t = threadIdx.x;
    const int x = t & 7, y = (t >> 3) & 7, z = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t zf = zflux[s0 >> 2] >> (8 * (s0 & 3));  // a byte per block; BPW divides 4
    const int f = z;                                       // this wave's face
    const bool fx = f < 2, fz = f >= 4, plus = f & 1;
    const int lane = x + 8 * y;
    // cell (x, y) of the face in the neighbour block and in the tile
    const int src = fx ? (plus ? 0 : 7) + 8 * lane : (fz ? lane + (plus ? 0 : 448) : x + (plus ? 0 : 56) + 64 * y);
    const int dst = fx ? P(plus ? 8 : -1, x, y) : (fz ? P(x, y, plus ? 8 : -1) : P(x, plus ? 8 : -1, y));
    Real pc[BPW], sc[BPW], ph[BPW];
    Stat4<Real> sv[BPW], hs[BPW];
#pragma unroll
    for (int j = 0; j < BPW; ++j) {
        const int s = s0 + j;
        if (s >= nslots) break;
        const size_t nb = (size_t)(f < 6 ? face_nb(prm.pos(s), f) : s) * BCELLS, base = (size_t)s * BCELLS;
        ph[j] = (phi + nb)[src];
        pc[j] = (phi + base)[t];
        sc[j] = (sig + base)[t];
        hs[j] = sv[j] = Stat4<Real>{0, 0, 0, 0};
        if (!((zf >> (8 * j)) & 0xffu)) {
            hs[j] = (st + nb)[src];
            sv[j] = (st + base)[t];
        }
    }
#pragma unroll
    for (int j = 0; j < BPW; ++j) {
        if (s0 + j >= nslots) break;
        if (f < 6) {
            s_phi[j][dst] = ph[j];
            s_out[j][dst] = ph[j] < hs[j].tau;
            if (f == FXM) s_Dx[j][y * 72 + x * 9] = hs[j].dx;
            else if (f == FYM) s_Dy[j][y * 72 + x] = hs[j].dy;
            else if (f == FZM) s_Dz[j][y * 8 + x] = hs[j].dz;
        }
        s_phi[j][P(x, y, z)] = pc[j];
        s_out[j][P(x, y, z)] = pc[j] < sv[j].tau;
        s_Dx[j][z * 72 + y * 9 + x + 1] = sv[j].dx;
        s_Dy[j][z * 72 + (y + 1) * 8 + x] = sv[j].dy;
        s_Dz[j][(z + 1) * 64 + y * 8 + x] = sv[j].dz;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < BPW; ++j) {
        const int s = s0 + j;
        if (s >= nslots) break;
        Real rho;
        double ih2, dt;
        prm.get(s, rho, ih2, dt);
        const Real d = rd_cell_rhs<Real>(
            s_Dx[j][z * 72 + y * 9 + x], sv[j].dx, s_Dy[j][z * 72 + y * 8 + x], sv[j].dy,
            s_Dz[j][z * 64 + y * 8 + x], sv[j].dz, s_phi[j][P(x - 1, y, z)], s_phi[j][P(x + 1, y, z)],
            s_phi[j][P(x, y - 1, z)], s_phi[j][P(x, y + 1, z)], s_phi[j][P(x, y, z - 1)], s_phi[j][P(x, y, z + 1)],
            s_out[j][P(x - 1, y, z)], s_out[j][P(x + 1, y, z)], s_out[j][P(x, y - 1, z)],
            s_out[j][P(x, y + 1, z)], s_out[j][P(x, y, z - 1)], s_out[j][P(x, y, z + 1)], pc[j], sc[j], rho, ih2);
        out[(size_t)s * BCELLS + t] = FUSED ? rd_update(pc[j], d, dt) : d;
    }
}
// rd_step_kernel over slots [0, nslots); zflux: a byte per slot, padded to four
template <typename Real, bool FUSED, int BPW, typename Params>
void launch_step_kernel(hipStream_t stream, int nslots, const DevBuf& zflux, const Real* in, Real* out,
                        const Stat4<Real>* st, const Real* sig, const Params& prm) {
    static_assert(BPW == 1 || BPW == 2 || BPW == 4, "a workgroup's flags lie in one word");
    const int per_xcd = ((nslots + BPW - 1) / BPW + 7) / 8;
    hipLaunchKernelGGL((rd_step_kernel<Real, FUSED, BPW, Params>), dim3(8 * per_xcd), dim3(512), 0, stream, nslots,
                       per_xcd, zflux.as<uint32_t>(), in, out, st, sig, prm);
}

// Zero is a fixed point of a block without diffusion: the reaction of 0 is 0.
// A group whose blocks have no cell in the domain at 0 (zflux = 2) and whose
// state is +0 in every cell keeps it for the rest of the solve, and its adjoint
// keeps its value (adj_cell's factor is 1 out of the domain, its sums are
// zeros).  Marks these groups once per solve and writes the zeros of the other
// state buffer; the launches that follow leave them out, 24 B per cell and pair
// of steps of a brain's surroundings (62-77 % of the blocks of a uniform head
// grid).  FP32, us per launch before and after: pair of steps 128^3 11.96 /
// 6.98, 256^3 84.7 / 26.8; reverse step 128^3 23.8 / 7.8.
template <typename Real>
__global__ __launch_bounds__(256) void still_kernel(int ngrp, const int2* __restrict__ grp,
                                                    const unsigned char* __restrict__ zflux,
                                                    const Real* __restrict__ phi, Real* __restrict__ out,
                                                    unsigned char* __restrict__ still) {
    const int i = blockIdx.x;
    if (i >= ngrp) return;
    const int2 v = grp[i];
    const size_t c0 = (size_t)v.x * BCELLS;
    bool moves = zflux[v.x] != 2;  // a group's blocks have one flag
    if (!moves)
        for (int c = threadIdx.x; c < v.y * BCELLS; c += 256) {
            const Real u = phi[c0 + c];
            moves |= u != (Real)0 || sign_of(u) != 0;
        }
    moves = __syncthreads_or(moves);
    if (threadIdx.x == 0) still[i] = moves ? 0 : 1;
    if (!moves)
        for (int c = threadIdx.x; c < v.y * BCELLS; c += 256) out[c0 + c] = (Real)0;
}
// The zeros of the still groups in the n state buffers out + k * stride (a
// tape's states, which no later launch writes there), in the blocks that a block
// with diffusion reads: those next to one, by a face, an edge or a corner: a
// hull of 20 % of 128^3 instead of 62 %, 0.28 us a state at 5.8 TB/s.
constexpr int STILL_ZERO_STATES = 8;  // per workgroup, which looks at a group's neighbours once
template <typename Real, typename Params>
__global__ __launch_bounds__(256) void still_zero_kernel(int ngrp, const int2* __restrict__ grp,
                                                         const unsigned char* __restrict__ still,
                                                         const unsigned char* __restrict__ zflux, Params prm,
                                                         Real* __restrict__ out, size_t stride, int n) {
    const int i = blockIdx.x;
    if (i >= ngrp || !still[i]) return;
    const int2 v = grp[i];
    __shared__ unsigned s_next;
    const int t = threadIdx.x;
    if (t == 0) s_next = 0;
    __syncthreads();
    const int blk = t >> 5, k = t & 31;  // neighbour k of block blk (27 of them, itself among them)
    if (blk < v.y && k < 27) {
        const BlockPos bp = prm.pos(v.x + blk);
        if (zflux[bp.nb(k % 3 - 1, k / 3 % 3 - 1, k / 9 - 1)] == 0) atomicOr(&s_next, 1u << blk);
    }
    __syncthreads();
    const unsigned next = s_next;
    if (next == 0) return;
    const int k0 = blockIdx.y * STILL_ZERO_STATES, k1 = min(n, k0 + STILL_ZERO_STATES);
    for (int q = k0; q < k1; ++q)
        for (int c = t; c < v.y * BCELLS; c += 256)
            if ((next >> (c / BCELLS)) & 1) out[(size_t)q * stride + (size_t)v.x * BCELLS + c] = (Real)0;
}
template <typename Real, typename Params>
void launch_still_zero(hipStream_t stream, int ngrp, const DevBuf& grp, const DevBuf& still, const DevBuf& zflux,
                       const Params& prm, Real* out, size_t stride, int64_t n) {
    static_assert(ZF_GROUP * 32 <= 256, "a lane per neighbour of a group's blocks");
    constexpr int64_t PART = 32768 * STILL_ZERO_STATES;  // (gridDim.y limit)
    for (int64_t q = 0; ngrp > 0 && q < n; q += PART) {
        const int m = (int)std::min(PART, n - q);
        hipLaunchKernelGGL((still_zero_kernel<Real, Params>),
                           dim3((unsigned)ngrp, (unsigned)((m + STILL_ZERO_STATES - 1) / STILL_ZERO_STATES)), dim3(256),
                           0, stream, ngrp, grp.as<int2>(), still.as<unsigned char>(), zflux.as<unsigned char>(), prm,
                           out + (size_t)q * stride, stride, m);
    }
}
// the work list of slots [0, cut.back()) from their zflux flags; nfull / ngrp (may be
// null) receive the list lengths after each of the slot counts in cut
// (ascending), at which groups end
inline void build_step_work(const unsigned char* z, const std::vector<size_t>& cut, std::vector<int32_t>& full,
                            std::vector<int2>& grp, std::vector<int>* nfull, std::vector<int>* ngrp) {
    full.clear();
    grp.clear();
    int s = 0;
    for (size_t e : cut) {
        while (s < (int)e) {
            if (!z[s]) {
                full.push_back(s++);
                continue;
            }
            int k = 1;
            while (s + k < (int)e && z[s + k] == z[s] && k < ZF_GROUP) ++k;
            grp.push_back(make_int2(s, k));
            s += k;
        }
        if (nfull) nfull->push_back((int)full.size());
        if (ngrp) ngrp->push_back((int)grp.size());
    }
}

// Where cell (a, b) of face f at depth d (1 or 2) outside the block sits:
// LDS offsets uu (state tile) and dm (coefficient tile) and the cell index in
// the neighbour block across the face, each base + a * step_a + b * step_b
// with wave-uniform bases and steps.
struct FaceMap {
    int uu, uua, uub;
    int dm, dma, dmb;
    int lo, loa, lob;
};
__device__ inline FaceMap face_map(int f, int d) {  // f = 2 axis + (plus side), by selects: no branch for a uniform f
    const bool ax = f < 2, az = f >= 4;
    const int su = ax ? 1 : (az ? 293 : 24), sm = ax ? 1 : (az ? 100 : 10), sl = ax ? 1 : (az ? 64 : 8);
    const int out = f & 1 ? 7 + d : -d, in = f & 1 ? d - 1 : 8 - d;
    return {UU(0, 0, 0) + su * out, ax ? 24 : 1, az ? 24 : 293, DMI(0, 0, 0) + sm * out, ax ? 10 : 1, az ? 10 : 100,
            sl * in, ax ? 8 : 1, az ? 8 : 64};
}
__device__ inline int mad24(int a, int b, int c) { return (int)__umul24((unsigned)a, (unsigned)b) + c; }

// 512 lanes: wave w has the interior plane z = w and one of eight halo roles
// (faces 0-5, then the two halves of the edge cells).  With 256 lanes of two
// planes and two roles each, 14 % fewer vector instructions per block, a pair of
// steps takes as long at 256^3 (27.5 us) and longer at 128^3 (6.6 -> 7.3 us):
// the loads and barriers of a block bound it.  TWO = false: one step only (no
// edges, no depth-2 halo); FP32 with still groups left out, against
// rd_step_kernel, which runs every block: 128^3 (1,572 of 4,096 blocks move) 5.4
// and 11.8 us, 256^3 (11,635 of 32,768) 29.5 and 82.9, 24 samples of 96^3 29.6
// and 104.8.
template <typename Real, typename Params, bool DOM, bool TWO>
__global__ __launch_bounds__(512) void rd_step2f_kernel(
    int nfull, int fper, const int32_t* __restrict__ full, const Real* __restrict__ phi,
    const Stat4<Real>* __restrict__ stf, int bpd, uint32_t magic, const int4* __restrict__ slots,
    const void* __restrict__ range, Real* __restrict__ out, Real* __restrict__ mid, Real rho_, double ih2_, double dt_,
    int ngrp, int gper, const int2* __restrict__ grp, const unsigned char* __restrict__ still) {
    const StepWork wk{nfull, fper, ngrp, gper, full, grp, still};
    const Params prm = Params::make(rho_, ih2_, dt_, bpd, magic, slots, range);
    constexpr bool POW2 = Params::kPow2;
    int nzf;
    typename Params::Item it;
    const int s = wk.item(prm, &nzf, it);
    if (s < 0) return;
    __shared__ Real s_uu[UU_SIZE];
    __shared__ Real s_dmx[1000], s_dmy[1000], s_dmz[1000];

    const int t = threadIdx.x;
    const size_t base = (size_t)s * BCELLS;
    Real rho;
    double ih2, dt;
    prm.get(it, rho, ih2, dt);  // a group's blocks belong to one solve
    if (nzf > 0) {             // uniform per workgroup
        for (int i = t; i < nzf * BCELLS; i += 512) {
            const size_t bc = base + (unsigned)i;
            const Real u0 = phi[bc];
            const bool in0 = sign_of(stf[bc].tau) != 0;
            const Real u1 = rd_update(u0, rd_rhs_reaction_only(u0, in0 || u0 > (Real)0., rho), dt);
            if (TWO && mid) mid[bc] = u1;
            out[bc] = TWO ? rd_update(u1, rd_rhs_reaction_only(u1, in0 || u1 > (Real)0., rho), dt) : u1;
        }
        return;
    }
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);  // wave = interior plane z; halo role
    const int a = t & 7, b = (t >> 3) & 7;
    const BlockPos bp = prm.pos(it);
    const unsigned ut = (unsigned)t;

    // ---- loads: (waves 0-5) the depth-1 and depth-2 cells of face w, (waves
    // 6-7) the 96 edge cells next to the depth-1 faces, then the own cell; all
    // offsets are computed first so the loads issue back to back; block base
    // pointers are wave-uniform, lane offsets 32-bit
    Real u_1 = 0, u_2 = 0, u_e = 0;  // depth-1, depth-2 and edge cell: of their own, so that no load waits for another
    Stat4<Real> st_1, st_2, st_e;
    int uu1 = 0, dm1 = 0, uu2 = 0, dm2 = 0;
    int ex = 0, ey = 0, ez = 0;  // edge cell: tile coordinates
    bool edge = false;
    if (w < 6) {
        const FaceMap m1 = face_map(w, 1), m2 = face_map(w, 2);
        const size_t nb = (size_t)face_nb(bp, w) * BCELLS;
        const unsigned l1 = (unsigned)mad24(b, m1.lob, mad24(a, m1.loa, m1.lo)) & (BCELLS - 1);
        uu1 = mad24(b, m1.uub, mad24(a, m1.uua, m1.uu));
        dm1 = mad24(b, m1.dmb, mad24(a, m1.dma, m1.dm));
        u_1 = (phi + nb)[l1];
        st_1 = (stf + nb)[l1];
        if (TWO) {
            const unsigned l2 = (l1 + (unsigned)(m2.lo - m1.lo)) & (BCELLS - 1);
            uu2 = uu1 + (m2.uu - m1.uu);
            dm2 = dm1 + (m2.dm - m1.dm);
            u_2 = (phi + nb)[l2];
            st_2 = (stf + nb)[l2];
        }
    } else if (TWO) {
        const int e = (w - 6) * 64 + (t & 63);
        edge = e < 96;
        if (edge) {
            const int k = e >> 3, i = e & 7;
            const int pair = k >> 2, s1 = k & 1, s2 = (k >> 1) & 1;
            const int c1 = s1 ? 8 : -1, c2 = s2 ? 8 : -1;  // tile coordinate on the two crossed axes
            const int m1 = s1 ? 0 : 7, m2 = s2 ? 0 : 7;    // coordinate in the diagonal block
            const int d1 = s1 ? 1 : -1, d2 = s2 ? 1 : -1;
            int sl, lc;
            if (pair == 0) {
                ex = c1; ey = c2; ez = i; lc = m1 + 8 * m2 + 64 * i; sl = bp.nb(d1, d2, 0);
            } else if (pair == 1) {
                ex = c1; ey = i; ez = c2; lc = m1 + 8 * i + 64 * m2; sl = bp.nb(d1, 0, d2);
            } else {
                ex = i; ey = c1; ez = c2; lc = i + 8 * m1 + 64 * m2; sl = bp.nb(0, d1, d2);
            }
            const size_t gs = (size_t)sl * BCELLS + lc;
            u_e = phi[gs];
            st_e = stf[gs];
        }
    }
    const Real u_c = (phi + base)[ut];
    const Stat4<Real> st_c = (stf + base)[ut];

    // ---- LDS: encoded step-0 state, minus-face coefficients of the step-1 cells
    const int uuc = mad24(w, 293, mad24(b, 24, a + UU(0, 0, 0)));
    const int dmc = mad24(w, 100, mad24(b, 10, a + DMI(0, 0, 0)));
    const Real tau_c = std::fabs(st_c.tau);
    Real tau_1 = 0;
    s_uu[uuc] = flag_in_sign(u_c, tau_c);
    s_dmx[dmc + 1] = st_c.dx;
    s_dmy[dmc + 10] = st_c.dy;
    s_dmz[dmc + 100] = st_c.dz;
    if (w < 6) {
        tau_1 = std::fabs(st_1.tau);
        s_uu[uu1] = flag_in_sign(u_1, tau_1);
        // depth-1 cell: every component whose target stays in [-1,9)^3 (one
        // step: the minus faces of interior cells); depth-2 cell: only the
        // normal component of a minus face
        if (TWO ? w != FXP : w == FXM) s_dmx[dm1 + 1] = st_1.dx;
        if (TWO ? w != FYP : w == FYM) s_dmy[dm1 + 10] = st_1.dy;
        if (TWO ? w != FZP : w == FZM) s_dmz[dm1 + 100] = st_1.dz;
        if (TWO) {
            s_uu[uu2] = flag_in_sign(u_2, std::fabs(st_2.tau));
            if (w == FXM) s_dmx[dm2 + 1] = st_2.dx;
            if (w == FYM) s_dmy[dm2 + 10] = st_2.dy;
            if (w == FZM) s_dmz[dm2 + 100] = st_2.dz;
        }
    } else if (TWO && edge) {
        s_uu[UU(ex, ey, ez)] = flag_in_sign(u_e, std::fabs(st_e.tau));
        // an edge cell feeds the minus face of a depth-1 cell across each of
        // its crossed axes at -1
        if (ex == -1) s_dmx[DMI(0, ey, ez)] = st_e.dx;
        if (ey == -1) s_dmy[DMI(ex, 0, ez)] = st_e.dy;
        if (ez == -1) s_dmz[DMI(ex, ey, 0)] = st_e.dz;
    }
    __syncthreads();

    // ---- step 1 on the interior cell and (waves 0-5) the depth-1 face cell;
    // the step-1 half of a row (offsets 13..22) is disjoint from the step-0
    // half (offsets 0..11), so the writes race with no read
    auto step = [&](Real dmx, Real dmy, Real dmz, const Stat4<Real>& st, int q, Real u) {
        return rd_step_enc<DOM, POW2>(dmx, st.dx, dmy, st.dy, dmz, st.dz, s_uu[q - 1], s_uu[q + 1], s_uu[q - 24],
                                      s_uu[q + 24], s_uu[q - 293], s_uu[q + 293], u, sign_of(st.tau) != 0, rho, ih2,
                                      dt);
    };
    const Real dmx_c = s_dmx[dmc], dmy_c = s_dmy[dmc], dmz_c = s_dmz[dmc];
    const Real u1c = step(dmx_c, dmy_c, dmz_c, st_c, uuc, u_c);
    if constexpr (!TWO) {
        (out + base)[ut] = u1c;
    } else {
        s_uu[uuc + UU1] = flag_in_sign(u1c, tau_c);
        if (mid) (mid + base)[ut] = u1c;  // the state after the first step, when asked for
        if (w < 6)
            s_uu[uu1 + UU1] = flag_in_sign(step(s_dmx[dm1], s_dmy[dm1], s_dmz[dm1], st_1, uu1, u_1), tau_1);
        __syncthreads();
        // ---- step 2 on the interior cell
        (out + base)[ut] = step(dmx_c, dmy_c, dmz_c, st_c, uuc + UU1, u1c);
    }
}

// rd_step2f_kernel by the anatomy (plain: DOM = false) and the number of steps
template <typename Real, typename Params>
inline void launch_step2f_kernel(hipStream_t stream, const StepWork& wk, bool plain, bool two, const Real* in,
                                 Real* out, Real* mid, const Stat4<Real>* stf, const Params& prm) {
    const auto q = prm.args();
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(wk.grid()), dim3(512), 0, stream, wk.nfull, wk.fper, wk.full, in, stf, q.bpd,
                           q.magic, q.slots, q.range, out, mid, q.rho, q.ih2, q.dt, wk.ngrp, wk.gper, wk.grp,
                           wk.still);
    };
    if (two) {
        if (plain) go(rd_step2f_kernel<Real, Params, false, true>);
        else go(rd_step2f_kernel<Real, Params, true, true>);
    } else {
        if (plain) go(rd_step2f_kernel<Real, Params, false, false>);
        else go(rd_step2f_kernel<Real, Params, true, false>);
    }
}

}  // namespace gh
