// gh_lik_common.h -- per-voxel terms and host-side combination of the
// HGG likelihood (tools/pi4u_lite/Inference/Likelihood/source/
// HGG_Likelihood.cpp:40-192), shared by the single-solve and batched kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "gh_internal.h"
#include "gh_rd_common.h"

namespace gh {

struct LikParams {
    double s2, b, uc1, uc2, is2;
    int stepPET, stepTi;
    uint32_t petMagic;  // ceil(2^32 / stepPET), capped at 2^32 - 1
    uint32_t petBits;   // bit i: stepPET divides i, for i < 8
};

// log of the Bernoulli term at distance diff = u - uc of the threshold
__device__ inline double log_bernoulli(double diff, bool y, double is2) {
    const double omega2 = (diff > 0.) ? 1. : diff * diff;
    const int sg = (diff < -0.0) ? -1 : (diff > 0.0);
    const double alpha = 0.5 + 0.5 * (double)sg * (1. - exp(-omega2 * is2));
    return log(y ? alpha : 1. - alpha);
}

__device__ inline double wave_get(double v, int lane) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), lane);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

constexpr int LIK_THREADS = 256;
constexpr int LIK_GRID = 1024;  // fixed: the reduction order never changes

// cell index -> lattice coordinates for dense (x-fastest) or block-major
// uniform layouts
struct Layout {
    int nx, ny, nz;  // dense when bpd == 0
    int bpd;
    uint32_t magic;  // bpd_magic(bpd)
    __device__ inline void coords(size_t c, int& ix, int& iy, int& iz) const {
        if (bpd == 0) {
            ix = (int)(c % nx);
            iy = (int)((c / nx) % ny);
            iz = (int)(c / ((size_t)nx * ny));
        } else {
            const BlockPos q = block_pos((int)(c / BCELLS), 0, bpd, magic);
            const int l = (int)(c % BCELLS);
            ix = q.bx * BS + (l & 7);
            iy = q.by * BS + ((l >> 3) & 7);
            iz = q.bz * BS + (l >> 6);
        }
    }
};
inline Layout block_layout(int bpd) { return Layout{0, 0, 0, bpd, bpd_magic(bpd)}; }

// bit i: coordinate base + i is on the PET lattice, for i < 8 and base <= 504
// (base / stepPET is exact there, and base - 1 for stepPET = 1)
__device__ inline uint32_t pet_row(const LikParams& p, int base) {
    const uint32_t r = (uint32_t)base - __umulhi((uint32_t)base, p.petMagic) * (uint32_t)p.stepPET;
    const uint32_t first = r ? (uint32_t)p.stepPET - r : 0;
    return first < 8 ? (p.petBits << first) & 0xffu : 0;
}

// Cells of a wave whose Bernoulli term is one of four constants: u lost in u - uc
// (in front of a tumour) or u above the threshold, with either label.  The constants
// come from the function that makes the other terms, once per workgroup.
struct BernoulliCount {
    int front = 0, front1 = 0, above = 0, above1 = 0;
    // counts the wave's cells and returns the others, whose terms take an exp and a
    // log; every lane takes part, `in`: it has a cell
    __device__ inline uint64_t rest(bool in, double u, bool y, double uc) {
        const double diff = u - uc;
        const uint64_t all = __ballot(in), one = __ballot(y);
        const uint64_t a = __ballot(diff > 0.) & all, f = __ballot(diff == 0. - uc) & all & ~a;
        above += __popcll(a);
        above1 += __popcll(a & one);
        front += __popcll(f);
        front1 += __popcll(f & one);
        return all & ~(a | f);
    }
};

// Cells of lane `tid` of workgroup `wg` from `base` on, K of them, LIK_GRID
// workgroups' cells apart, with every load before the first use.  The workgroup's
// place among them moves from one to the next, so that none is at the tumour all
// the time.
template <int K, bool BLOCKS, typename T>
__device__ inline void lik_cells(int wg, size_t base, size_t ncells, const Layout& lay, const T* __restrict__ u,
                                 const unsigned char* __restrict__ t1, const unsigned char* __restrict__ fl,
                                 const double* __restrict__ pet, bool bern, const LikParams& p, BernoulliCount& b1,
                                 BernoulliCount& b2, double& sse, double& npet, double& l1, double& l2) {
    constexpr size_t stride = (size_t)LIK_GRID * LIK_THREADS;
    const int tid = threadIdx.x;
    T uv[K];
    double pv[K];
    unsigned char y1[K], y2[K];
    bool in[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int turn = (int)(base / stride) + k;
        const size_t c0 = base + k * stride + (size_t)((wg + 389 * turn) & (LIK_GRID - 1)) * LIK_THREADS, c = c0 + tid;
        uv[k] = 0;
        pv[k] = 0.;
        y1[k] = y2[k] = 0;
        in[k] = BLOCKS ? c0 < ncells : c < ncells;  // (blocks of 512: all of a workgroup's cells or none)
        if (in[k]) {
            uv[k] = u[c];
            y1[k] = t1[c];
            y2[k] = fl[c];
            if (BLOCKS) {  // a wave's 64 cells are a z plane of one block
                const int w = __builtin_amdgcn_readfirstlane((int)(c / 64)), l = tid & 63;
                const BlockPos q = block_pos(w >> 3, 0, lay.bpd, lay.magic);
                if ((pet_row(p, q.bz * BS) >> (w & 7)) & 1) {
                    const uint32_t mx = pet_row(p, q.bx * BS), my = pet_row(p, q.by * BS);
                    if ((mx >> (l & 7)) & (my >> (l >> 3)) & 1) pv[k] = pet[c];
                }
            } else {
                int ix, iy, iz;
                lay.coords(c, ix, iy, iz);
                if ((ix % p.stepPET == 0) && (iy % p.stepPET == 0) && (iz % p.stepPET == 0)) pv[k] = pet[c];
            }
        }
    }
    uint64_t any = 0;
    int y[K];  // bit 0, 1: this cell's terms are to be formed, bit 2, 3: its labels
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const double uc = (double)uv[k];
        if (pv[k] > 0.) {
            const double r = uc - p.b * pv[k];
            sse += r * r;
            npet += 1;
        }
        if (bern) {
            const uint64_t r1 = b1.rest(in[k], uc, y1[k] != 0, p.uc1), r2 = b2.rest(in[k], uc, y2[k] != 0, p.uc2);
            any |= r1 | r2;
            y[k] = (y1[k] != 0 ? 4 : 0) | (y2[k] != 0 ? 8 : 0) | ((r1 >> (tid & 63)) & 1) | (((r2 >> (tid & 63)) & 1) << 1);
        }
    }
    if (any == 0) return;
#pragma clang loop unroll(disable)  // unrolled, the exponentials and logarithms are 10 KB of code
    for (int k = 0; k < K; ++k) {
        const double uc = (double)uv[0];
        if (y[0] & 1) l1 += log_bernoulli(uc - p.uc1, y[0] & 4, p.is2);
        if (y[0] & 2) l2 += log_bernoulli(uc - p.uc2, y[0] & 8, p.is2);
#pragma unroll
        for (int i = 0; i + 1 < K; ++i) {
            uv[i] = uv[i + 1];
            y[i] = y[i + 1];
        }
    }
}

// stage 1: partials {sse, npet, L_T1, L_T2} of workgroup wg of LIK_GRID
// (LIK_THREADS lanes each), sum q at partials[q * LIK_GRID + wg]; the fixed grid
// fixes the summation order.
//
// Two exponentials and two logarithms in FP64 per cell bound it, and one cell's
// loads after another's.  Now cells in front of a tumour and above a threshold are
// counted by ballots on the scalar side, the others' terms are formed where a wave
// has any, and a lane has four cells' loads in flight (eight do not help one state
// and cost 24 samples of 96^3 a quarter: lanes without a cell).  128^3 FP32, PET on
// every third cell, a quarter of the cells on the tumour's flank: 28 -> 15.8 us;
// 24 samples of 96^3 230 -> 164 us.
template <typename T>
__device__ inline void lik_partials_body(int wg, size_t ncells, const Layout& lay, const T* __restrict__ u,
                                         const unsigned char* __restrict__ t1, const unsigned char* __restrict__ fl,
                                         const double* __restrict__ pet, const int4* __restrict__ roi, int nroi,
                                         const LikParams& p, double* __restrict__ partials) {
    double sse = 0, npet = 0, l1 = 0, l2 = 0;
    const bool bern = roi == nullptr;
    BernoulliCount b1, b2;
    constexpr size_t stride = (size_t)LIK_GRID * LIK_THREADS;
    if (lay.bpd > 0) {
        for (size_t c = 0; c < ncells; c += 4 * stride)
            lik_cells<4, true, T>(wg, c, ncells, lay, u, t1, fl, pet, bern, p, b1, b2, sse, npet, l1, l2);
    } else {
        for (size_t c = 0; c < ncells; c += stride)
            lik_cells<1, false, T>(wg, c, ncells, lay, u, t1, fl, pet, bern, p, b1, b2, sse, npet, l1, l2);
    }
    if (!bern) {
        for (size_t i = (size_t)wg * LIK_THREADS + threadIdx.x; i < (size_t)nroi; i += stride) {
            const int4 q = roi[i];  // {cell, ix, iy, iz}
            if ((q.y % p.stepTi == 0) && (q.z % p.stepTi == 0) && (q.w % p.stepTi == 0)) {
                const double uc = (double)u[q.x];
                l1 += log_bernoulli(uc - p.uc1, t1[q.x] != 0, p.is2);
                l2 += log_bernoulli(uc - p.uc2, fl[q.x] != 0, p.is2);
            }
        }
    }
    __shared__ double red[4][LIK_THREADS / 64];
    __shared__ int cnt[LIK_THREADS / 64][8];
    const int w = threadIdx.x / 64, lane = threadIdx.x % 64;
    const double a = wave_sum2(sse, npet), b = wave_sum2(l1, l2);
    if ((lane & 31) == 0) {
        red[lane >> 5][w] = a;
        red[2 + (lane >> 5)][w] = b;
    }
    if (lane == 0) {
        const int n[8] = {b1.front - b1.front1, b1.front1, b1.above - b1.above1, b1.above1,
                          b2.front - b2.front1, b2.front1, b2.above - b2.above1, b2.above1};
        for (int i = 0; i < 8; ++i) cnt[w][i] = n[i];
    }
    __syncthreads();
    if (w != 0) return;
    // lane l < 8: the counted terms of threshold l / 4, above it l & 2, label l & 1
    const int l = lane & 7;
    int n = 0;
    for (int k = 0; k < LIK_THREADS / 64; ++k) n += cnt[k][l];
    double v = log_bernoulli((l & 2) ? 1. : 0. - ((l & 4) ? p.uc2 : p.uc1), l & 1, p.is2);
    v = n ? (double)n * v : 0.;  // (a label that no cell has may have no finite term)
    v += __shfl_xor(v, 1, 64);
    v += __shfl_xor(v, 2, 64);  // lanes 0..3: the sum of threshold 0, 4..7: of threshold 1
    const double c1 = wave_get(v, 0), c2 = wave_get(v, 4);
    if (lane < 4) {
        double s = lane < 2 ? 0. : (lane == 2 ? c1 : c2);
        for (int k = 0; k < LIK_THREADS / 64; ++k) s += red[lane][k];
        partials[lane * LIK_GRID + wg] = s;
    }
}

// stage 2: one workgroup of 256 lanes, a wave to a sum, adds the partials in a
// fixed order: every 256th, then halves onto halves
__device__ inline void lik_final_body(const double* __restrict__ partials, double* __restrict__ out) {
    const int q = threadIdx.x / 64, lane = threadIdx.x % 64;
    double v[LIK_GRID / 64];
#pragma unroll
    for (int i = 0; i < LIK_GRID / 64; ++i) v[i] = partials[q * LIK_GRID + 64 * i + lane];
    double s[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        s[m] = 0;
#pragma unroll
        for (int i = m; i < LIK_GRID / 64; i += 4) s[m] += v[i];
    }
    double t = (s[0] + s[2]) + (s[1] + s[3]);
    for (int w = 32; w > 0; w >>= 1) t += __shfl_down(t, w, 64);
    if (lane == 0) out[q] = t;
}

// d/du of log(alpha) (y == 1) or log(1 - alpha): 0 for u >= uc (alpha is
// constant above uc and flat at uc), alpha = e/2 with e = exp(-(u-uc)^2/slope) below
__device__ inline double dlog_bernoulli(double u, bool y, double uc, double is2) {
    const double diff = u - uc;
    if (!(diff < 0.)) return 0.;
    const double a = 0.5 * exp(-diff * diff * is2);
    const double da = a * (-2. * diff * is2);
    return y ? da / a : -da / (1. - a);
}

// g = dJ/du of J = -logL at cell c: PET lattice term and (without ROI) the Bernoulli terms
template <typename T>
__device__ inline void lik_seed_cell(size_t c, const Layout& lay, const T* __restrict__ u,
                                     const unsigned char* __restrict__ t1, const unsigned char* __restrict__ fl,
                                     const double* __restrict__ pet, const LikParams& p, int full_bern,
                                     double* __restrict__ g) {
    int ix, iy, iz;
    lay.coords(c, ix, iy, iz);
    const double uc = (double)u[c];
    double v = 0;
    if ((ix % p.stepPET == 0) && (iy % p.stepPET == 0) && (iz % p.stepPET == 0) && pet[c] > 0.)
        v += (uc - p.b * pet[c]) / p.s2;
    if (full_bern) v -= dlog_bernoulli(uc, t1[c] != 0, p.uc1, p.is2) + dlog_bernoulli(uc, fl[c] != 0, p.uc2, p.is2);
    g[c] = v;
}

template <typename T>
__global__ __launch_bounds__(256) void lik_seed_kernel(size_t ncells, Layout lay, const T* __restrict__ u,
                                                       const unsigned char* __restrict__ t1,
                                                       const unsigned char* __restrict__ fl,
                                                       const double* __restrict__ pet, LikParams p, int full_bern,
                                                       double* __restrict__ g) {
    const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncells) return;
    lik_seed_cell<T>(c, lay, u, t1, fl, pet, p, full_bern, g);
}

// Bernoulli terms at ROI points on the stepMRI lattice (a point listed twice counts twice)
template <typename T>
__global__ __launch_bounds__(256) void lik_seed_roi_kernel(int nroi, const int4* __restrict__ roi,
                                                           const T* __restrict__ u,
                                                           const unsigned char* __restrict__ t1,
                                                           const unsigned char* __restrict__ fl, LikParams p,
                                                           double* __restrict__ g) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nroi) return;
    const int4 q = roi[i];
    if ((q.y % p.stepTi != 0) || (q.z % p.stepTi != 0) || (q.w % p.stepTi != 0)) return;
    const double uc = (double)u[q.x];
    atomicAdd(&g[q.x], -(dlog_bernoulli(uc, t1[q.x] != 0, p.uc1, p.is2) +
                         dlog_bernoulli(uc, fl[q.x] != 0, p.uc2, p.is2)));
}

inline int check_params(const double* params, int stepPET, int stepTi, LikParams& p) {
    if (!params) return set_error(GH_EINVAL, "likelihood: params is NULL");
    if (stepPET < 1 || stepTi < 1) return set_error(GH_EINVAL, "likelihood: steps must be >= 1");
    if (!(params[0] > 0) || !(params[4] != 0)) return set_error(GH_EINVAL, "likelihood: PETsigma2 > 0 and slope != 0");
    p.s2 = params[0];
    p.b = params[1];
    p.uc1 = params[2];
    p.uc2 = params[3];
    p.is2 = 1. / params[4];
    p.stepPET = stepPET;
    p.stepTi = stepTi;
    p.petMagic = stepPET == 1 ? 0xffffffffu : (uint32_t)((0x100000000ull + (uint64_t)stepPET - 1) / (uint64_t)stepPET);
    p.petBits = 0;
    for (int i = 0; i < 8; ++i) p.petBits |= i % stepPET == 0 ? 1u << i : 0u;
    return GH_OK;
}

// combine on the host in long double, as HGG_Likelihood::run does
inline void finish(const double sums[4], const LikParams& p, double out[4], int64_t* npet) {
    const long double p1 = (long double)(-0.5 * (double)sums[1] * std::log(2. * M_PI * p.s2));
    const long double p2 = (long double)(-0.5 * (1. / p.s2)) * (long double)sums[0];
    const long double lpet = p1 + p2;
    const long double cost = lpet + (long double)sums[2] + (long double)sums[3];
    out[0] = (double)(-cost);
    out[1] = (double)lpet;
    out[2] = sums[2];
    out[3] = sums[3];
    if (npet) *npet = (int64_t)llround(sums[1]);
}

}  // namespace gh
