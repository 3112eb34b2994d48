// One steady pseudo-step on the device: local time step, SSP-RK3 stages with
// positivity projection and modal filter, FP64 residual norm.
//
//   k_dt_local     src/autoflowcfd/core/fr_solver/cfl.py:12-147 (primitives with the
//                  floors of src/autoflowcfd/core/fr_solver/state.py:76-97)
//   k_rk_stage     src/autoflowcfd/core/time_integration/base.py:250-335 (Shu-Osher
//                  stage), positivity.py:13-45, src/autoflowcfd/core/fr_solver/filter.py:29-43
//   k_sq_partial / k_sum_partials
//                  src/autoflowcfd/core/fr_solver/state.py:99-107 (RMS, FP64 accumulation,
//                  fixed summation order: deterministic)
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/afr.h"
#include "afr_meanflow.hpp"
#include "afr_physics.hpp"
#include "afr_step.hpp"

using namespace afr;

namespace afr_step {

constexpr int kThreads = 256;

// local time step of one solution point i of cell c (h = cbrt |vol[c]|)
template <typename real>
__device__ __forceinline__ real dt_point(const real* __restrict__ U, const StateOff& so, const real* __restrict__ mu_t,
                                         const real* __restrict__ det, const real* __restrict__ mfs, int64_t i,
                                         int64_t c, double h, double mu, int order, int nut_mode) {
    const double cfl = 0.1, fa = 1.0 / (2 * order + 1), fv = fa * fa;
    double u5[5];
    load_state(U, i, so, c, u5);
    const double rho = u5[0] > 1e-10 ? u5[0] : 1e-10;
    const double ir = 1.0 / rho;
    const double u = u5[1] * ir, v = u5[2] * ir, w = u5[3] * ir;
    const double ke = 0.5 * (u * u + v * v + w * w);
    double p = (u5[4] - rho * ke) * 0.4;
    p = p > 1.0 ? p : 1.0;
    double a2 = 1.4 * p / rho;
    a2 = a2 > 1e-10 ? a2 : 1e-10;
    double ws = sqrt(u * u + v * v + w * w) + sqrt(a2);
    ws = ws > 1e-10 ? ws : 1e-10;
    const double dta = cfl * fa * h / ws;
    // nut_mode: the eddy-viscosity array holds nu_t and mu_t = rho nu_t
    double me = mu + (mu_t ? (nut_mode ? rho * (double)mu_t[i] : (double)mu_t[i]) : 0.0);
    me = me > 1e-30 ? me : 1e-30;
    const double dtv = 0.25 * cfl * fv * rho * h * h / me;
    double den = (double)mfs[i] * ws;
    den = den > 1e-300 ? den : 1e-300;
    const double dtg = cfl * fabs((double)det[i]) / den;
    double d = dta < dtv ? dta : dtv;
    d = d < dtg ? d : dtg;
    return (real)d;
}

// any points per cell: one thread per point, grid-stride
template <typename real>
__global__ void __launch_bounds__(kThreads) k_dt_local(const real* __restrict__ U, StateOff so,
                                                       const real* __restrict__ mu_t,
                                                       const real* __restrict__ det, const real* __restrict__ mfs,
                                                       const real* __restrict__ vol, real* __restrict__ dt,
                                                       int64_t n_cells, int ns, double mu, int order, int nut_mode) {
    const int64_t n = n_cells * ns;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t c = i / ns;
        dt[i] = dt_point(U, so, mu_t, det, mfs, i, c, cbrt(fabs((double)vol[c])), mu, order, nut_mode);
    }
}

// NS points per cell: a workgroup takes CPB = 256 / NS consecutive cells at a time, one thread
// per point (a 32-bit division by the constant NS instead of a 64-bit one; no barrier, so the
// loads of successive passes overlap; the same values as k_dt_local)
template <int NS, typename real>
__global__ void __launch_bounds__(kThreads) k_dt_cells(const real* __restrict__ U, StateOff so,
                                                       const real* __restrict__ mu_t,
                                                       const real* __restrict__ det, const real* __restrict__ mfs,
                                                       const real* __restrict__ vol, real* __restrict__ dt,
                                                       int64_t n_cells, double mu, int order, int nut_mode) {
    constexpr int CPB = kThreads / NS;
    const int t = threadIdx.x;
    if (t >= CPB * NS) return;
    const int lc = t / NS;
    for (int64_t cb = (int64_t)blockIdx.x * CPB; cb < n_cells; cb += (int64_t)gridDim.x * CPB) {
        const int64_t c = cb + lc;
        if (c < n_cells) {
            const int64_t i = cb * NS + t;
            dt[i] = dt_point(U, so, mu_t, det, mfs, i, c, cbrt(fabs((double)vol[c])), mu, order, nut_mode);
        }
    }
}

// U_out = c0 U0 + c1 Ua + c2 dt R, then positivity (rho >= 1e-6, |u| <= 1e4,
// p >= p_floor) per solution point and the modal filter per cell.  Ua may alias U_out, U0 may
// alias U_out (the cells of a pass are read completely before any of them is written).  With a
// state offset the three states are offsets from the cell's reference: the stage combination is the
// same (c0 + c1 = 1), the positivity test sees the absolute state, a projected component is stored
// back as its offset, and the filter (which keeps constants) acts on the offset.
//
// A wavefront takes whole cells (lane = (cell, point): 8 cells at P1, 2 at P2, 1 at P3) and needs no
// barrier.  Values cross HBM in consecutive order; a lane holds its filter row in registers for the
// whole kernel (again when the wave passes from prisms to tets) and reads each point's five values
// from LDS at once.  Bound: HBM (5 values from 3 arrays and dt in, 5 out, per point).  1024 workgroups
// are what the device holds at once at P2; us at 512 / 1024 / 2048 / 4096 (filter rows loaded by more waves):
// 66.5k P2 prisms FP32 46 / 35 / 35 / 37, 304k P1 prisms 49 / 38 / 36 / 35, 24.6k P3 tets FP64 90 / 97 / 111 / 137.
// Measured, 66.5k P2 prisms FP32: 36.8 us, 58.6 with one thread per filtered value and the filter in LDS;
// 10.3k P2 tets FP64 15.6 us (25.4), P1 tets FP64 8.4 (11.8).
template <int NS> struct RK {
    static constexpr int LW = NS <= 8 ? 8 : (NS <= 32 ? 32 : 64), CPW = 64 / LW, WAVES = 4, PS = 8;
    static constexpr int NE = CPW * NS * 5, IT = (NE + 63) / 64;   // values of a pass, per lane
    static constexpr bool REG = NS <= 27;   // filter row in registers; P3: columns in LDS
    template <typename real> static constexpr int wpe() { return !REG ? 2 : (NS <= 8 ? (sizeof(real) == 4 ? 5 : 4) : (sizeof(real) == 4 ? 4 : 3)); }
};

template <int NS, typename real>
__global__ void __launch_bounds__((64 * RK<NS>::WAVES))
    __attribute__((amdgpu_waves_per_eu(RK<NS>::template wpe<real>())))
    k_rk_stage(const real* U0, const real* Ua, const real* __restrict__ R, const real* __restrict__ dt, real* U_out,
               StateOff so, const real* __restrict__ filt0, const real* __restrict__ filt1, int64_t n_cells,
               int64_t n_prism, double c0, double c1, double c2, double p_floor) {
    using L = RK<NS>;
    using v4 = typename afr_mean::V4<real>::type;
    constexpr int LW = L::LW, CPW = L::CPW, PS = L::PS;
    __shared__ __attribute__((aligned(16))) real s_w[L::WAVES][CPW * NS * PS];
    __shared__ real s_f[2][L::REG ? 1 : NS * NS];
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t0 = threadIdx.x & 63;
    if constexpr (!L::REG) {
        for (int q = threadIdx.x; q < NS * NS; q += 64 * L::WAVES) {
            s_f[0][q % NS * NS + q / NS] = filt0[q];
            s_f[1][q % NS * NS + q / NS] = filt1[q];
        }
        __syncthreads();
    }
#pragma unroll 1
    for (int ct = 0; ct < 2; ++ct) {
        const int64_t begin = ct == 0 ? 0 : n_prism, end = ct == 0 ? n_prism : n_cells;
        real f[L::REG ? NS : 1];
        if constexpr (L::REG) {
            const real* row = (ct == 0 ? filt0 : filt1) + (t0 % LW < NS ? t0 % LW : 0) * NS;
#pragma unroll
            for (int j = 0; j < NS; ++j) f[j] = row[j];
        }
        for (CellWalk cw((end - begin + CPW - 1) / CPW, L::WAVES, wid); cw.it < cw.hi; cw.it += cw.step) {
            const int t = afr_mean::lane_fresh(t0), h = t / LW, s = t % LW < NS ? t % LW : 0;
            real* const sx = s_w[wid];
            real* const sc = sx + h * NS * PS;
            const int64_t cb = begin + cw.it * CPW;
            const int nc = (int)(end - cb < CPW ? end - cb : CPW);
            const int64_t i0 = cb * NS;
            real x0[L::IT], xr[L::IT], xa[L::IT], xd[L::IT];
#pragma unroll
            for (int q = 0; q < L::IT; ++q) {
                const int o = t + q * 64;
                if (o < nc * NS * 5) {
                    x0[q] = U0[i0 * 5 + o];
                    xr[q] = R[i0 * 5 + o];
                    xd[q] = dt[i0 + o / 5];
                    xa[q] = c1 != 0.0 ? Ua[i0 * 5 + o] : real(0);
                }
            }
#pragma unroll
            for (int q = 0; q < L::IT; ++q) {
                const int o = t + q * 64;
                if (o < nc * NS * 5) {
                    double val = c0 * (double)x0[q] + c2 * (double)xd[q] * (double)xr[q];
                    if (c1 != 0.0) val += c1 * (double)xa[q];
                    sx[o / 5 * PS + o % 5] = (real)val;   // stage value in the storage precision
                }
            }
            afr_mean::wave_sync();
            const bool live = t % LW < NS && h < nc;
            if (live) {
                real* x = sc + s * PS;
                double off[5], qa[5];
                so.row(cb + h, off);
#pragma unroll
                for (int v = 0; v < 5; ++v) qa[v] = so.mode ? (double)x[v] + off[v] : (double)x[v];
                const bool low_rho = !(qa[0] > 1e-6);
                const double rho = low_rho ? 1e-6 : qa[0];
                const double mm = qa[1] * qa[1] + qa[2] * qa[2] + qa[3] * qa[3];
                if (low_rho || mm > 1e8 * rho * rho || 0.4 * (qa[4] - 0.5 * mm * recip(rho)) < p_floor) {
                    double vx = qa[1] / rho, vy = qa[2] / rho, vz = qa[3] / rho;
                    const double vm = sqrt(vx * vx + vy * vy + vz * vz);
                    const bool fast = vm > 1e4;
                    double m1 = qa[1], m2 = qa[2], m3 = qa[3];
                    if (fast) {
                        const double g = 1e4 / vm;
                        vx *= g; vy *= g; vz *= g;
                        m1 = rho * vx; m2 = rho * vy; m3 = rho * vz;
                    }
                    const double ke = 0.5 * rho * (vx * vx + vy * vy + vz * vz);
                    // a component the projection left alone stays as it was (exact); a projected one is
                    // stored as its (absolute) value less the offset
                    if (low_rho) x[0] = (real)(rho - off[0]);
                    if (fast) {
                        x[1] = (real)(m1 - off[1]);
                        x[2] = (real)(m2 - off[2]);
                        x[3] = (real)(m3 - off[3]);
                    }
                    if (0.4 * (qa[4] - ke) < p_floor) x[4] = (real)(p_floor / 0.4 + ke - off[4]);
                }
            }
            afr_mean::wave_sync();
            v4 acc = {0, 0, 0, 0};
            real acc4 = 0;
            auto add = [&](int j, real w) {
                const v4 y = afr_mean::ld4(sc + j * PS);
                const real z = sc[j * PS + 4];
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[v] += w * y[v];
                acc4 += w * z;
            };
            if constexpr (L::REG) {
#pragma unroll
                for (int j = 0; j < NS; ++j) {
                    add(j, f[j]);
                    if (j % 5 == 4) __builtin_amdgcn_sched_barrier(0);   // five points in flight: registers
                }
            } else {
#pragma unroll 4
                for (int j = 0; j < NS; ++j) add(j, s_f[ct][j * NS + s]);
            }
            // formed here: sunk into the branch below, the sums would keep all their operands alive
            real out[5] = {acc[0], acc[1], acc[2], acc[3], acc4};
#pragma unroll
            for (int v = 0; v < 5; ++v) asm volatile("" : "+v"(out[v]));
            afr_mean::wave_sync();
            if (live) {
#pragma unroll
                for (int v = 0; v < 5; ++v) sc[s * PS + v] = out[v];
            }
            afr_mean::wave_sync();
#pragma unroll
            for (int q = 0; q < L::IT; ++q) {
                const int o = t + q * 64;
                if (o < nc * NS * 5) U_out[i0 * 5 + o] = sx[o / 5 * PS + o % 5];
            }
            afr_mean::wave_sync();
        }
    }
}

// Partial sums of x^2 in FP64, one per workgroup, for a group of cases at once.  A case is the logical
// array x[a0, a0 + n0) followed by x[a1, a1 + n1) (the prism and the tet cells of one case of a
// batched mesh), summed by `parts` workgroups in the partition and order that one contiguous array of
// n0 + n1 values alone would have, so a case's norm has the same bits in any batch.  One launch pair
// per group instead of one per case: ten cases of 8k to 150k cells took 100 us in 20 launches of 5 us,
// 11 us now.
template <typename real>
__global__ void __launch_bounds__(kThreads) k_sq_partial(const real* __restrict__ x, NormGroup g, double* part) {
    __shared__ double s[kThreads];
    int c = 0;
    while (c + 1 < g.n && (int)blockIdx.x >= g.c[c + 1].first) ++c;
    const int64_t a0 = g.c[c].a0, n0 = g.c[c].n0, a1 = g.c[c].a1, n = n0 + g.c[c].n1;
    const int blk = (int)blockIdx.x - g.c[c].first, parts = g.c[c].parts;
    double acc = 0.0;
    for (int64_t i = (int64_t)blk * kThreads + threadIdx.x; i < n; i += (int64_t)parts * kThreads) {
        const double v = (double)x[i < n0 ? a0 + i : a1 + (i - n0)];
        acc += v * v;
    }
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int m = kThreads / 2; m > 0; m >>= 1) {
        if (threadIdx.x < m) s[threadIdx.x] += s[threadIdx.x + m];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

__global__ void __launch_bounds__(kThreads) k_sum_partials(const double* part, NormGroup g, double* out) {
    __shared__ double s[kThreads];
    const int c = blockIdx.x, first = g.c[c].first, parts = g.c[c].parts;
    const double n_total = g.c[c].n_total;
    double acc = 0.0;
    for (int i = threadIdx.x; i < parts; i += kThreads) acc += part[first + i];
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int m = kThreads / 2; m > 0; m >>= 1) {
        if (threadIdx.x < m) s[threadIdx.x] += s[threadIdx.x + m];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[c] = n_total > 0 ? sqrt(s[0] / n_total) : 0.0;
}

static int grid_for(int64_t n, int per) {
    int64_t b = (n + per - 1) / per;
    return (int)(b < 1 ? 1 : (b > 4096 ? 4096 : b));
}

template <typename real>
int launch_dt_local(const real* U, StateOff so, const real* mu_t, const real* det, const real* mfs,
                    const real* vol, real* dt, int64_t n_cells, int ns, double mu, int order, int nut_mode,
                    hipStream_t st) {
#define AFR_DT_CELLS(NSV)                                                                                    \
    hipLaunchKernelGGL((k_dt_cells<NSV, real>), dim3(grid_for(n_cells, kThreads / NSV)), dim3(kThreads), 0, st, U, \
                       so, mu_t, det, mfs, vol, dt, n_cells, mu, order, nut_mode)
    if (ns == 1)
        AFR_DT_CELLS(1);
    else if (ns == 8)
        AFR_DT_CELLS(8);
    else if (ns == 27)
        AFR_DT_CELLS(27);
    else if (ns == 64)
        AFR_DT_CELLS(64);
    else
        hipLaunchKernelGGL((k_dt_local<real>), dim3(grid_for(n_cells * ns, kThreads)), dim3(kThreads), 0, st, U,
                           so, mu_t, det, mfs, vol, dt, n_cells, ns, mu, order, nut_mode);
#undef AFR_DT_CELLS
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <typename real>
int launch_rk_stage(int ns, const real* U0, const real* Ua, const real* R, const real* dt, real* U_out,
                    StateOff so, const real* filt0, const real* filt1, int64_t n_cells, int64_t n_prism,
                    double c0, double c1, double c2, double p_floor, hipStream_t st) {
    auto go = [&](auto NS) {
        using L = RK<decltype(NS)::value>;
        const int64_t units = (n_prism + L::CPW - 1) / L::CPW + (n_cells - n_prism + L::CPW - 1) / L::CPW;
        hipLaunchKernelGGL((k_rk_stage<decltype(NS)::value, real>), dim3(walk_grid(units, L::WAVES, 1024)),
                           dim3(64 * L::WAVES), 0, st, U0, Ua, R, dt, U_out, so, filt0, filt1, n_cells, n_prism, c0, c1,
                           c2, p_floor);
    };
    using std::integral_constant;
    if (ns == 8) go(integral_constant<int, 8>());
    else if (ns == 27) go(integral_constant<int, 27>());
    else if (ns == 64) go(integral_constant<int, 64>());
    else return -1;
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <typename real>
__global__ void __launch_bounds__(kThreads) k_fill(real* __restrict__ x, int64_t n, double v) {
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads)
        x[i] = (real)v;
}

template <typename real>
int launch_fill(real* x, int64_t n, double v, hipStream_t st) {
    hipLaunchKernelGGL((k_fill<real>), dim3(grid_for(n, kThreads)), dim3(kThreads), 0, st, x, n, v);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template int launch_fill<float>(float*, int64_t, double, hipStream_t);
template int launch_fill<double>(double*, int64_t, double, hipStream_t);

// out[i] for every case of the list, as many cases per launch pair as the group and the partial sums hold
template <typename real>
int launch_norm_cases(const real* x, const NormCase* cases, int n, double* part, int n_part_max, double* out,
                      hipStream_t st) {
    for (int i = 0; i < n;) {
        NormGroup g;
        g.n = 0;
        int blocks = 0;
        for (; i + g.n < n && g.n < kNormGroup; ++g.n) {
            NormCase c = cases[i + g.n];
            c.parts = grid_for(c.n0 + c.n1, kThreads * 8);
            c.parts = c.parts < n_part_max ? c.parts : n_part_max;
            c.first = blocks;
            if (blocks + c.parts > n_part_max) break;
            blocks += c.parts;
            g.c[g.n] = c;
        }
        // the partial sums are reused group after group (stream order)
        hipLaunchKernelGGL((k_sq_partial<real>), dim3(blocks), dim3(kThreads), 0, st, x, g, part);
        if (hipGetLastError() != hipSuccess) return -1;
        hipLaunchKernelGGL(k_sum_partials, dim3(g.n), dim3(kThreads), 0, st, (const double*)part, g, out + i);
        if (hipGetLastError() != hipSuccess) return -1;
        i += g.n;
    }
    return 0;
}

template <typename real>
int launch_norm(const real* x, int64_t n, double n_total, double* part, int n_part_max, double* out, hipStream_t st) {
    const NormCase c = {0, n, 0, 0, n_total, 0, 0};
    return launch_norm_cases(x, &c, 1, part, n_part_max, out, st);
}

template int launch_dt_local<float>(const float*, StateOff, const float*, const float*, const float*, const float*,
                                    float*, int64_t, int, double, int, int, hipStream_t);
template int launch_dt_local<double>(const double*, StateOff, const double*, const double*, const double*,
                                     const double*, double*, int64_t, int, double, int, int, hipStream_t);
template int launch_rk_stage<float>(int, const float*, const float*, const float*, const float*, float*, StateOff,
                                    const float*, const float*, int64_t, int64_t, double, double, double, double,
                                    hipStream_t);
template int launch_rk_stage<double>(int, const double*, const double*, const double*, const double*, double*,
                                     StateOff, const double*, const double*, int64_t, int64_t, double, double, double,
                                     double, hipStream_t);
template int launch_norm_cases<float>(const float*, const NormCase*, int, double*, int, double*, hipStream_t);
template int launch_norm_cases<double>(const double*, const NormCase*, int, double*, int, double*, hipStream_t);
template int launch_norm<float>(const float*, int64_t, double, double*, int, double*, hipStream_t);
template int launch_norm<double>(const double*, int64_t, double, double*, int, double*, hipStream_t);

}  // namespace afr_step
