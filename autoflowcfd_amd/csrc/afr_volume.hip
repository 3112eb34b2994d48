// Volume terms of the mean-flow residual (gfx950).
//
//   k_visc_volume  U -> gradients of (u, v, w, T), viscous flux, its divergence, and the per-point
//                  pack of the interface kernel (gradients.py:23-90, flux_kernels.py:72-137,
//                  viscous_flux.py:113-302 under src/autoflowcfd/core/fr_operators, fr_residual)
//   k_inv_volume   U -> over-integrated inviscid divergence of the prisms, by the Kronecker factors
//                  of the collapsed prism basis (src/autoflowcfd/fr/collapsed_basis.py:197-230,
//                  src/autoflowcfd/core/fr_residual/inviscid.py:139-345):
//                      X = c2f_c dQ,  Qf = c2f_ab X,  F~ = adj_fine (F(Q_ref + Qf) - F(Q_ref)),
//                      Y = A_a F~_a + A_b F~_b,  W = B_c F~_c,  div = f2c_c Y + f2c_ab W + gcl F(Q_ref)
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/afr.h"
#include "afr_meanflow.hpp"
#include "afr_physics.hpp"
#include "afr_prism.hpp"

using namespace afr;

namespace afr_mean {

// acc += w x by components: a vector product would keep w splatted over four registers
template <typename V, typename real> __device__ __forceinline__ void fma4(V& acc, real w, V x) {
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q] += w * x[q];
}

// viscous flux of a point and its contravariant components g[m] = (momentum 3, energy); gr[n][f] = d f / dx_n
template <typename real, typename V, typename Q>
__device__ __forceinline__ void visc_flux(const V gr[3], const real* dq, real mt, const real* ad, real mu, real Pr, real Prt,
                                          Q qref, V g[3]) {
    const real mts = mu + mt;
    const real lam = real(-2.0 / 3.0) * mts * (gr[0][0] + gr[1][1] + gr[2][2]);
    const real cp = real(kGamma * kRair / (kGamma - 1.0));
    const real kc = mu * cp / Pr + mt * cp / Prt;
    real tau[3][3], e[3], vel[3];
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int q = 0; q < 3; ++q) tau[p][q] = mts * (gr[q][p] + gr[p][q]) + (p == q ? lam : real(0));
#pragma unroll
    for (int p = 0; p < 3; ++p) vel[p] = (real)(qref[1 + p] + (double)dq[1 + p]);
#pragma unroll
    for (int p = 0; p < 3; ++p) e[p] = vel[0] * tau[0][p] + vel[1] * tau[1][p] + vel[2] * tau[2][p] - kc * gr[p][3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
#pragma unroll
        for (int v = 0; v < 3; ++v) g[m][v] = ad[m * 3] * tau[0][v] + ad[m * 3 + 1] * tau[1][v] + ad[m * 3 + 2] * tau[2][v];
        g[m][3] = ad[m * 3] * e[0] + ad[m * 3 + 1] * e[1] + ad[m * 3 + 2] * e[2];
    }
}

// ------------------------------------------------------------------ viscous volume kernel
// Lanes of a wavefront: (cell, solution point), LW lanes per cell (P1: 8 cells of 8 lanes, P2: 2
// cells of 27 of 32 lanes).  A lane keeps the non-zeros of its derivative rows in registers for the
// whole kernel (d/da couples the N1 points of an a line, d/db the N1^2 of an (a, b) plane, d/dc the
// N1 of a c line for a prism and all points for a tet, whose d/dc rows stay in LDS), reads its
// neighbours' four fields with one 16-byte LDS load per non-zero at a fixed offset, and keeps its
// gradients, stress and metrics in registers from the gradient to the flux.
// Bound: HBM (reads U, mu_t, adj, det; writes the 16-value pack and the 4-value divergence: 4.5 GB at
// 82^3 P2 FP32, 830 us = 5.4 TB/s).  Before: 2080 us with gradients staged through LDS, an 18-of-20-value
// pack and a divided residual.  304k P1 prisms 57 us (285).
template <int P, int CT, typename real> struct VV {
    static constexpr int N1 = P + 1, NS = N1 * N1 * N1;
    static constexpr int LW = NS <= 8 ? 8 : 32, CPW = 64 / LW;
    static constexpr int KP = kPack + 4;    // LDS stride of a pack point (bank-conflict-free 16-byte access)
    static constexpr int PER = NS * 4 + NS * KP;
    static constexpr int WAVES = 4;
    static constexpr int DT = CT == 1 ? NS * (NS | 1) : 4;   // d/dc rows of a tet
};

template <int P, int CT, typename real>
__global__ void __launch_bounds__((64 * VV<P, CT, real>::WAVES)) k_visc_volume(MeanArgs<real> a) {
    using L = VV<P, CT, real>;
    using v4 = typename V4<real>::type;
    constexpr int N1 = L::N1, NS = L::NS, LW = L::LW, CPW = L::CPW, KP = L::KP, WAVES = L::WAVES;
    constexpr int RS = NS | 1;
    __shared__ __attribute__((aligned(16))) real s_w[WAVES][CPW * L::PER];
    __shared__ real s_dc[L::DT];
    const int tid = threadIdx.x, wid = __builtin_amdgcn_readfirstlane(tid >> 6), t = tid & 63;
    const int h = t / LW, s = t % LW;
    const bool on = s < NS;
    const int sp = on ? s : 0, i = sp / (N1 * N1), j = (sp / N1) % N1, k = sp % N1;
    if constexpr (CT == 1) {
        for (int q = tid; q < NS * NS; q += 64 * WAVES) s_dc[(q / NS) * RS + q % NS] = a.D[2 * NS * NS + q];
        __syncthreads();
    }
    real* const sF = s_w[wid] + h * L::PER;   // (du, dv, dw, dT) [s][4]
    real* const sP = sF + NS * 4;             // pack [s][KP], then G~ [m][s][4]
    real wa[N1], wb[N1 * N1], wc[N1];
#pragma unroll
    for (int q = 0; q < N1; ++q) {
        wa[q] = a.D[sp * NS + (q * N1 + j) * N1 + k];
        wc[q] = CT == 0 ? a.D[(2 * NS + sp) * NS + (i * N1 + j) * N1 + q] : real(0);
    }
#pragma unroll
    for (int q = 0; q < N1 * N1; ++q) wb[q] = a.D[(NS + sp) * NS + q * N1 + k];
    // sum_k row_m[k] x[k] over a field of 4 values per point
    auto apply = [&](int m, const real* x) -> v4 {
        v4 acc = {0, 0, 0, 0};
        if (m == 0) {
#pragma unroll
            for (int q = 0; q < N1; ++q) fma4(acc, wa[q], ld4(x + (q * N1 * N1 + j * N1 + k) * 4));
        } else if (m == 1) {
#pragma unroll
            for (int q = 0; q < N1 * N1; ++q) fma4(acc, wb[q], ld4(x + (q * N1 + k) * 4));
        } else if constexpr (CT == 0) {
#pragma unroll
            for (int q = 0; q < N1; ++q) fma4(acc, wc[q], ld4(x + ((i * N1 + j) * N1 + q) * 4));
        } else {
#pragma unroll
            for (int q = 0; q < NS; ++q) fma4(acc, s_dc[sp * RS + q], ld4(x + q * 4));
        }
        return acc;
    };
    const double T0 = a.qref[4] / (rmax(a.qref[0], 1e-10) * kRair);
    const int64_t n_units = (a.n_cells + CPW - 1) / CPW;
    for (CellWalk cw(n_units, WAVES, wid); cw.it < cw.hi; cw.it += cw.step) {
        const int64_t c0 = cw.it * CPW;
        const int nc = (int)(a.n_cells - c0 < CPW ? a.n_cells - c0 : CPW);
        const bool live = on && h < nc;
        const int64_t cell = a.cell_begin + c0 + (h < nc ? h : 0);
        const int64_t pt = cell * NS + sp;
        real ad[9], dq[5], mt = real(0), idet = real(0);
        if (live) {
#pragma unroll
            for (int q = 0; q < 9; ++q) ad[q] = a.adj[pt * 9 + q];
            idet = a.det[pt];
            if (a.mu_t) mt = a.mu_t[pt];
            double u[5], q[5];
            load_state(a.U, pt, a.so, cell, u);
            cons2prim(u, q);
#pragma unroll
            for (int v = 0; v < 5; ++v) dq[v] = (real)(q[v] - a.qref[v]);
            const double T = q[4] / (rmax(q[0], 1e-10) * kRair);
            st4(sF + s * 4, (v4){dq[1], dq[2], dq[3], (real)(T - T0)});
            if (a.dQ_out) {
#pragma unroll
                for (int v = 0; v < 5; ++v) {
                    a.dQ_out[pt * 5 + v] = dq[v];
                    sP[s * 5 + v] = (real)fabs(u[v]);
                }
            }
            idet = recip(idet);
        }
        wave_sync();
        if (a.dQ_out) {   // per-cell mean |U| (outlier reference) of callers that prepare the state
            if (h < nc && s < 5) {
                real acc = 0;
                for (int q = 0; q < NS; ++q) acc += sP[q * 5 + s];
                a.umean_out[cell * 5 + s] = acc / real(NS);
            }
            wave_sync();
        }
        v4 gr[3];   // gr[n][f] = d f / dx_n
        if (live) {
            const v4 d0 = apply(0, sF), d1 = apply(1, sF), d2 = apply(2, sF);
#pragma unroll
            for (int n = 0; n < 3; ++n) gr[n] = (ad[n] * d0 + ad[3 + n] * d1 + ad[6 + n] * d2) * idet;
            real* vp = sP + s * KP;
            st4(vp, (v4){dq[0], dq[1], dq[2], dq[3]});
            st4(vp + 4, (v4){dq[4], gr[0][0] + gr[0][0], gr[1][1] + gr[1][1], gr[2][2] + gr[2][2]});
            st4(vp + 8, (v4){gr[1][0] + gr[0][1], gr[2][0] + gr[0][2], gr[2][1] + gr[1][2], gr[0][3]});
            st4(vp + 12, (v4){gr[1][3], gr[2][3], mt, real(0)});
        }
        wave_sync();
        // the packs of the wave's cells, contiguous in HBM: whole-line stores
        {
            real* dst = a.pack + (a.cell_begin + c0) * NS * kPack;
            for (int o = t; o < nc * NS * 4; o += 64) {
                const int c = o / (NS * 4), r = o % (NS * 4);
                st4(dst + o * 4, ld4(s_w[wid] + c * L::PER + NS * 4 + (r >> 2) * KP + (r & 3) * 4));
            }
        }
        wave_sync();
        if (live) {
            v4 g[3];
            visc_flux(gr, dq, mt, ad, (real)a.mu, (real)a.Pr, (real)a.Prt, a.qref, g);
#pragma unroll
            for (int m = 0; m < 3; ++m) st4(sP + (m * NS + s) * 4, g[m]);
        }
        wave_sync();
        if (live) {
            const v4 r = apply(0, sP) + apply(1, sP + NS * 4) + apply(2, sP + 2 * NS * 4);
            st4(a.rvisc + pt * 4, r);
        }
        wave_sync();
    }
}

// ------------------------------------------------------------------ viscous volume kernel (P3 tets, FP64)
// Dense derivative rows (their round-off entries count): both contractions, D x fields and D x
// contravariant fluxes, on the matrix cores.  A workgroup takes 8 cells x 4 fields = 2 x 16 columns; wave
// w holds the fragments of rows 16 w .. 16 w + 15 of the three D for the whole kernel.  A quad of lanes
// ends the first product with four rows of the four fields of one cell: transposed within the quad, each
// lane has the gradients of one point, whose state and metrics it has held from the start.
// Measured: 24.6k cells 179 us, 590 with a lane per point reading its dense rows from global memory.
struct V3 {
    static constexpr int NS = 64, CPT = 8, CT = 2, LD = CPT * 4 + 2, KS = NS / 4;
};

// x of the lane at quad position (lane ^ M)
template <int M> __device__ __forceinline__ double quad_xor(double x) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), M == 1 ? 0xB1 : 0x4E, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), M == 1 ? 0xB1 : 0x4E, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
// within each quad of lanes: entry g of lane f becomes entry f of lane g (all lanes take part)
__device__ __forceinline__ d4 quad_transpose(d4 x, int lane) {
    const bool b0 = lane & 1, b1 = lane & 2;
    const double s0 = quad_xor<1>(b0 ? x[0] : x[1]), s1 = quad_xor<1>(b0 ? x[2] : x[3]);
    const d4 y = {b0 ? s0 : x[0], b0 ? x[1] : s0, b0 ? s1 : x[2], b0 ? x[3] : s1};
    const double t0 = quad_xor<2>(b1 ? y[0] : y[2]), t1 = quad_xor<2>(b1 ? y[1] : y[3]);
    return (d4){b1 ? t0 : y[0], b1 ? t1 : y[1], b1 ? y[2] : t0, b1 ? y[3] : t1};
}

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_visc_volume_p3(MeanArgs<double> a) {
    using L = V3;
    constexpr int NS = L::NS, CPT = L::CPT, CT = L::CT, LD = L::LD, KS = L::KS;
    __shared__ __attribute__((aligned(16))) double s_x[NS * LD];       // (du, dv, dw, dT) [s][cell, field]
    __shared__ __attribute__((aligned(16))) double s_g[3 * NS * LD];   // contravariant fluxes [m][s][cell, component]
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), t = tid & 63;
    const int ln = t % 16, lk = t / 16;
    const int s = 16 * w + 4 * (t % 4) + lk;             // this lane's point, of the cells ct * 4 + ln / 4
    double fd[3][KS];
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
        for (int k = 0; k < KS; ++k) fd[m][k] = a.D[(m * NS + 16 * w + ln) * NS + 4 * k + lk];
    const double T0 = a.qref[4] / (rmax(a.qref[0], 1e-10) * kRair);
    const int64_t n_tiles = (a.n_cells + CPT - 1) / CPT;
    for (CellWalk cw(n_tiles, 1, 0); cw.it < cw.hi; cw.it += cw.step) {
        const int64_t c0 = a.cell_begin + cw.it * CPT;
        const int nc = (int)(a.n_cells - cw.it * CPT < CPT ? a.n_cells - cw.it * CPT : CPT);
        double dq[CT][5];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const int c = ct * 4 + ln / 4;
            d4 f = {0, 0, 0, 0};
#pragma unroll
            for (int v = 0; v < 5; ++v) dq[ct][v] = 0.0;
            if (c < nc) {
                const int64_t pt = (c0 + c) * NS + s;
                double u[5], q[5];
                load_state(a.U, pt, a.so, c0 + c, u);
                cons2prim(u, q);
#pragma unroll
                for (int v = 0; v < 5; ++v) dq[ct][v] = q[v] - a.qref[v];
                f = (d4){dq[ct][1], dq[ct][2], dq[ct][3], q[4] / (rmax(q[0], 1e-10) * kRair) - T0};
                if (a.dQ_out) {
#pragma unroll
                    for (int v = 0; v < 5; ++v) {
                        a.dQ_out[pt * 5 + v] = dq[ct][v];
                        s_g[(c * NS + s) * 5 + v] = fabs(u[v]);
                    }
                }
            }
            st4(s_x + s * LD + c * 4, f);
        }
        __syncthreads();
        if (a.dQ_out) {   // per-cell mean |U| (outlier reference) of callers that prepare the state
            if (tid < nc * 5) {
                double acc = 0;
                for (int q = 0; q < NS; ++q) acc += s_g[(tid / 5 * NS + q) * 5 + tid % 5];
                a.umean_out[(c0 + tid / 5) * 5 + tid % 5] = acc / NS;
            }
            __syncthreads();
        }
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const int c = ct * 4 + ln / 4;
            const int64_t pt = (c0 + (c < nc ? c : 0)) * NS + s;
            double ad[9];
#pragma unroll
            for (int q = 0; q < 9; ++q) ad[q] = a.adj[pt * 9 + q];
            const double mt = a.mu_t ? a.mu_t[pt] : 0.0, idet = recip(a.det[pt]);
            d4 d[3] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
            for (int k = 0; k < KS; ++k) {
                const double x = s_x[(4 * k + lk) * LD + ct * 16 + ln];
#pragma unroll
                for (int m = 0; m < 3; ++m) d[m] = mma(fd[m][k], x, d[m]);
            }
#pragma unroll
            for (int m = 0; m < 3; ++m) d[m] = quad_transpose(d[m], t);
            d4 gr[3], g[3];
#pragma unroll
            for (int n = 0; n < 3; ++n) gr[n] = (ad[n] * d[0] + ad[3 + n] * d[1] + ad[6 + n] * d[2]) * idet;
            visc_flux(gr, dq[ct], mt, ad, a.mu, a.Pr, a.Prt, a.qref, g);
            if (c < nc) {
                double* vp = a.pack + pt * kPack;
                st4(vp, (d4){dq[ct][0], dq[ct][1], dq[ct][2], dq[ct][3]});
                st4(vp + 4, (d4){dq[ct][4], gr[0][0] + gr[0][0], gr[1][1] + gr[1][1], gr[2][2] + gr[2][2]});
                st4(vp + 8, (d4){gr[1][0] + gr[0][1], gr[2][0] + gr[0][2], gr[2][1] + gr[1][2], gr[0][3]});
                st4(vp + 12, (d4){gr[1][3], gr[2][3], mt, 0.0});
            }
#pragma unroll
            for (int m = 0; m < 3; ++m) st4(s_g + (m * NS + s) * LD + c * 4, g[m]);
        }
        __syncthreads();
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const int c = ct * 4 + ln / 4;
            d4 r[3] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};   // per direction, as the sums were
#pragma unroll
            for (int k = 0; k < KS; ++k)
#pragma unroll
                for (int m = 0; m < 3; ++m) r[m] = mma(fd[m][k], s_g[(m * NS + 4 * k + lk) * LD + ct * 16 + ln], r[m]);
            const d4 sum = quad_transpose(r[0] + r[1] + r[2], t);
            if (c < nc) st4(a.rvisc + ((c0 + c) * NS + s) * 4, sum);
        }
        __syncthreads();
    }
}

template <int P, int CT, typename real>
int launch_visc_volume(const MeanArgs<real>& a, hipStream_t st) {
    if (a.n_cells <= 0) return 0;
    const int cap = a.grid_cap > 0 ? a.grid_cap : 8192;
    if constexpr (P == 3) {
        hipLaunchKernelGGL(k_visc_volume_p3, dim3(walk_grid((a.n_cells + V3::CPT - 1) / V3::CPT, 1, cap)), dim3(256), 0, st, a);
    } else {
        using L = VV<P, CT, real>;
        const int grid = walk_grid((a.n_cells + L::CPW - 1) / L::CPW, L::WAVES, cap);
        hipLaunchKernelGGL((k_visc_volume<P, CT, real>), dim3(grid), dim3(64 * L::WAVES), 0, st, a);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// the state offset out of the kernel arguments, field by field (scalar loads where it is used)
__device__ __forceinline__ StateOff state_off(const __attribute__((address_space(4))) StateOff& x) {
    StateOff so;
    so.table = x.table;
    so.cell_case = x.cell_case;
#pragma unroll
    for (int v = 0; v < 5; ++v) so.one[v] = x.one[v];
    so.mode = x.mode;
    so.sorted = x.sorted;
    so.split = x.split;
    return so;
}

// ------------------------------------------------------------------ inviscid volume kernel (prisms)
// A workgroup of N1 wavefronts takes CPT cells at a time (P2: 3 waves, 3 cells; P1: 2 waves, 4
// cells).  In every contraction the wave index is the output row group, so the operator entries are
// the same for all lanes of a wave and come from scalar loads; the lanes are (cell, fine line
// coordinate, variable), 60 of 64, and hold their inputs in registers.  LDS carries only the data
// from stage to stage; the row stride of F~ and W is padded so that 16-byte reads of successive
// rows fall on different banks.
// Bound: waits (59% of the wave cycles: barriers between the stages, scalar loads of the operators);
// VALU issue takes 0.86 ms of it, HBM 3.5 GB.  Measured (82^3 P2 FP32): 1.21 ms; with the arguments held
// in registers over the tile loop 1.48 ms.  Before, jumps included: 2.98 ms (one wave per cell, LDS
// operator tables).  304k P1 prisms 143 us (1014 with jumps).
template <int P, typename real> struct IV {
    using K = afr_prism::PK<P>;
    static constexpr int N1 = K::N1, NAB = K::NAB, NF1 = K::NF1, NABF = K::NABF, NF = K::NF, NS = K::NS;
    static constexpr int NW = N1, CPT = 64 / (NF1 * 5);
    static constexpr int QB = (NABF + 3) / 4, RS = QB * 4 + (QB % 2 == 0 ? 4 : 0);
    static constexpr int CPWV = CPT / NW;                       // cells per wave at the fine points
    static constexpr int OQ = 0, OX = OQ + NAB * 20, OF = OX + NAB * 20;   // q, X [ab][v][4], Qf [f][5]
    static constexpr int OW = 0, OY = OW + N1 * 5 * RS;         // W [c][v][RS], Y [ab][v][4] (over q, X, Qf)
    static constexpr int N0 = (OF + NF * 5 > OY + NAB * 20 ? OF + NF * 5 : OY + NAB * 20);
    static constexpr int OT = (N0 + 3) / 4 * 4;                 // F~ [m][cf][v][RS]
    static constexpr int PER = OT + 3 * NF1 * 5 * RS;
    static constexpr int WPE = sizeof(real) == 4 ? (P == 1 ? 5 : 6) : 3;
    static_assert(CPT % NW == 0 && CPWV * NF <= 64 && QB == NF1 && NAB == NW * N1, "lane maps");
};

template <int P, typename real>
__global__ void __launch_bounds__((64 * IV<P, real>::NW))
    __attribute__((amdgpu_waves_per_eu(IV<P, real>::WPE))) k_inv_volume(MeanArgs<real> args) {
    using L = IV<P, real>;
    using K = typename L::K;
    using v4 = typename V4<real>::type;
    using uni = typename Uni<real>::type;
    constexpr int N1 = L::N1, NAB = L::NAB, NF1 = L::NF1, NABF = L::NABF, NF = L::NF, NS = L::NS;
    constexpr int CPT = L::CPT, NW = L::NW, RS = L::RS, QB = L::QB, PER = L::PER, CPWV = L::CPWV;
    __shared__ __attribute__((aligned(16))) real s_w[CPT * PER];
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), t = tid & 63;
    // the arguments and the operator table are read anew in every stage (scalar loads): held over the
    // tile loop they would be spilled to vector lanes
    typedef const __attribute__((address_space(4))) MeanArgs<real> Args;
    Args* const kernarg = (Args*)__builtin_amdgcn_kernarg_segment_ptr();
    auto fresh = [&]() -> Args* {
        Args* p = kernarg;
        asm volatile("" : "+s"(p));
        return p;
    };
    if constexpr (NABF % 4 != 0) {   // the padding of the F~ rows is read (times zero) and never written
        for (int q = tid; q < CPT * PER; q += 64 * NW) s_w[q] = real(0);
        __syncthreads();
    }
    // fine point of this lane: cell fc of the tile, point ff
    const int fc = w * CPWV + t / NF, ff = t % NF;
    const bool fon = t < CPWV * NF;
    // contraction lanes: (cell lc, line coordinate cf, variable lv)
    const int lc = t / (NF1 * 5), cf = (t / 5) % NF1, lv = t % 5;
    const bool con = t < CPT * NF1 * 5;
    // output lanes: (cell oc, c coordinate, variable)
    const int oc = t / (N1 * 5), ocl = (t / 5) % N1;
    const bool oon = t < CPT * N1 * 5;
    real fcc[NF1];
#pragma unroll
    for (int q = 0; q < NF1; ++q) fcc[q] = args.tab[K::O_F2CC + (oon ? ocl : 0) * NF1 + q];
    real fr[3];                       // F(q_ref) of the lane's variable
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        fr[m] = (real)args.fref[m * 5];
#pragma unroll
        for (int v = 1; v < 5; ++v) fr[m] = lv == v ? (real)args.fref[m * 5 + v] : fr[m];
    }

    const int64_t n_cells = args.n_cells, n_tiles = (n_cells + CPT - 1) / CPT;
    for (CellWalk cw(n_tiles, 1, 0); cw.it < cw.hi; cw.it += cw.step) {
        Args* a = fresh();
        const int64_t c0 = a->cell_begin + cw.it * CPT;
        const int64_t left = n_cells - cw.it * CPT;
        const int nc = (int)(left < CPT ? left : CPT);
        // the adjugate of this lane's fine point, loaded before the stages that lead to it
        real ad[9];
        if (fon && fc < nc) {
            GlobalPtr<real> src = (GlobalPtr<real>)a->adjf + ((c0 + fc) * NF + ff) * 9;
#pragma unroll
            for (int q = 0; q < 9; ++q) ad[q] = src[q];
        }
        // 0. dQ of the tile
        for (int o = tid; o < nc * NS; o += 64 * NW) {
            const int c = o / NS, s = o % NS;
            real* x = s_w + c * PER + L::OQ + (s / N1) * 20 + s % N1;
            if (a->dQ) {
#pragma unroll
                for (int v = 0; v < 5; ++v) x[v * 4] = ((GlobalPtr<real>)a->dQ)[(c0 * NS + o) * 5 + v];
            } else {
                double u[5], q[5];
                // (field by field at P1: 159 -> 153 us at 304k prisms, no scalar spills; P2: no gain, +0.3%)
                if constexpr (P == 1) load_state(a->U, c0 * NS + o, state_off(a->so), c0 + c, u);
                else load_state(args.U, c0 * NS + o, args.so, c0 + c, u);
                cons2prim(u, q);
#pragma unroll
                for (int v = 0; v < 5; ++v) x[v * 4] = (real)(q[v] - a->qref[v]);
            }
        }
        __syncthreads();
        // 1. coarse -> fine along c
        uni tab = (uni)fresh()->tab;
        for (int o = tid; o < nc * NAB * 5; o += 64 * NW) {
            real* cell = s_w + (o / (NAB * 5)) * PER;
            const int r = o % (NAB * 5);
            const v4 q = ld4(cell + L::OQ + r * 4);
            v4 x = {0, 0, 0, 0};
#pragma unroll
            for (int f = 0; f < NF1; ++f)
#pragma unroll
                for (int c = 0; c < N1; ++c) x[f] += (real)tab[K::O_C2FC + f * N1 + c] * q[c];
            st4(cell + L::OX + r * 4, x);
        }
        __syncthreads();
        // 2. coarse -> fine along (a, b): wave w takes the fine rows w, w + NW, ...
        tab = (uni)fresh()->tab;
        if (con && lc < nc) {
            real* cell = s_w + lc * PER;
            real x[NAB];
#pragma unroll
            for (int ab = 0; ab < NAB; ++ab) x[ab] = cell[L::OX + (ab * 5 + lv) * 4 + cf];
            for (int f = w; f < NABF; f += NW) {
                real acc = 0;
#pragma unroll
                for (int ab = 0; ab < NAB; ++ab) acc += (real)tab[K::O_C2FAB + f * NAB + ab] * x[ab];
                cell[L::OF + (f * NF1 + cf) * 5 + lv] = acc;
            }
        }
        __syncthreads();
        // 3. contravariant flux perturbation at the fine points: F~_m = adj_m . (F(q_ref + dq) -
        //    F(q_ref)) by the exact algebraic expansion about q_ref (every term carries a
        //    perturbation factor, so nothing cancels in the storage precision)
        if (fon && fc < nc) {
            a = fresh();
            const real r0 = (real)a->qref[0], u0 = (real)a->qref[1], v0 = (real)a->qref[2], w0 = (real)a->qref[3];
            const real p0 = (real)a->qref[4];
            const real H0 = (real)(kGamma / (kGamma - 1.0) * a->qref[4] * recip(a->qref[0]) +
                                   0.5 * (a->qref[1] * a->qref[1] + a->qref[2] * a->qref[2] + a->qref[3] * a->qref[3]));
            real* cell = s_w + fc * PER;
            const real* d = cell + L::OF + ff * 5;
            const real dr = d[0], du = d[1], dv = d[2], dw = d[3], dp = d[4];
            const real dpr = (dp * r0 - p0 * dr) * recip(r0 * (r0 + dr));
            const real dH = real(kGamma / (kGamma - 1.0)) * dpr + (u0 * du + v0 * dv + w0 * dw) +
                            real(0.5) * (du * du + dv * dv + dw * dw);
            real* o = cell + L::OT + (ff % NF1) * 5 * RS + ff / NF1;
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                const real a0 = ad[m * 3], a1 = ad[m * 3 + 1], a2 = ad[m * 3 + 2];
                const real un0 = u0 * a0 + v0 * a1 + w0 * a2;
                const real dun = du * a0 + dv * a1 + dw * a2;
                const real m0 = r0 * un0;
                const real dm = r0 * dun + dr * (un0 + dun);
                real* om = o + m * NF1 * 5 * RS;
                om[0] = dm;
                om[RS] = m0 * du + dm * (u0 + du) + dp * a0;
                om[2 * RS] = m0 * dv + dm * (v0 + dv) + dp * a1;
                om[3 * RS] = m0 * dw + dm * (w0 + dw) + dp * a2;
                om[4 * RS] = m0 * dH + dm * (H0 + dH);
            }
        }
        __syncthreads();
        tab = (uni)fresh()->tab;
        // 4. Y (rows ab of group w) and W (c = w)
        if (con && lc < nc) {
            real* cell = s_w + lc * PER;
            real acc[N1];
#pragma unroll
            for (int r = 0; r < N1; ++r) acc[r] = 0;
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                const real* f = cell + L::OT + ((m * NF1 + cf) * 5 + lv) * RS;
#pragma unroll
                for (int qa = 0; qa < QB; ++qa) {
                    const v4 x = ld4(f + 4 * qa);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (4 * qa + e < NABF) {
#pragma unroll
                            for (int r = 0; r < N1; ++r)
                                acc[r] += (real)tab[(m == 0 ? K::O_AA : K::O_AB) + (w * N1 + r) * NABF + 4 * qa + e] * x[e];
                        }
                }
            }
#pragma unroll
            for (int r = 0; r < N1; ++r) cell[L::OY + ((w * N1 + r) * 5 + lv) * 4 + cf] = acc[r];
            // here the lane's cf is the quad index of the fine (a, b) points
            v4 s4 = {0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < NF1; ++q)
                s4 += (real)tab[K::O_BC + w * NF1 + q] * ld4(cell + L::OT + ((2 * NF1 + q) * 5 + lv) * RS + 4 * cf);
            st4(cell + L::OW + (w * 5 + lv) * RS + 4 * cf, s4);
        }
        __syncthreads();
        a = fresh();
        tab = (uni)a->tab;
        // 5. divergence at the solution points of the rows ab of group w
        if (oon && oc < nc) {
            const real* cell = s_w + oc * PER;
            const int64_t p0s = (c0 + oc) * NS;
            real acc[N1];
#pragma unroll
            for (int r = 0; r < N1; ++r) {
                const v4 y = ld4(cell + L::OY + ((w * N1 + r) * 5 + lv) * 4);
                acc[r] = 0;
#pragma unroll
                for (int q = 0; q < NF1; ++q) acc[r] += fcc[q] * y[q];
            }
#pragma unroll
            for (int qa = 0; qa < QB; ++qa) {
                const v4 x = ld4(cell + L::OW + (ocl * 5 + lv) * RS + 4 * qa);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (4 * qa + e < NABF) {
#pragma unroll
                        for (int r = 0; r < N1; ++r)
                            acc[r] += (real)tab[K::O_F2CAB + (w * N1 + r) * NABF + 4 * qa + e] * x[e];
                    }
            }
#pragma unroll
            for (int r = 0; r < N1; ++r) {
                const int64_t pt = p0s + (w * N1 + r) * N1 + ocl;
                GlobalPtr<real> g = (GlobalPtr<real>)a->gcl + pt * 3;
                typedef __attribute__((address_space(1))) real GlobalReal;
                ((GlobalReal*)a->R)[pt * 5 + lv] = acc[r] + g[0] * fr[0] + g[1] * fr[1] + g[2] * fr[2];
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------ inviscid volume kernel (tets, FP64)
// Dense operators (the collapsed tet basis does not factor): two matrix products per tile of 16 cells,
// c2f x (16 cells x 5 variables) and Op x the contravariant fluxes, on the matrix cores.  Each wave keeps its operator fragments in registers for the whole kernel: a row tile of
// c2f, and of Op a row tile (P1, P2: its share of the columns; the shares meet in LDS).  The operands
// pass through LDS as [point][cell, variable], row stride 81: free of bank conflicts for the fragments
// (16 columns of 4 rows) and for the point phases (16 points of a cell).  The flux is formed once per
// fine point in FP64, lane = (cell, fine point), 16 fine points of all three directions at a time.
// Bound: latency of the stages (barriers) at two or three workgroups per CU; the products take about a
// quarter of the time.  Measured: P1, 24.6k tets 24.6 us, P2, 10.3k tets 42, P3, 24.6k tets 185; with
// scalar operands and vector FMAs 25, 60 and 285 (waits for operators that the scalar cache does not hold).
template <int P> struct IT {
    static constexpr int N1 = P + 1, NS = N1 * N1 * N1, OV = (2 * P < 3 ? 2 * P : 3), NF = (OV + 1) * (OV + 1) * (OV + 1);
    static constexpr int CPT = 16, NT = 256, LD = CPT * 5 + 1, CT = CPT * 5 / 16;   // columns: 5 tiles of 16
    static constexpr int KS = (NS + 3) / 4;                     // steps of 4 over the solution points
    static constexpr int RA = (NF + 15) / 16, WA = 4 / RA;      // row tiles of c2f, waves that share one
    static constexpr int RC = (NS + 15) / 16, WC = 4 / RC;      // row tiles of Op, waves that share one
    static constexpr int JS = 4 / WC;                           // steps of 4 fine points of a wave, chunk and direction
    static constexpr int NQ = 16 * RA > 4 * KS ? 16 * RA : 4 * KS;   // rows of the first work area
    static constexpr int N_LDS = (NQ + 48) * LD;
    static_assert(RA * WA == 4 && RC * WC == 4 && NQ + 48 >= 64, "wave shares");
};

template <int P>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_inv_volume_tet_f64(MeanArgs<double> args) {
    typedef double real;
    using L = IT<P>;
    constexpr int NS = L::NS, NF = L::NF, CPT = L::CPT, NT = L::NT, LD = L::LD, KS = L::KS, RA = L::RA, RC = L::RC;
    constexpr int JS = L::JS, CT = L::CT;
    // dQ [s][n], then Qf [j][n]; F~ [m][16 j][n]; then the shares of the result [part][s][n]
    __shared__ double s_q[L::N_LDS];
    double* const s_f = s_q + L::NQ * LD;
    typedef const __attribute__((address_space(4))) MeanArgs<double> Args;
    Args* const kernarg = (Args*)__builtin_amdgcn_kernarg_segment_ptr();
    auto fresh = [&]() -> Args* {        // arguments read anew in every stage instead of held in registers
        Args* p = kernarg;
        asm volatile("" : "+s"(p));
        return p;
    };
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), t = tid & 63;
    const int ln = t % 16, lk = t / 16;
    const int ra = w % RA, rc = w % RC, part = w / RC;
    double fa[KS], fo[RA][3][JS];
#pragma unroll
    for (int k = 0; k < KS; ++k) {
        const int j = ra * 16 + ln, s = 4 * k + lk;
        fa[k] = j < NF && s < NS ? args.c2f[j * NS + s] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < RA; ++k)
#pragma unroll
        for (int m = 0; m < 3; ++m)
#pragma unroll
            for (int q = 0; q < JS; ++q) {
                const int s = rc * 16 + ln, j = k * 16 + (part * JS + q) * 4 + lk;
                fo[k][m][q] = s < NS && j < NF ? args.op[(s * 3 + m) * NF + j] : 0.0;
            }
    const int64_t n_cells = args.n_cells, n_tiles = (n_cells + CPT - 1) / CPT;
    for (CellWalk cw(n_tiles, 1, 0); cw.it < cw.hi; cw.it += cw.step) {
        Args* a = fresh();
        const int64_t c0 = a->cell_begin + cw.it * CPT;
        const int nc = (int)(n_cells - cw.it * CPT < CPT ? n_cells - cw.it * CPT : CPT);
        const int fc = tid / 16, fj = tid % 16;      // fine point of this thread: cell, point of the chunk
        real ad[9];
        auto take_adj = [&](int k) {
            if (fc < nc && k * 16 + fj < NF) {
                GlobalPtr<real> src = (GlobalPtr<real>)fresh()->adjf + ((c0 + fc) * NF + k * 16 + fj) * 9;
#pragma unroll
                for (int e = 0; e < 9; ++e) ad[e] = src[e];
            }
        };
        take_adj(0);
        if constexpr (4 * KS > NS) {     // rows past the points: zero
            for (int o = tid; o < (4 * KS - NS) * LD; o += NT) s_q[NS * LD + o] = real(0);
        }
        for (int o = tid; o < nc * NS; o += NT) {
            const int c = o / NS, s = o % NS;
            real* x = s_q + s * LD + c * 5;
            if (a->dQ) {
#pragma unroll
                for (int v = 0; v < 5; ++v) x[v] = ((GlobalPtr<real>)a->dQ)[(c0 * NS + o) * 5 + v];
            } else {
                double u[5], q[5];
                load_state(a->U, c0 * NS + o, state_off(a->so), c0 + c, u);
                cons2prim(u, q);
#pragma unroll
                for (int v = 0; v < 5; ++v) x[v] = (real)(q[v] - a->qref[v]);
            }
        }
        __syncthreads();
        {
            constexpr int NC = (CT + L::WA - 1) / L::WA;
            d4 q[NC];
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                const int ct = w / RA + i * L::WA;
                q[i] = (d4){0, 0, 0, 0};
                if (ct < CT) {
#pragma unroll
                    for (int k = 0; k < KS; ++k) q[i] = mma(fa[k], s_q[(4 * k + lk) * LD + ct * 16 + ln], q[i]);
                }
            }
            __syncthreads();             // Qf takes the place of dQ
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                const int ct = w / RA + i * L::WA;
                if (ct < CT) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) s_q[(ra * 16 + 4 * e + lk) * LD + ct * 16 + ln] = (real)q[i][e];
                }
            }
        }
        __syncthreads();
        d4 acc[CT];
#pragma unroll
        for (int i = 0; i < CT; ++i) acc[i] = (d4){0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < RA; ++k) {
            // point flux in FP64 about the reference state, its three contravariant components
            a = fresh();
            if (fc < nc) {
                real f[3][5];
#pragma unroll
                for (int i = 0; i < 15; ++i) f[i / 5][i % 5] = real(0);
                if (k * 16 + fj < NF) {
                    double q5[5], F[3][5];
#pragma unroll
                    for (int v = 0; v < 5; ++v) q5[v] = a->qref[v] + (double)s_q[(k * 16 + fj) * LD + fc * 5 + v];
                    euler_flux(q5, F);
                    real d[3][5];
#pragma unroll
                    for (int i = 0; i < 3; ++i)
#pragma unroll
                        for (int v = 0; v < 5; ++v) d[i][v] = (real)(F[i][v] - a->fref[i * 5 + v]);
#pragma unroll
                    for (int m = 0; m < 3; ++m)
#pragma unroll
                        for (int v = 0; v < 5; ++v)
                            f[m][v] = ad[m * 3] * d[0][v] + ad[m * 3 + 1] * d[1][v] + ad[m * 3 + 2] * d[2][v];
                }
#pragma unroll
                for (int i = 0; i < 15; ++i) s_f[(i / 5 * 16 + fj) * LD + fc * 5 + i % 5] = f[i / 5][i % 5];
            }
            if (k + 1 < RA) take_adj(k + 1);
            __syncthreads();
#pragma unroll
            for (int m = 0; m < 3; ++m)
#pragma unroll
                for (int q = 0; q < JS; ++q) {
                    const real* x = s_f + (m * 16 + (part * JS + q) * 4 + lk) * LD + ln;
#pragma unroll
                    for (int i = 0; i < CT; ++i) acc[i] = mma(fo[k][m][q], x[i * 16], acc[i]);
                }
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < CT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                s_q[((part * RC + rc) * 16 + 4 * e + lk) * LD + i * 16 + ln] = acc[i][e];
        __syncthreads();
        a = fresh();
        for (int o = tid; o < nc * NS * 5; o += NT) {
            const int v = o % 5, s = o / 5 % NS, c = o / (5 * NS);
            GlobalPtr<real> g = (GlobalPtr<real>)a->gcl + (c0 * NS + o / 5) * 3;
            double sum = s_q[s * LD + c * 5 + v];
#pragma unroll
            for (int q = 1; q < L::WC; ++q) sum += s_q[(q * RC * 16 + s) * LD + c * 5 + v];
            const real r = (real)sum;
            real fr[3];
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                fr[m] = (real)a->fref[m * 5];
#pragma unroll
                for (int e = 1; e < 5; ++e) fr[m] = v == e ? (real)a->fref[m * 5 + e] : fr[m];
            }
            typedef __attribute__((address_space(1))) real GlobalReal;
            ((GlobalReal*)a->R)[c0 * NS * 5 + o] = r + g[0] * fr[0] + g[1] * fr[1] + g[2] * fr[2];
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------ inviscid volume kernel (tets, FP32)
// Dense operators (the collapsed tet basis does not factor), vector FMAs: the FP32 matrix instruction
// left 1.0e-6 against 64 bits on P1 tets where these sums leave 8e-7, and FP64 products on the matrix
// cores took 67 us where this takes 50 (70k tets).  A workgroup takes 12 cells; in the two contractions
// lane = (cell, variable), 60 of 64, with the operand column in registers and the operator entries from
// scalar loads (one entry serves 60 products; no operator in LDS).  The fluxes are formed once per fine
// point, lane = (cell, fine point), in FP64, and all three contravariant components of a chunk of CH
// points pass through LDS.  P1: three waves, wave m takes direction m of all rows (a value read from LDS
// serves eight rows) and the three parts meet in LDS.  P2: four waves, each its own rows.
// Bound: the waits for scalar operands.  70k P1 tets 50 us (76 with a flux pass per direction and split
// rows).
template <int P> struct IV32 {
    static constexpr int N1 = P + 1, NS = N1 * N1 * N1, OV = (2 * P < 3 ? 2 * P : 3), NF = (OV + 1) * (OV + 1) * (OV + 1);
    static constexpr bool SPLIT = P == 1;                       // waves split directions instead of rows
    static constexpr int CPT = 12, NW = SPLIT ? 3 : 4, NT = 64 * NW;
    static constexpr int RW = SPLIT ? NS : (NS + NW - 1) / NW;  // Op rows of a wave
    static constexpr int CH = SPLIT ? NF : 16, NCH = NF / CH;   // fine points at a time
    // columns of Op whose scalars share one wait (scalar loads return out of order: a wait is for all of
    // them), about 60 of the wave's 102 scalar registers
    static constexpr int KB = SPLIT ? 9 : 8;
    // sums per direction at P2, where the three cancel (operators up to 4e5); P1: a wave has one direction
    static constexpr int AD = SPLIT ? 1 : 3;
    static constexpr int NP = (CPT * CH + NT - 1) / NT;         // fine points of a thread and chunk
    static constexpr int QS = (NS * 5) | 1, FS = (NF * 5) | 1, CS = (CH * 5) | 1;
    static constexpr int N_Q = CPT * (QS > FS ? QS : FS), N_F = 3 * CPT * CS;
    static_assert(NF % CH == 0 && CH % KB == 0, "whole chunks");
    static_assert(NS * 5 <= FS && (!SPLIT || 3 * CPT * NS * 5 <= N_F), "results over the work areas");
};

template <int P>
__global__ void __launch_bounds__((IV32<P>::NT)) k_inv_volume_tet_f32(MeanArgs<float> args) {
    typedef float real;
    using L = IV32<P>;
    using uni = typename Uni<real>::type;
    constexpr int NS = L::NS, NF = L::NF, CPT = L::CPT, NW = L::NW, NT = L::NT, RW = L::RW, NP = L::NP, FS = L::FS;
    constexpr int QS = L::QS, CH = L::CH, CS = L::CS, KB = L::KB;
    __shared__ real s_q[L::N_Q];         // dQ [c][s][5], then Qf [c][j][5], then (rows split) the result
    __shared__ real s_f[L::N_F];         // F~ [m][c][j][5] of a chunk, then (directions split) the parts of the result
    typedef const __attribute__((address_space(4))) MeanArgs<float> Args;
    Args* const kernarg = (Args*)__builtin_amdgcn_kernarg_segment_ptr();
    auto fresh = [&]() -> Args* {        // arguments read anew in every stage instead of held in registers
        Args* p = kernarg;
        asm volatile("" : "+s"(p));
        return p;
    };
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), t = tid & 63;
    const int lc = t / 5, lv = t % 5;
    const int64_t n_cells = args.n_cells, n_tiles = (n_cells + CPT - 1) / CPT;
    for (CellWalk cw(n_tiles, 1, 0); cw.it < cw.hi; cw.it += cw.step) {
        Args* a = fresh();
        const int64_t c0 = a->cell_begin + cw.it * CPT;
        const int nc = (int)(n_cells - cw.it * CPT < CPT ? n_cells - cw.it * CPT : CPT);
        const bool on = t < 5 * CPT && lc < nc;
        // adjugates of this thread's fine points of chunk k
        real ad[NP][9];
        auto take_adj = [&](int k) {
            GlobalPtr<real> src = (GlobalPtr<real>)fresh()->adjf;
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                const int o = tid + NT * q, c = o / CH, j = k * CH + o % CH;
                if (o < nc * CH) {
#pragma unroll
                    for (int e = 0; e < 9; ++e) ad[q][e] = src[((c0 + c) * NF + j) * 9 + e];
                }
            }
        };
        take_adj(0);
        for (int o = tid; o < nc * NS; o += NT) {
            const int c = o / NS, s = o % NS;
            real* x = s_q + c * QS + s * 5;
            if (a->dQ) {
#pragma unroll
                for (int v = 0; v < 5; ++v) x[v] = ((GlobalPtr<real>)a->dQ)[(c0 * NS + o) * 5 + v];
            } else {
                double u[5], q[5];
                load_state(a->U, c0 * NS + o, state_off(a->so), c0 + c, u);
                cons2prim(u, q);
#pragma unroll
                for (int v = 0; v < 5; ++v) x[v] = (real)(q[v] - a->qref[v]);
            }
        }
        __syncthreads();
        {
            real x[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) x[s] = s_q[(on ? lc : 0) * QS + s * 5 + lv];
            __syncthreads();
            const uni c2f = (uni)fresh()->c2f;
#pragma unroll 1
            for (int j = w; j < NF; j += NW) {
                real acc = 0, c[NS];
#pragma unroll
                for (int e = 0; e < NS; ++e) c[e] = (real)c2f[j * NS + e];
#pragma unroll
                for (int e = 0; e < NS; ++e) acc += c[e] * x[e];
                if (on) s_q[lc * FS + j * 5 + lv] = acc;
            }
        }
        __syncthreads();
        constexpr int AD = L::AD;
        real acc[AD][RW];
#pragma unroll
        for (int m = 0; m < AD; ++m)
#pragma unroll
            for (int r = 0; r < RW; ++r) acc[m][r] = 0;
#pragma unroll 1
        for (int k = 0; k < L::NCH; ++k) {
            // point flux in FP64 about the reference state, its three contravariant components
            a = fresh();
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                const int o = tid + NT * q, c = o / CH, j = o % CH;
                if (o < nc * CH) {
                    const real* dq = s_q + c * FS + (k * CH + j) * 5;
                    double q5[5], F[3][5];
#pragma unroll
                    for (int v = 0; v < 5; ++v) q5[v] = a->qref[v] + (double)dq[v];
                    euler_flux(q5, F);
                    real f[3][5];
#pragma unroll
                    for (int i = 0; i < 3; ++i)
#pragma unroll
                        for (int v = 0; v < 5; ++v) f[i][v] = (real)(F[i][v] - a->fref[i * 5 + v]);
#pragma unroll
                    for (int m = 0; m < 3; ++m)
#pragma unroll
                        for (int v = 0; v < 5; ++v)
                            s_f[(m * CPT + c) * CS + j * 5 + v] =
                                ad[q][m * 3] * f[0][v] + ad[q][m * 3 + 1] * f[1][v] + ad[q][m * 3 + 2] * f[2][v];
                }
            }
            if (k + 1 < L::NCH) take_adj(k + 1);
            __syncthreads();
            const uni op = (uni)fresh()->op;
            auto row = [&](int r) { return L::SPLIT ? r : (w * RW + r < NS ? w * RW + r : NS - 1); };
            auto columns = [&](int m, int j0, real* sum) {   // sum += op[rows][m][k CH + j0 ..] F~_m
                real y[KB];
                const real* f = s_f + (m * CPT + (on ? lc : 0)) * CS + j0 * 5 + lv;
#pragma unroll
                for (int e = 0; e < KB; ++e) y[e] = f[e * 5];
                const uni o0 = op + m * NF + k * CH + j0;
                real c[RW][KB];
#pragma unroll
                for (int r = 0; r < RW; ++r)
#pragma unroll
                    for (int e = 0; e < KB; ++e) c[r][e] = (real)o0[row(r) * 3 * NF + e];
#pragma unroll
                for (int r = 0; r < RW; ++r)
#pragma unroll
                    for (int e = 0; e < KB; ++e) sum[r] += c[r][e] * y[e];
            };
            if constexpr (L::SPLIT) {
#pragma unroll 1
                for (int j0 = 0; j0 < CH; j0 += KB) columns(w, j0, acc[0]);
            } else {
                auto direction = [&](int m, real* sum) {
#pragma unroll 1
                    for (int j0 = 0; j0 < CH; j0 += KB) columns(m, j0, sum);
                };
                direction(0, acc[0]);
                direction(1, acc[1]);
                direction(2, acc[2]);
            }
            __syncthreads();
        }
        real* const out = L::SPLIT ? s_f + w * CPT * NS * 5 : s_q;
        if (on) {
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                const int s = L::SPLIT ? r : w * RW + r;
                if (s < NS) out[(lc * NS + s) * 5 + lv] = AD == 1 ? acc[0][r] : acc[0][r] + acc[AD > 1 ? 1 : 0][r] + acc[AD > 1 ? 2 : 0][r];
            }
        }
        __syncthreads();
        a = fresh();
        for (int o = tid; o < nc * NS * 5; o += NT) {
            const int v = o % 5;
            const int64_t pt = c0 * NS + o / 5;
            GlobalPtr<real> g = (GlobalPtr<real>)a->gcl + pt * 3;
            real r;
            if constexpr (L::SPLIT) r = s_f[o] + s_f[CPT * NS * 5 + o] + s_f[2 * CPT * NS * 5 + o];
            else r = s_q[o];
            real fr[3];
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                fr[m] = (real)a->fref[m * 5];
#pragma unroll
                for (int e = 1; e < 5; ++e) fr[m] = v == e ? (real)a->fref[m * 5 + e] : fr[m];
            }
            typedef __attribute__((address_space(1))) real GlobalReal;
            ((GlobalReal*)a->R)[c0 * NS * 5 + o] = r + g[0] * fr[0] + g[1] * fr[1] + g[2] * fr[2];
        }
        __syncthreads();
    }
}

template <int P, int CT, typename real>
int launch_inv_volume(const MeanArgs<real>& a, hipStream_t st) {
    if (a.n_cells <= 0) return 0;
    if constexpr (CT == 0) {
        using L = IV<P, real>;
        const int64_t tiles = (a.n_cells + L::CPT - 1) / L::CPT;
        const int grid = walk_grid(tiles, 1, a.grid_cap > 0 ? a.grid_cap : 8192);
        hipLaunchKernelGGL((k_inv_volume<P, real>), dim3(grid), dim3(64 * L::NW), 0, st, a);
    } else {
        using L = std::conditional_t<sizeof(real) == 8, IT<P>, IV32<P>>;
        const int64_t tiles = (a.n_cells + L::CPT - 1) / L::CPT;
        const dim3 grid(walk_grid(tiles, 1, a.grid_cap > 0 ? a.grid_cap : 4096));
        if constexpr (sizeof(real) == 8) hipLaunchKernelGGL((k_inv_volume_tet_f64<P>), grid, dim3(L::NT), 0, st, a);
        else hipLaunchKernelGGL((k_inv_volume_tet_f32<P>), grid, dim3(L::NT), 0, st, a);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

#define AFR_VOL_INST(P, CT, T)                                                       \
    template int launch_visc_volume<P, CT, T>(const MeanArgs<T>&, hipStream_t);      \
    template int launch_inv_volume<P, CT, T>(const MeanArgs<T>&, hipStream_t);
AFR_VOL_INST(1, 0, float)
AFR_VOL_INST(2, 0, float)
AFR_VOL_INST(1, 0, double)
AFR_VOL_INST(2, 0, double)
AFR_VOL_INST(1, 1, float)
AFR_VOL_INST(2, 1, float)
AFR_VOL_INST(1, 1, double)
AFR_VOL_INST(2, 1, double)
AFR_VOL_INST(3, 1, double)

}  // namespace afr_mean
