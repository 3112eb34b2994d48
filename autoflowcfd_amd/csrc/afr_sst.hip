// SST k-omega turbulence step on the device (once per pseudo-step, before the
// mean-flow stages), FP64 arithmetic on storage-precision fields.
//
//   k_sst_cell    per cell: strain rate from the gradient of the conserved momentum,
//                 clipped grad k / grad omega, F1, F2, nu_t (viscosity-ratio cap),
//                 production / destruction / cross diffusion with mu = 1.8e-5
//                 (src/autoflowcfd/core/turbulence/sst.py:21-330,
//                  src/autoflowcfd/core/fr_solver/turbulence.py:178-330);
//                 transport volume terms -D.(adj rho u phi)/det, -D.(adj Gamma grad phi)/det
//                 and the face pack (src/autoflowcfd/core/turbulence/transport.py:122-360)
//   k_sst_face    per face record and flux point: upwind convection and BR1-type
//                 diffusion corrections from the owner side, Neumann ghost on records
//                 without neighbour sources, Dirichlet-zero k on WALL records
//                 (src/autoflowcfd/core/turbulence/transport_kernel.py:103-170)
//   k_sst_update  per cell: record corrections gathered with the owner's / neighbour's
//                 flux-point maps (transport_kernel.py:200-260), / rho, outlier zeroing,
//                 point-implicit source damping and explicit update with the local time
//                 step, floors (src/autoflowcfd/core/turbulence/sst.py:335-479)
//   k_wall_distance  nearest wall node per solution point, FP64 brute force
//                 (src/autoflowcfd/core/fr_solver/turbulence.py:112-121 uses a KD-tree)
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/afr.h"
#include "afr_meanflow.hpp"
#include "afr_physics.hpp"
#include "afr_sst.hpp"
#include "afr_sst_point.hpp"
#include "afr_outlier.hpp"

using namespace afr;

namespace afr_sst {

constexpr int kWaves = 4;

using afr_mean::V4;
using afr_mean::ld4;
using afr_mean::st4;
using afr_mean::wave_sync;
template <typename real> struct V2;
template <> struct V2<float> { typedef float type __attribute__((ext_vector_type(2))); };
template <> struct V2<double> { typedef double type __attribute__((ext_vector_type(2))); };

// acc += w x by components: a vector product would keep w splatted over as many registers
template <typename V, typename real> __device__ __forceinline__ void fma_to(V& acc, real w, V x) {
    if constexpr (std::is_same<V, real>::value) acc += w * x;
    else {
#pragma unroll
        for (int q = 0; q < (int)(sizeof(V) / sizeof(real)); ++q) acc[q] += w * x[q];
    }
}

// Lanes of a wavefront: (cell, solution point), LW lanes per cell: 8 cells at P1, 2 (27 of 32 lanes) at P2
template <int P, int CT> struct SO {
    static constexpr int N1 = P + 1, NS = N1 * N1 * N1, NFP = N1 * N1, NSLOT = CT == 0 ? 5 : 4;
    static constexpr int LW = NS <= 8 ? 8 : 32, CPW = 64 / LW;
};

// ------------------------------------------------------------------ per-cell sources and volume terms
// The contractions (gradients D x, face traces E x, volume divergence D F) run in the storage
// precision on per-cell perturbations x - x_0 (x_0: the value at the cell's first solution point; D
// rows sum to zero and E rows to one, so D x = D (x - x_0) and E x = x_0 + E (x - x_0)), which keeps
// FP32 contractions as accurate as FP64 ones on FP32 data.  The SST source terms are FP64 (the blend
// functions FP32 on the FP32 path).
//
// A lane keeps the non-zeros of its derivative rows in registers for the whole kernel (d/da: an a
// line, d/db: an (a, b) plane, d/dc: a c line of a prism, every point of a tet from LDS).  The trace rows
// lie in LDS; a prism's flux points are dealt out to the lanes with the N1^2-wide b face last, so that only
// the last round is wide.  Fields lie in LDS as 16-byte vectors of perturbations, so a non-zero
// costs one or two LDS reads and no subtraction.  Traces are written for slots that own a face
// record only: no other is read.
//
// Bound: FP64 source arithmetic and HBM together (4.3 GB at 82^3 P2 FP32).  Measured there 1165 us,
// before (rows as index / weight tables in LDS, one 4-byte read and one subtraction per product, every
// slot's trace) 1938; 304k P1 prisms FP32 95 us (252, 24 of 64 lanes busy).
template <int P, int CT> struct SC {
    using O = SO<P, CT>;
    static constexpr int NS = O::NS, NI = O::NSLOT * O::NFP, RD = (NI + O::LW - 1) / O::LW;
    static constexpr int PER = (NS * 14 + 3) / 4 * 4;           // two 4-vectors and three pairs per point
    static constexpr int DT = CT == 1 ? NS * (NS | 1) : 1;      // d/dc rows of a tet
    // flux points in the order they are dealt out: prism slots 0, 1, 3, 4, 2
    static constexpr __device__ int slot(int o) {
        const int q = o / O::NFP;
        return CT == 1 ? q : (q < 2 ? q : (q == 4 ? 2 : q + 1));
    }
    // non-zeros of a prism's trace rows in round r
    static constexpr int nnz(int r) { return (r + 1) * O::LW > 4 * O::NFP ? O::N1 * O::N1 : O::N1; }
    static constexpr int first(int r) { return r == 0 ? 0 : first(r - 1) + nnz(r - 1); }
    static constexpr int ET = CT == 1 ? NI * (NS | 1) : first(RD) * O::LW;   // trace rows: tets (row, point)
    template <typename real> static constexpr int wpe() { return sizeof(real) == 4 ? (P == 2 && CT == 0 ? 3 : 4) : (P == 2 && CT == 1 ? 1 : 2); }
};

template <int P, int CT, typename real>
__global__ void __launch_bounds__(64 * kWaves)
    __attribute__((amdgpu_waves_per_eu(SC<P, CT>::template wpe<real>()))) k_sst_cell(SstArgs<real> a) {
    using O = SO<P, CT>;
    using L = SC<P, CT>;
    using v4 = typename V4<real>::type;
    using v2 = typename V2<real>::type;
    constexpr int N1 = O::N1, NS = O::NS, NFP = O::NFP, LW = O::LW, CPW = O::CPW, RS = NS | 1;
    __shared__ __attribute__((aligned(16))) real s_w[kWaves][CPW * L::PER];
    __shared__ real s_dc[L::DT], s_e[L::ET];
    __shared__ int s_eb[L::RD * LW];
    const int tid = threadIdx.x, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t0 = tid & 63;
    if constexpr (CT == 1) {
        for (int q = tid; q < NS * NS; q += 64 * kWaves) s_dc[(q / NS) * RS + q % NS] = a.D[2 * NS * NS + q];
        for (int q = tid; q < L::NI * NS; q += 64 * kWaves) s_e[(q / NS) * RS + q % NS] = a.E[q];
        __syncthreads();
    }
    real wa[N1], wb[N1 * N1], wc[N1];
    {
    const int tl = t0 % LW, sp = tl < NS ? tl : 0, i = sp / (N1 * N1), j = (sp / N1) % N1, k = sp % N1;
#pragma unroll
    for (int q = 0; q < N1; ++q) {
        wa[q] = a.D[sp * NS + (q * N1 + j) * N1 + k];
        wc[q] = CT == 0 ? a.D[(2 * NS + sp) * NS + (i * N1 + j) * N1 + q] : real(0);
    }
#pragma unroll
    for (int q = 0; q < N1 * N1; ++q) wb[q] = a.D[(NS + sp) * NS + q * N1 + k];
    }
    // trace rows of the lanes' flux points: weights and first point
    if constexpr (CT == 0) {
        for (int x = tid; x < L::RD * LW; x += 64 * kWaves) {
            const int r = x / LW, o = x < L::NI ? x : 0, slot = L::slot(o), fp = o % NFP;
            const int y = fp / N1, z = fp % N1;      // a: (b, c), b: (a, c), c: (a, b)
            const int n = slot == 2 ? N1 * N1 : N1, st = slot < 2 ? N1 * N1 : (slot == 2 ? N1 : 1);
            const int b = slot < 2 ? y * N1 + z : (slot == 2 ? z : (y * N1 + z) * N1);
            s_eb[x] = b;
            for (int q = 0; q < L::nnz(r); ++q)
                s_e[(L::first(r) + q) * LW + x % LW] = q < n ? a.E[(slot * NFP + fp) * NS + b + q * st] : real(0);
        }
        __syncthreads();
    }
    const double mu = a.mu_molecular;
    const int64_t n_units = (a.n_cells + CPW - 1) / CPW;
    for (CellWalk cw(n_units, kWaves, wid); cw.it < cw.hi; cw.it += cw.step) {
        const int64_t c0 = cw.it * CPW;
        // the lane's indexes are formed anew for every cell: held over the loop, the addresses made from
        // them would take the registers that the contractions need
        const int t = afr_mean::lane_fresh(t0);
        const int h = t / LW, tl = t % LW;               // cell of the wave, lane within the cell
        const int sp = tl < NS ? tl : 0, i = sp / (N1 * N1), j = (sp / N1) % N1, k = sp % N1;
        real* const sA = s_w[wid] + h * L::PER;          // m1, m2, m3, k, then rho, u, v, w
        real* const sB = sA + NS * 4;                    // k, omega, Gamma_k, Gamma_omega
        real* const sV = sA + NS * 8;                    // omega, then the contravariant fluxes [m][s][k, omega]
        // row m of this lane's point applied to a 4-vector field / a field of stride 1 / of pairs
        auto apply = [&](int m, auto zero, auto get) {
            auto acc = zero;
            if (m == 0) {
    #pragma unroll
                for (int q = 0; q < N1; ++q) fma_to(acc, wa[q], get(q * N1 * N1 + j * N1 + k));
            } else if (m == 1) {
    #pragma unroll
                for (int q = 0; q < N1 * N1; ++q) fma_to(acc, wb[q], get(q * N1 + k));
            } else if constexpr (CT == 0) {
    #pragma unroll
                for (int q = 0; q < N1; ++q) fma_to(acc, wc[q], get((i * N1 + j) * N1 + q));
            } else {
    #pragma unroll 4
                for (int q = 0; q < NS; ++q) fma_to(acc, s_dc[sp * RS + q], get(q));
            }
            return acc;
        };
        auto at0 = [&](real x) { return __shfl(x, h * LW); };   // the value at the cell's first point
        const int nc = (int)(a.n_cells - c0 < CPW ? a.n_cells - c0 : CPW);
        const bool live = tl < NS && h < nc;
        const int64_t cell = a.cell_begin + c0 + (h < nc ? h : 0);
        const int64_t pt = cell * NS + sp;
        // codes of the faces whose records this cell owns
        int own = 0;
        if (tl < kInc) {
            const int e = a.inc[cell * kInc + tl];
            own = e >= 0 && !(e & 8) ? 1 << (e & 7) : 0;
        }
#pragma unroll
        for (int m = 1; m < kInc; m <<= 1) own |= __shfl_xor(own, m);
        if constexpr (LW > kInc) own = __shfl(own, h * LW);
        real ad[9], u5[5];
#pragma unroll
        for (int q = 0; q < 9; ++q) ad[q] = a.adj[pt * 9 + q];
        const real ks0 = a.k[pt], ws0 = a.w[pt], dw = a.d_wall[pt], idet = recip(a.det[pt]);
        {
            double off[5];
            a.so.row(cell, off);
#pragma unroll
            for (int v = 0; v < 5; ++v)
                u5[v] = a.so.mode ? (real)((double)a.U[pt * 5 + v] + off[v]) : a.U[pt * 5 + v];
        }
        const real rr = u5[0] > real(1e-10) ? u5[0] : real(1e-10);
        const real k0 = at0(ks0), w0 = at0(ws0);
        {
            const real m0[3] = {at0(u5[1]), at0(u5[2]), at0(u5[3])};
            if (live) {
                st4(sA + sp * 4, (v4){u5[1] - m0[0], u5[2] - m0[1], u5[3] - m0[2], ks0 - k0});
                sV[sp] = ws0 - w0;
            }
        }
        wave_sync();
        real gm[3][3], gk[3], gw[3];
        {
            v4 d[3];
            real e[3];
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                d[m] = apply(m, (v4){0, 0, 0, 0}, [&](int q) { return ld4(sA + q * 4); });
                e[m] = apply(m, real(0), [&](int q) { return sV[q]; });
                __builtin_amdgcn_sched_barrier(0);   // one row's loads in flight at a time: registers
            }
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                const v4 g = (ad[n] * d[0] + ad[3 + n] * d[1] + ad[6 + n] * d[2]) * idet;
                gm[0][n] = g[0];
                gm[1][n] = g[1];
                gm[2][n] = g[2];
                gk[n] = g[3];
                gw[n] = (ad[n] * e[0] + ad[3 + n] * e[1] + ad[6 + n] * e[2]) * idet;
            }
        }
        // sources of the point (FP64), mu = 1.8e-5 as the reference's source terms
        const double rho = (double)rr, kd = (double)ks0, wd = (double)ws0, dd = (double)dw;
        const double irho = recip(dmax(rho, 1e-10));
        real Gk, Gw;
        {
            double S2 = 0.0;
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                const double q = (double)gm[p][p], o = (double)gm[p][(p + 1) % 3] + (double)gm[(p + 1) % 3][p];
                S2 += q * q + 0.5 * (o * o);
            }
            const double SS2 = 2.0 * S2, S = sqrt(SS2);
            // clipped gradients of k and omega
            double fk = 1.0, fw = 1.0, mk = 0.0, mw = 0.0, gd = 0.0;
#pragma unroll
            for (int n = 0; n < 3; ++n) {
                mk += (double)gk[n] * (double)gk[n];
                mw += (double)gw[n] * (double)gw[n];
            }
            if (mk > 1e12) fk = dmin(dmax(1e6 / dmax(sqrt(mk), 1e-10), 0.0), 1.0);
            if (mw > 1e12) fw = dmin(dmax(1e6 / dmax(sqrt(mw), 1e-10), 0.0), 1.0);
#pragma unroll
            for (int n = 0; n < 3; ++n) gd += (fk * (double)gk[n]) * (fw * (double)gw[n]);
            const double musrc = 1.8e-5;
            const double ks = dmin(kd, 1e40), wsf = dmax(dmin(wd, 1e40), 1e-10);
            const double cross = 2.0 * rho * SW2 * recip(wsf) * gd;
            double F1, F2;
            __builtin_amdgcn_sched_barrier(0);
            Blend<real>::both(ks, wsf, dd, musrc * irho, rho, dmax(cross, 1e-10), F1, F2);
            const double beta = F1 * B1 + (1.0 - F1) * B2;
            const double kk = dmax(ks, 1e-10), SS = dmax(S, 1e-10);
            double nut = A1 * kk * recip(dmax(A1 * wsf, F2 * SS));
            nut = dmin(nut, 1.0e5 * musrc * irho);
            nut = isfinite(nut) ? nut : 0.0;
            const double rnut = rho * nut, Dk = BSTAR * rho * ks * wsf;
            double Sk = dmin(rnut * S * S, 10.0 * Dk) - Dk;
            const double g1 = B1 / BSTAR - SW1 * KAP * KAP / sqrt(BSTAR);
            const double g2 = B2 / BSTAR - SW2 * KAP * KAP / sqrt(BSTAR);
            const double gam = F1 * g1 + (1.0 - F1) * g2;
            double Sw = rho * gam * S * S - rho * beta * wsf * wsf + (1.0 - F1) * cross;
            Sk = finite_or(Sk, 0.0);
            Sw = finite_or(Sw, 0.0);
            // diffusivities with the transport's own F1 (molecular mu, raw k / omega): the same
            // arguments as the sources' F1 unless mu differs or k, omega were clipped
            double F1t = F1;
            if (!(mu == musrc && kd <= 1e40 && wd <= 1e40)) {
                const double CDt = dmax(2.0 * rho * SW2 / dmax(wd, 1e-10) * gd, 1e-10);
                F1t = Blend<real>::F1(kd, wd, dd, mu * irho, rho, CDt);
            }
            Gk = (real)(mu + (F1t * SK1 + (1.0 - F1t) * SK2) * rnut);
            Gw = (real)(mu + (F1t * SW1 + (1.0 - F1t) * SW2) * rnut);
            if (live) {
                a.src[pt * 3 + 0] = (real)(Sk * irho);
                a.src[pt * 3 + 1] = (real)(Sw * irho);
                a.src[pt * 3 + 2] = (real)beta;
                a.nu_t[pt] = (real)nut;
                a.mu_t[pt] = (real)rnut;
                st4(a.nbp + pt * 4, (v4){ks0, ws0, Gk, Gw});
            }
        }
        const v4 xa = {rr, (real)((double)u5[1] * irho), (real)((double)u5[2] * irho), (real)((double)u5[3] * irho)};
        const v4 xb = {ks0, ws0, Gk, Gw};
        const v4 a0 = {at0(xa[0]), at0(xa[1]), at0(xa[2]), at0(xa[3])};
        const v4 b0 = {k0, w0, at0(Gk), at0(Gw)};
        wave_sync();
        // contravariant transport fluxes (raw gradients in the diffusion), convective + diffusive
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            const real fr = ad[m * 3] * (rr * xa[1]) + ad[m * 3 + 1] * (rr * xa[2]) + ad[m * 3 + 2] * (rr * xa[3]);
            const real fk = fr * ks0 + Gk * (ad[m * 3] * gk[0] + ad[m * 3 + 1] * gk[1] + ad[m * 3 + 2] * gk[2]);
            const real fw = fr * ws0 + Gw * (ad[m * 3] * gw[0] + ad[m * 3 + 1] * gw[1] + ad[m * 3 + 2] * gw[2]);
            const v2 f = {fk - at0(fk), fw - at0(fw)};
            if (live) *reinterpret_cast<v2*>(sV + (m * NS + sp) * 2) = f;
        }
        if (live) {
            st4(sA + sp * 4, xa - a0);
            st4(sB + sp * 4, xb - b0);
        }
        wave_sync();
        // owner-side face traces of (rho, u, v, w, k, omega, Gamma_k, Gamma_omega)
#pragma unroll
        for (int r = 0; r < L::RD; ++r) {
            const int o = tl + r * LW, slot = L::slot(o), fp = o % NFP;
            if (o < L::NI && h < nc && (own >> (slot < 3 ? slot : slot + 1) & 1)) {
                v4 ta = {0, 0, 0, 0}, tb = ta;   // the perturbation alone: one rounding at the size of x_0
                if constexpr (CT == 0) {
                    const int b = s_eb[o], st = slot < 2 ? N1 * N1 : (slot == 2 ? N1 : 1);
#pragma unroll
                    for (int q = 0; q < L::nnz(r); ++q) {
                        const int x = q < N1 || slot == 2 ? b + q * st : 0;   // narrow rows: padding
                        const real w = s_e[(L::first(r) + q) * LW + tl];
                        fma_to(ta, w, ld4(sA + x * 4));
                        fma_to(tb, w, ld4(sB + x * 4));
                    }
                } else {
#pragma unroll 2
                    for (int q = 0; q < NS; ++q) {
                        const real e = s_e[o * RS + q];
                        fma_to(ta, e, ld4(sA + q * 4));
                        fma_to(tb, e, ld4(sB + q * 4));
                    }
                }
                real* ov = a.pack + ((cell * 5 + slot) * NFP + fp) * kPack;
                st4(ov, a0 + ta);
                st4(ov + 4, b0 + tb);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // volume terms: -(D.F)/det for k and omega
        {
            v2 acc = {0, 0};
#pragma unroll
            for (int m = 0; m < 3; ++m)
                acc += apply(m, (v2){0, 0}, [&](int q) { return *reinterpret_cast<const v2*>(sV + (m * NS + q) * 2); });
            if (live) *reinterpret_cast<v2*>(a.vol + pt * 2) = -acc * idet;
        }
        wave_sync();
    }
}

// ------------------------------------------------------------------ per face record corrections
template <int P, int KMAX, typename real>
__global__ void __launch_bounds__(256) k_sst_face(SstArgs<real> a) {
    constexpr int N1 = P + 1, NS = N1 * N1 * N1, NFP = N1 * N1;
    // the deduplicated neighbour row blocks in LDS when they fit (8 blocks for a graded prism box)
    constexpr int ROWS_CAP = 8 * NFP + 1;
    __shared__ real s_rw[ROWS_CAP * KMAX];
    __shared__ int s_ri[ROWS_CAP * KMAX];
    const bool rows_lds = a.n_rows + 1 <= ROWS_CAP;
    if (rows_lds) {
        for (int i = threadIdx.x; i < (a.n_rows + 1) * KMAX; i += 256) {   // the rows and one of zeros
            const bool in = i < a.n_rows * KMAX;
            s_rw[i] = in ? a.rows_w[i] : real(0);
            s_ri[i] = in ? a.rows_idx[i] : 0;
        }
    }
    __syncthreads();
    const int64_t n = a.n_records * NFP;
    for (int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x; g < n; g += (int64_t)gridDim.x * 256) {
        const int64_t r = g / NFP;
        const int fp = (int)(g % NFP);
        const int64_t o = a.rec_owner[r];
        const int slot = a.rec_oslot[r];
        const int flags = a.rec_flags[r];
        double po[kPack], pn[4];
        const real* tr = a.pack + ((o * 5 + slot) * NFP + fp) * kPack;
#pragma unroll
        for (int q = 0; q < kPack; ++q) po[q] = (double)tr[q];
        if (flags & 1) {
            // neighbour k, omega, Gammas at the owner's flux points through the owner's face slot
            const int64_t sidx = o * 5 + slot;
            const int src = (a.slot_mask[sidx] >> fp) & 1;
            int row = a.slot_blk[sidx * 2 + src] * NFP + fp;
            const int nbc = a.slot_nb[sidx * 2 + src];
            const bool have = row >= 0 && row < a.n_rows && nbc >= 0;
            const int64_t nb = have ? nbc : 0;
            if (!have) row = rows_lds ? a.n_rows : 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) pn[q] = 0.0;
            int spk[KMAX];
            real wk[KMAX];
            if (rows_lds) {
#pragma unroll
                for (int kk = 0; kk < KMAX; ++kk) {  // rows are KMAX wide (zero-padded)
                    spk[kk] = s_ri[row * KMAX + kk];
                    wk[kk] = s_rw[row * KMAX + kk];
                }
            } else {
#pragma unroll
                for (int kk = 0; kk < KMAX; ++kk) {
                    spk[kk] = a.rows_idx[(int64_t)row * KMAX + kk];
                    const real w = a.rows_w[(int64_t)row * KMAX + kk];
                    wk[kk] = have ? w : real(0);
                }
            }
#pragma unroll
            for (int kk = 0; kk < KMAX; ++kk) {
                const real* pk = a.nbp + (nb * NS + spk[kk]) * 4;
                const double wgt = (double)wk[kk];
#pragma unroll
                for (int q = 0; q < 4; ++q) pn[q] += wgt * (double)pk[q];
            }
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) pn[q] = po[4 + q];
            if (flags & 2) pn[0] = -po[4];  // k = 0 on no-slip walls: mirrored ghost
        }
        const double n0 = (double)a.rec_tn[r * 3 + 0], n1 = (double)a.rec_tn[r * 3 + 1], n2 = (double)a.rec_tn[r * 3 + 2];
        const double mass = po[0] * (po[1] * n0 + po[2] * n1 + po[3] * n2);
        double c[2];
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            const double phio = po[4 + f], phin = pn[f];
            const double up = mass >= 0.0 ? phio : phin;
            const double gface = 0.5 * (po[6 + f] + pn[2 + f]);
            c[f] = mass * (up - phio) - gface * (0.5 * (phio + phin) - phio);
        }
        a.crec[g * 2 + 0] = (real)c[0];
        a.crec[g * 2 + 1] = (real)c[1];
    }
}

// ------------------------------------------------------------------ gather, outlier zeroing, update
// One lane per solution point takes both fields through gather, zeroing and update in registers.  The
// outlier rule's certificate (at most (NS - 1) / 2 values below 1e-4 of the largest: then the median
// is too large for any value to be zeroed) takes the maximum over the cell's lanes and counts in a
// ballot, on values rounded to FP32: its margin of 1e-4 of the threshold covers the rounding, and
// values that FP32 could not tell from zero or infinity go the exact way.
// Bound: HBM and the gather of record corrections.  Measured (82^3 P2 FP32): 621 us, 1298 with one cell
// per wavefront and the FP64 certificate through LDS; 304k P1 prisms 51 us (308).
template <int LW> __device__ __forceinline__ float cell_max(float x) {
    x = fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xf, 0xf, false)));    // xor 1
    x = fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xf, 0xf, false)));    // xor 2
    x = fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x141, 0xf, 0xf, false)));   // half row
    if constexpr (LW > 8) {
        x = fmaxf(x, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x140, 0xf, 0xf, false)));   // row
        x = fmaxf(x, __shfl_xor(x, 16));
    }
    return x;
}

template <int P, int CT, typename real>
__global__ void __launch_bounds__(64 * kWaves) k_sst_update(SstArgs<real> a) {
    using O = SO<P, CT>;
    using v2 = typename V2<real>::type;
    constexpr int NS = O::NS, NFP = O::NFP, LW = O::LW, CPW = O::CPW;
    constexpr int k1 = (NS - 1) / 2, k2 = NS / 2;
    __shared__ double s_x[kWaves][CPW * NS * 2], s_med[kWaves][CPW * 4];
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t = threadIdx.x & 63;
    const int h = t / LW, tl = t % LW, s = tl < NS ? tl : 0;
    const uint64_t group = (LW == 64 ? ~0ull : ((1ull << LW) - 1)) << (h * LW);
    // flux point of the point on each axis, correction-function values at its coordinate
    int fps[3];
    real gl[3], gr[3];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        fps[ax] = a.fp_of_sp[ax * NS + s];
        const int cs = a.coord_of_sp[ax * NS + s];
        gl[ax] = a.gL[cs];
        gr[ax] = a.gR[cs];
    }
    const int64_t n_units = (a.n_cells + CPW - 1) / CPW;
    for (CellWalk cw(n_units, kWaves, wid); cw.it < cw.hi; cw.it += cw.step) {
        const int64_t c0 = cw.it * CPW;
        const int nc = (int)(a.n_cells - c0 < CPW ? a.n_cells - c0 : CPW);
        const bool live = tl < NS && h < nc;
        const int64_t pos = c0 + (h < nc ? h : 0);
        const int64_t cell = a.cell_begin + (a.schedule ? a.schedule[pos] : pos);
        const int64_t i = cell * NS + s;
        int ev[kInc];
#pragma unroll
        for (int q = 0; q < kInc; ++q) ev[q] = a.inc[cell * kInc + q];
        v2 cv[kInc];
#pragma unroll
        for (int q = 0; q < kInc; ++q) {
            const int e = ev[q], axis = (e & 7) >> 1;
            const int fp = axis == 0 ? fps[0] : (axis == 1 ? fps[1] : fps[2]);
            cv[q] = (v2){0, 0};
            if (e >= 0) cv[q] = *reinterpret_cast<const v2*>(a.crec + ((int64_t)(e >> 4) * NFP + fp) * 2);
        }
        const v2 vol = *reinterpret_cast<const v2*>(a.vol + i * 2);
        const real det = a.det[i], u0 = a.U[i * 5], kr = a.k[i], wr = a.w[i], dtr = a.dt[i];
        const real s0 = a.src[i * 3], s1 = a.src[i * 3 + 1], s2 = a.src[i * 3 + 2];
        double off[5];
        a.so.row(cell, off);
        double ak = 0.0, aw = 0.0;
#pragma unroll
        for (int q = 0; q < kInc; ++q) {
            const int e = ev[q], axis = (e & 7) >> 1;
            const real gm = axis == 0 ? gl[0] : (axis == 1 ? gl[1] : gl[2]);
            const real gp = axis == 0 ? gr[0] : (axis == 1 ? gr[1] : gr[2]);
            double g = (double)((e & 1) ? gp : gm);
            g = e < 0 ? 0.0 : ((e & 8) ? g : -g);
            ak += g * (double)cv[q][0];
            aw += g * (double)cv[q][1];
        }
        const double irho = recip(dmax((double)u0 + off[0], 1e-10)), idet = recip((double)det);
        double tk = ((double)vol[0] + ak * idet) * irho, tw = ((double)vol[1] + aw * idet) * irho;
        // outlier zeroing per field (troubled_cell.py:339-408 with n_vars = 1, once for k and once
        // for omega, each field's own mean |value| as the reference magnitude), then non-finite
        // transport values -> 0 (transport.py:509-515)
        {
            const float xk = live ? (float)fabs(tk) : 0.0f, xw = live ? (float)fabs(tw) : 0.0f;
            const float mk = cell_max<LW>(xk), mw = cell_max<LW>(xw);
            const int nk = __popcll(__ballot(live && xk < mk * 1.0001e-4f) & group);
            const int nw = __popcll(__ballot(live && xw < mw * 1.0001e-4f) & group);
            const bool out = mk > 3e38f || mw > 3e38f || (tk != 0.0 && mk < 1e-30f) || (tw != 0.0 && mw < 1e-30f);
            if (__any(nk > k1 || nw > k1 || (live && out))) {
                double* const sx = s_x[wid] + h * NS * 2;
                double* const sm = s_med[wid] + h * 4;
                if (live) {
                    sx[s * 2] = fabs(tk);
                    sx[s * 2 + 1] = fabs(tw);
                }
                if (tl < 4) sm[tl] = -1.0;
                wave_sync();
                if (live) {   // rank of the lane's two values among the finite ones of their field
                    for (int f = 0; f < 2; ++f) {
                        const double x = fabs(f ? tw : tk);
                        int lt = 0, le = 0;
                        for (int q = 0; q < NS; ++q) {
                            lt += sx[q * 2 + f] < x;
                            le += sx[q * 2 + f] <= x;
                        }
                        if (lt <= k1 && k1 < le) sm[f * 2] = x;         // equal values write the same
                        if (lt <= k2 && k2 < le) sm[f * 2 + 1] = x;
                    }
                }
                wave_sync();
                if (live) {
                    for (int f = 0; f < 2; ++f) {
                        const double m1 = sm[f * 2], m2 = sm[f * 2 + 1];
                        if (m1 < 0.0 || m2 < 0.0) continue;             // NaN median: nothing zeroed
                        double um = 0.0;
                        for (int q = 0; q < NS; ++q) um += fabs((double)(f ? a.w : a.k)[cell * NS + q]);
                        double ref = nan_max((NS % 2) ? m1 : 0.5 * (m1 + m2), 1e-9 * (um / NS));
                        ref = nan_max(ref, Tiny<double>::v);
                        if (fabs(f ? tw : tk) > 1e4 * ref) (f ? tw : tk) = 0.0;
                    }
                }
                wave_sync();   // k and omega are read by every lane before any is updated
            }
        }
        if (!isfinite(tk)) tk = 0.0;
        if (!isfinite(tw)) tw = 0.0;
        if (live) {
            const double dt = (double)dtr, k = (double)kr, w = (double)wr;
            const double wsafe = dmax(w, 1e-10);
            double dk = (double)s0 / (1.0 + dt * BSTAR * wsafe);
            double dw = (double)s1 / (1.0 + dt * (double)s2 * wsafe);
            dk = finite_or(dk, 0.0) + tk;
            dw = finite_or(dw, 0.0) + tw;
            dk = finite_or(dk, 0.0);
            dw = finite_or(dw, 0.0);
            if (a.rates) {
                // residual evaluation only: dk/dt and domega/dt of the update, fields untouched
                *reinterpret_cast<v2*>(a.rates + i * 2) = (v2){(real)dk, (real)dw};
            } else {
                double kn = k + dt * dk, wn = w + dt * dw;
                kn = isfinite(kn) ? kn : 1e-12;
                wn = isfinite(wn) ? wn : 1e-12;
                a.k[i] = (real)dmax(kn, 1e-12);
                a.w[i] = (real)dmax(wn, 1e-12);
            }
        }
    }
}

// nearest wall node (FP64 brute force, wall nodes staged through LDS)
template <typename real>
__global__ void __launch_bounds__(256) k_wall_distance(const double* __restrict__ xyz, int64_t n,
                                                       const double* __restrict__ wall, int n_wall, real* out) {
    __shared__ double s_w[256 * 3];
    for (int64_t base = (int64_t)blockIdx.x * 256; base < n; base += (int64_t)gridDim.x * 256) {
        const int64_t i = base + threadIdx.x;
        double x = 0, y = 0, z = 0;
        if (i < n) {
            x = xyz[i * 3 + 0];
            y = xyz[i * 3 + 1];
            z = xyz[i * 3 + 2];
        }
        double best = 1e300;
        for (int w0 = 0; w0 < n_wall; w0 += 256) {
            __syncthreads();
            const int m = n_wall - w0 < 256 ? n_wall - w0 : 256;
            if (threadIdx.x < m) {
                s_w[threadIdx.x * 3 + 0] = wall[(int64_t)(w0 + threadIdx.x) * 3 + 0];
                s_w[threadIdx.x * 3 + 1] = wall[(int64_t)(w0 + threadIdx.x) * 3 + 1];
                s_w[threadIdx.x * 3 + 2] = wall[(int64_t)(w0 + threadIdx.x) * 3 + 2];
            }
            __syncthreads();
            for (int j = 0; j < m; ++j) {
                const double dx = x - s_w[j * 3 + 0], dy = y - s_w[j * 3 + 1], dz = z - s_w[j * 3 + 2];
                const double d2 = dx * dx + dy * dy + dz * dz;
                best = d2 < best ? d2 : best;
            }
        }
        if (i < n) out[i] = (real)sqrt(best);
    }
}

template <int P, int CT, typename real>
int launch_sst_cell(const SstArgs<real>& a, hipStream_t st) {
    if (a.n_cells <= 0) return 0;
    const int64_t units = (a.n_cells + SO<P, CT>::CPW - 1) / SO<P, CT>::CPW;
    hipLaunchKernelGGL((k_sst_cell<P, CT, real>), dim3((unsigned)walk_grid(units, kWaves, a.grid_cap > 0 ? a.grid_cap : 4096)),
                       dim3(64 * kWaves), 0, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int P, typename real>
int launch_sst_face(const SstArgs<real>& a, hipStream_t st) {
    if (a.n_records <= 0) return 0;
    const int64_t n = a.n_records * (P + 1) * (P + 1);
    const int64_t need = (n + 255) / 256;
    constexpr int KS = (P + 1) * (P + 1), NS = KS * (P + 1);
    const int64_t cap = a.grid_cap_face > 0 ? a.grid_cap_face : 8192;
    const dim3 grid((unsigned)(need < cap ? need : cap));
    if (a.knz == KS)
        hipLaunchKernelGGL((k_sst_face<P, KS, real>), grid, dim3(256), 0, st, a);
    else if (a.knz == NS)
        hipLaunchKernelGGL((k_sst_face<P, NS, real>), grid, dim3(256), 0, st, a);
    else
        return -1;
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int P, int CT, typename real>
int launch_sst_update(const SstArgs<real>& a, hipStream_t st) {
    if (a.n_cells <= 0) return 0;
    const int64_t units = (a.n_cells + SO<P, CT>::CPW - 1) / SO<P, CT>::CPW;
    hipLaunchKernelGGL((k_sst_update<P, CT, real>), dim3((unsigned)walk_grid(units, kWaves, a.grid_cap > 0 ? a.grid_cap : 4096)),
                       dim3(64 * kWaves), 0, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_wall_distance(const double* sp_xyz, int64_t n_pts, const double* wall_xyz, int n_wall, void* d_out,
                         int dtype, hipStream_t st) {
    const int64_t need = (n_pts + 255) / 256;
    const dim3 grid((unsigned)(need < 16384 ? (need > 0 ? need : 1) : 16384));
    if (dtype == AFR_F32)
        hipLaunchKernelGGL((k_wall_distance<float>), grid, dim3(256), 0, st, sp_xyz, n_pts, wall_xyz, n_wall,
                           (float*)d_out);
    else
        hipLaunchKernelGGL((k_wall_distance<double>), grid, dim3(256), 0, st, sp_xyz, n_pts, wall_xyz, n_wall,
                           (double*)d_out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

#define AFR_SST_INST(P, CT, T)                                                  \
    template int launch_sst_cell<P, CT, T>(const SstArgs<T>&, hipStream_t);     \
    template int launch_sst_update<P, CT, T>(const SstArgs<T>&, hipStream_t);
AFR_SST_INST(1, 0, float)
AFR_SST_INST(2, 0, float)
AFR_SST_INST(1, 1, float)
AFR_SST_INST(2, 1, float)
AFR_SST_INST(1, 0, double)
AFR_SST_INST(2, 0, double)
AFR_SST_INST(1, 1, double)
AFR_SST_INST(2, 1, double)
template int launch_sst_face<1, float>(const SstArgs<float>&, hipStream_t);
template int launch_sst_face<2, float>(const SstArgs<float>&, hipStream_t);
template int launch_sst_face<1, double>(const SstArgs<double>&, hipStream_t);
template int launch_sst_face<2, double>(const SstArgs<double>&, hipStream_t);

}  // namespace afr_sst
