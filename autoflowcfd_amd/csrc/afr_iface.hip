// Interface terms of the mean-flow residual (gfx950): AUSM+up and BR1 jumps of every face slot,
// their distribution into the cell, division by det J, outlier zeroing, the residual.
//
// Reference semantics: src/autoflowcfd/core/fr_residual/inviscid_kernel.py:87-284,
// src/autoflowcfd/core/fr_residual/viscous_flux_kernel.py:59-289,
// src/autoflowcfd/core/fr_operators/troubled_cell.py:339-408.
//
// A workgroup of four waves takes CPT cells at a time, lane = (slot, cell, flux point), slot by slot
// (lane maps in IF).  An own trace takes N1 points on a faces and on a prism's c faces, N1^2 on b
// faces, all on a tet's c face.  The own packs are staged in LDS (every
// point is read by several slots); the other side is gathered from global memory by the slot's
// interpolation rows.  The jumps meet in LDS, from where one thread per solution point distributes
// them; the outlier test runs on the residual in LDS, one lane per (cell, variable).
//
// Bound: latency of the gathers (VALU issue takes about half of the time, HBM traffic 8.2 GB at 82^3 P2
// FP32).  What this form is there for: one set of traces, slot tables and one residual write serve both
// jumps, four resident waves per SIMD at no spill, the next tile's tables and own points in flight while
// this one computes.  Tried and slower: five waves per workgroup with one slot per wave (2 or 3 resident
// workgroups, uneven SIMDs: 5.0 ms), a lane's gather of all 15 values on its own instead of four lanes
// sharing 16-byte loads (4.1 ms), a budget of five waves per SIMD (spills).
// Measured (82^3 hex, 1.1 M prisms, P2 FP32): 2.43 ms; two kernels before, 2.88 ms for the viscous jumps
// and about half of 2.98 ms for the inviscid ones.  304k P1 prisms FP32 254 us (401 + half of 1014).
// P2 and P3 tets FP64: see the matrix products below.
#include <hip/hip_runtime.h>

#include <type_traits>

// Products are fused with the sums of their own expression only.  Fused wherever the optimiser meets a
// pair, which it meets depends on the form of the kernel (row width, index width), and a case in a batch,
// whose rows are padded to the widest of the batch, would differ from itself alone in the last bits.
#pragma clang fp contract(on)

#include "../../include/afr.h"
#include "afr_meanflow.hpp"
#include "afr_outlier.hpp"
#include "afr_physics.hpp"

using namespace afr;

namespace afr_mean {

template <int P, int CT, typename real, bool INV, bool VISC> struct IF {
    static constexpr int N1 = P + 1, NS = N1 * N1 * N1, NFP = N1 * N1, NSLOT = CT == 0 ? 5 : 4;
    // cells of a tile, and the lane stride of a slot's block of (cell, flux point) lanes: tets one wave
    // per slot (P1 16 cells, P2 7, P3 4), prisms the five blocks back to back in four waves (P1 12
    // cells, 240 of 256 lanes; P2 5 cells, 225)
    static constexpr int NT = 256, CPT = CT == 0 ? NT / (NSLOT * NFP) : 64 / NFP, IPS = CT == 0 ? CPT * NFP : 64;
    static constexpr int NP = VISC ? kPackUsed : 5;             // values of a trace
    static constexpr int PS = VISC ? kPack + 4 : 5;             // LDS stride of an own point
    static constexpr int NI = INV ? 5 : 0, NV = VISC ? 4 : 0, NR = NI + NV;   // jump / residual values
    static constexpr int JS = NR | 1;
    static constexpr int KW = N1 * N1;                          // own-row weights kept in LDS
    static constexpr int N_OWN = CPT * NS * PS, N_J = CPT * NSLOT * NFP * JS, N_RES = CPT * NS * NR;
    static constexpr int N_MMA = CT == 1 && P >= 2 && VISC && sizeof(real) == 8 ? 4 * 16 * 17 : 0;   // products of the waves
    static constexpr int N_A = N_RES > N_MMA ? N_RES : N_MMA;
    // 16-byte chunks (viscous pack) or values (dQ) of a tile's own points, and how many a thread stages
    static constexpr int N_ST = CPT * NS * (VISC ? kPack / 4 : 5), SQ = (N_ST + NT - 1) / NT;
    static constexpr int WPE = sizeof(real) == 4 ? 4 : 2;       // waves per SIMD the registers are budgeted for
};

// face code of a slot: prism a=-1, a=+1, b=-1, c=-1, c=+1; tet a=-1, a=+1, b=-1, c=-1
__device__ __forceinline__ int face_code(int slot) { return slot < 3 ? slot : slot + 1; }

// Element numbers into the mesh arrays: 32-bit byte offsets from a scalar base (one VALU
// instruction per address) where the largest array is under 4 GiB, 64-bit ones otherwise.
template <bool BIG> struct Index { typedef uint32_t type; };
template <> struct Index<true> { typedef int64_t type; };
template <bool BIG, typename T>
__device__ __forceinline__ T at(const T* p, typename Index<BIG>::type i) {
    if constexpr (BIG) return ((GlobalPtr<T>)p)[i];
    else return *(GlobalPtr<T>)((GlobalPtr<char>)p + (uint32_t)(i * (uint32_t)sizeof(T)));
}
// cell * n (+ ...): 24-bit multiplication where the cell count allows it
template <bool BIG> __device__ __forceinline__ typename Index<BIG>::type times(int cell, int n) {
    if constexpr (BIG) return (int64_t)cell * n;
    else return __umul24((unsigned)cell, (unsigned)n);
}

// ---- gather of pack points from global memory by quads of lanes
// A pack point is four 16-byte chunks (32-byte in FP64).  If every lane read the four chunks of its
// own point, each load instruction would touch 64 cache lines and the four of them the same lines
// again while they are still on their way.  Instead lane i of a quad reads chunk i of the points of
// all four lanes (a load instruction then touches 16 whole points) and accumulates that chunk for
// all four; one transposition per trace brings every lane its own 16 values.
template <int J> __device__ __forceinline__ int quad_lane(int x) {
    return __builtin_amdgcn_update_dpp(0, x, J * 0x55, 0xf, 0xf, true);
}
template <int J> __device__ __forceinline__ float quad_lane(float x) {
    return __int_as_float(quad_lane<J>(__float_as_int(x)));
}
template <int J> __device__ __forceinline__ double quad_lane(double x) {
    return __hiloint2double(quad_lane<J>(__double2hiint(x)), quad_lane<J>(__double2loint(x)));
}
template <int M> __device__ __forceinline__ int quad_xor(int x) {   // value of lane ^ M, M = 1 or 2
    return __builtin_amdgcn_update_dpp(0, x, M == 1 ? 0xB1 : 0x4E, 0xf, 0xf, true);
}
template <int M> __device__ __forceinline__ float quad_xor(float x) {
    return __int_as_float(quad_xor<M>(__float_as_int(x)));
}
template <int M> __device__ __forceinline__ double quad_xor(double x) {
    return __hiloint2double(quad_xor<M>(__double2hiint(x)), quad_xor<M>(__double2loint(x)));
}

// acc[j] += (weight of lane j of the quad) x (chunk i of lane j's point), for N points; pt: this
// lane's point numbers, w its weights (0 and any valid point where it has none)
template <int N, bool BIG, typename real>
__device__ __forceinline__ void quad_gather(typename V4<real>::type acc[4], const real* pack,
                                            const typename Index<BIG>::type* pt, const real* w, int i) {
    typedef typename V4<real>::type v4;
    constexpr uint32_t PB = kPack * sizeof(real);
    v4 x[N][4];
#pragma unroll
    for (int k = 0; k < N; ++k) {
        if constexpr (BIG) {
            const int lo = (int)(uint32_t)pt[k], hi = (int)(pt[k] >> 32);
#define AFR_QUAD_LOAD(J)                                                                                        \
    x[k][J] = *(GlobalPtr<v4>)((GlobalPtr<char>)pack +                                                         \
                               ((int64_t)quad_lane<J>(hi) << 32 | (uint32_t)quad_lane<J>(lo)) * PB + (PB / 4) * i);
            AFR_QUAD_LOAD(0) AFR_QUAD_LOAD(1) AFR_QUAD_LOAD(2) AFR_QUAD_LOAD(3)
#undef AFR_QUAD_LOAD
        } else {
            const int off = (int)(pt[k] * PB);
#define AFR_QUAD_LOAD(J)                                                                                        \
    x[k][J] = *(GlobalPtr<v4>)((GlobalPtr<char>)pack + (uint32_t)(quad_lane<J>(off) + (int)(PB / 4) * i));
            AFR_QUAD_LOAD(0) AFR_QUAD_LOAD(1) AFR_QUAD_LOAD(2) AFR_QUAD_LOAD(3)
#undef AFR_QUAD_LOAD
        }
    }
#pragma unroll
    for (int k = 0; k < N; ++k) {
        acc[0] += quad_lane<0>(w[k]) * x[k][0];
        acc[1] += quad_lane<1>(w[k]) * x[k][1];
        acc[2] += quad_lane<2>(w[k]) * x[k][2];
        acc[3] += quad_lane<3>(w[k]) * x[k][3];
    }
}

// out[4 c + e] of lane j = acc[j][e] of lane c of the quad
template <typename real>
__device__ __forceinline__ void quad_transpose(const typename V4<real>::type acc[4], real* out, int i) {
    const bool b0 = i & 1, b1 = i & 2;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        // (every exchange by all lanes, then the selection)
        const real x0 = quad_xor<1>(acc[0][e]), x1 = quad_xor<1>(acc[1][e]);
        const real x2 = quad_xor<1>(acc[2][e]), x3 = quad_xor<1>(acc[3][e]);
        const real t0 = b0 ? x1 : acc[0][e], t1 = b0 ? acc[1][e] : x0;
        const real t2 = b0 ? x3 : acc[2][e], t3 = b0 ? acc[3][e] : x2;
        const real y0 = quad_xor<2>(t0), y1 = quad_xor<2>(t1), y2 = quad_xor<2>(t2), y3 = quad_xor<2>(t3);
        out[e] = b1 ? y2 : t0;
        out[4 + e] = b1 ? y3 : t1;
        out[8 + e] = b1 ? t2 : y0;
        out[12 + e] = b1 ? t3 : y1;
    }
}

// acc[q] += w x[q] of one own point (LDS)
template <int NP, typename real>
__device__ __forceinline__ void add_point(real* acc, real w, const real* x) {
    if constexpr (NP == kPackUsed) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const typename V4<real>::type f = ld4(x + 4 * c);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (4 * c + e < NP) acc[4 * c + e] += w * f[e];
        }
    } else {
#pragma unroll
        for (int q = 0; q < NP; ++q) acc[q] += w * x[q];
    }
}

// A . G of the viscous flux from a trace (values 1..3 of q: velocity; g: S (6), grad T (3), mu_t)
template <typename real>
__device__ __forceinline__ void visc_dot(const real* q, const real* g, real mu, real Pr, real Prt, const real A[3],
                                         real out[4]) {
    const real mut = g[9], mt = mu + mut;
    const real lam = real(-1.0 / 3.0) * mt * (g[0] + g[1] + g[2]);
    const real S[3][3] = {{g[0], g[3], g[4]}, {g[3], g[1], g[5]}, {g[4], g[5], g[2]}};
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        real acc = lam * A[j];
#pragma unroll
        for (int i = 0; i < 3; ++i) acc += A[i] * (mt * S[i][j]);
        out[j] = acc;
    }
    const real cp = real(kGamma * kRair / (kGamma - 1.0));
    const real k = mu * cp / Pr + mut * cp / Prt;
    out[3] = q[1] * out[0] + q[2] * out[1] + q[3] * out[2] - k * (A[0] * g[6] + A[1] * g[7] + A[2] * g[8]);
}

// ---- traces of FP64 tets at P2 and P3 as matrix products
// Own rows are dense and source rows up to NS wide: per (cell, slot) both traces are products of 16 flux
// points x NS points x 16 pack values, on the matrix cores.  The own rows' fragments stay in registers (a
// wave has one slot); the interpolation rows are laid out as fragments [block][step][lane] in a scratch
// array at the start of every call (a few blocks of NFP rows: 5 us).
template <int P> struct FR {
    static constexpr int N1 = P + 1, NS = N1 * N1 * N1, NFP = N1 * N1, KS = (NS + 3) / 4;
};
template <int P>
__global__ void __launch_bounds__(256) k_row_fragments(const int* nnz, const int* idx, const double* w, int knz, int n_rows,
                                                       double* out) {
    using L = FR<P>;
    __shared__ double s_r[16 * (4 * L::KS + 1)];   // a block's rows, dense
    constexpr int LD = 4 * L::KS + 1;
    const int blocks = (n_rows + L::NFP - 1) / L::NFP;
    for (int b = blockIdx.x; b < blocks; b += gridDim.x) {
        for (int q = threadIdx.x; q < 16 * LD; q += 256) s_r[q] = 0.0;
        __syncthreads();
        for (int q = threadIdx.x; q < L::NFP * knz; q += 256) {
            const int r = b * L::NFP + q / knz, e = q % knz;
            if (r < n_rows && e < nnz[r]) s_r[q / knz * LD + idx[(int64_t)r * knz + e]] = w[(int64_t)r * knz + e];
        }
        __syncthreads();
        for (int q = threadIdx.x; q < L::KS * 64; q += 256) {
            const int l = q % 64;
            out[(int64_t)b * (L::KS * 64) + q] = s_r[l % 16 * LD + 4 * (q / 64) + l / 16];
        }
        __syncthreads();
    }
}

template <int P, int CT, int KMAX, typename real, bool INV, bool VISC, bool BIG, bool MMA>
__global__ void __launch_bounds__((IF<P, CT, real, INV, VISC>::NT))
    __attribute__((amdgpu_waves_per_eu(IF<P, CT, real, INV, VISC>::WPE))) k_iface(MeanArgs<real> args) {
    using L = IF<P, CT, real, INV, VISC>;
    using Idx = typename Index<BIG>::type;
    using v4 = typename V4<real>::type;
    constexpr int N1 = L::N1, NS = L::NS, NFP = L::NFP, NSLOT = L::NSLOT, CPT = L::CPT, NT = L::NT;
    constexpr int NP = L::NP, PS = L::PS, NI = L::NI, NR = L::NR, JS = L::JS, KW = L::KW;
    // tets at P2 and P3: every own row is dense (the round-off entries of the collapsed basis reach
    // 1e-12 there at P2, 1e-7 at P3; outlier decisions next to a jump see them)
    constexpr bool DENSE = CT == 1 && P >= 2;
    constexpr int ROWS_CAP = CT == 0 && KMAX == N1 * N1 ? 8 * NFP : 1;
    __shared__ __attribute__((aligned(16))) real s_own[L::N_OWN];
    __shared__ real s_a[L::N_A];
    __shared__ real s_j[L::N_J];
    __shared__ real s_rw[ROWS_CAP * KMAX];
    __shared__ uint8_t s_ri[ROWS_CAP * KMAX];   // bit 7 of a row's first: it has more than N1 non-zeros
    __shared__ real s_ew[DENSE ? 1 : NSLOT * NFP * KW];   // own-trace weights
    __shared__ real s_med[2][CPT * NR];
    __shared__ int s_list[CPT * NR], s_bad;    // columns (cell, value) that need their median, how many
    __shared__ int s_cell[2][CPT];             // cells of this tile and of the next
    const int tid = threadIdx.x;
    // The arguments are read anew in every stage (fresh()): held over the tile loop, some 90 scalar
    // registers of pointers and constants would be spilled to vector lanes and read back from there.
    typedef const __attribute__((address_space(4))) MeanArgs<real> Args;
    Args* const kernarg = (Args*)__builtin_amdgcn_kernarg_segment_ptr();
    auto fresh = [&]() -> Args* {
        Args* p = kernarg;
        asm volatile("" : "+s"(p));
        return p;
    };
    // the deduplicated interpolation rows in LDS when the mesh has few blocks (8 for a graded
    // prism box; a batch of cases or a tet mesh has more and reads them from global memory)
    const int n_rows = args.n_rows;
    const bool rows_lds = ROWS_CAP > 1 && n_rows <= ROWS_CAP;
    if (rows_lds) {
#pragma unroll
        for (int u = 0; u < (ROWS_CAP * KMAX + NT - 1) / NT; ++u) {
            const int q = tid + u * NT, r = q / KMAX;
            if (r < n_rows) {
                const int i = args.rows_idx[q], nnz = args.rows_nnz[r];
                s_rw[q] = args.rows_w[q];
                s_ri[q] = (uint8_t)(i | (q == r * KMAX && nnz > N1 ? 128 : 0));
            }
        }
    }
    if (tid == 0) s_bad = 0;
    // Lane role, packed: slot, cell of the tile, flux point, in use.  The prism blocks are ordered with
    // the b face last, so that the waves with its wider own rows are not those with the (usually) wider
    // neighbour rows.
    struct Role {
        int slot, lc, fp;
        bool in;
    };
    int role_bits;
    {
        const int pos = tid / L::IPS, r = tid % L::IPS;
        const int slot = CT == 0 ? (pos == 4 ? 2 : pos + (pos >> 1)) : pos;
        role_bits = pos < NSLOT && r / NFP < CPT ? slot | (r / NFP) << 3 | (r % NFP) << 8 | 1 << 13 : 0;
    }
    auto role = [&]() -> Role { return {role_bits & 7, (role_bits >> 3) & 31, (role_bits >> 8) & 31, role_bits != 0}; };
    // MMA: fragments of this wave's own rows
    double fe[MMA ? FR<P>::KS : 1];
    if constexpr (MMA) {
#pragma unroll
        for (int k = 0; k < FR<P>::KS; ++k) {
            const int f = tid & 15, s = 4 * k + ((tid >> 4) & 3);
            fe[k] = f < NFP && s < NS ? args.E[((int64_t)(tid >> 6) * NFP + f) * NS + s] : 0.0;
        }
    }
    // own-trace rows: base + k step, k < kt (DENSE: every point)
    auto own_base = [&](int axis, int f) { return axis == 0 ? f : (axis == 1 ? f % N1 : (CT == 0 ? f * N1 : 0)); };
    auto own_step = [&](int axis) { return axis == 0 ? N1 * N1 : (axis == 1 ? N1 : 1); };
    if constexpr (!DENSE) {
        for (int q = tid; q < NSLOT * NFP * KW; q += NT) {
            const int sf = q / KW, k = q % KW, ax = face_code(sf / NFP) >> 1;
            s_ew[q] = k < (ax == 1 || CT == 1 ? KW : N1)
                          ? args.E[(int64_t)sf * NS + own_base(ax, sf % NFP) + k * own_step(ax)] : real(0);
        }
    }
    // solution point of a distribution thread, packed: cell of the tile, point
    const int dist_bits = tid / NS | (tid % NS) << 8;
    // chunks (viscous pack) or values (dQ) of the own points staged by a thread: cell, place in the cell
    int stage_bits[L::SQ];
#pragma unroll
    for (int q = 0; q < L::SQ; ++q) {
        const int o = tid + q * NT < L::N_ST ? tid + q * NT : L::N_ST - 1, per = L::N_ST / CPT;
        stage_bits[q] = o / per | (o % per) << 8;
    }

    // Where a lane takes its other side from: the boundary code, the source cell and the interpolation
    // row (-1: none).
    struct Slot {
        int mask, bc, blk0, blk1, nb0, nb1;
    };
    auto load_slot = [&](int cell, int slot) -> Slot {
        Args* a = fresh();
        Slot x;
        const Idx sidx = times<BIG>(cell, 5) + slot;
        x.mask = at<BIG>(a->slot_mask, sidx);
        x.bc = at<BIG>(a->slot_bc, sidx);
        x.blk0 = at<BIG>(a->slot_blk, sidx * 2);
        x.blk1 = at<BIG>(a->slot_blk, sidx * 2 + 1);
        x.nb0 = at<BIG>(a->slot_nb, sidx * 2);
        x.nb1 = at<BIG>(a->slot_nb, sidx * 2 + 1);
        return x;
    };
    int bc = 0, nb = 0, row = -1;
    auto take_slot = [&](const Slot& x, int fp) {
        const bool second = (x.mask >> fp) & 1;
        bc = x.bc;
        nb = second ? x.nb1 : x.nb0;
        row = (second ? x.blk1 : x.blk0) * NFP + fp;
        if (bc != BC_INTERIOR || nb < 0 || row < 0 || row >= n_rows) row = -1;
    };
    // cell of list position p (the last cell for lanes and tiles past the end)
    auto cell_at = [&](int64_t p) -> int {
        Args* a = fresh();
        const int64_t q = p < a->n_cells ? p : a->n_cells - 1;
        return (int)a->cell_begin + (a->schedule ? at<BIG>(a->schedule, (Idx)q) : (int)q);
    };

    // The slot table and the own points of a tile are loaded during the last stages of the tile before
    // it, and its cell numbers one tile earlier still: at the top of a tile the neighbour gather starts
    // at once instead of after four dependent round trips.
    const int64_t n_cells = args.n_cells, n_tiles = (n_cells + CPT - 1) / CPT;
    CellWalk cw(n_tiles, 1, 0);
    if (cw.it >= cw.hi) return;
    int cell, next_cell;
    {
        const Role x = role();
        cell = cell_at(cw.it * CPT + x.lc);
        next_cell = cell_at((cw.it + cw.step) * CPT + x.lc);
        take_slot(load_slot(cell, x.slot), x.fp);
        if (x.in && x.slot == 0 && x.fp == 0) s_cell[0][x.lc] = cell;
    }
    __syncthreads();
    // own points of a tile: global -> registers -> LDS
    typedef typename std::conditional<VISC, v4, real>::type Stg;
    Stg stg[L::SQ];
    auto load_own = [&](const int* cells) {
        Args* a = fresh();
#pragma unroll
        for (int q = 0; q < L::SQ; ++q) {
            const int c = cells[stage_bits[q] & 255], r = stage_bits[q] >> 8;
            if constexpr (VISC) stg[q] = at<BIG>((const v4*)a->pack, times<BIG>(c, NS * 4) + r);
            else stg[q] = at<BIG>(a->dQ, times<BIG>(c, NS * 5) + r);
        }
    };
    auto store_own = [&]() {
#pragma unroll
        for (int q = 0; q < L::SQ; ++q) {
            const int o = tid + q * NT;
            if (o < L::N_ST) {
                if constexpr (VISC) st4(s_own + (o >> 2) * PS + (o & 3) * 4, stg[q]);
                else s_own[o] = stg[q];
            }
        }
    };
    load_own(s_cell[0]);
    store_own();
    __syncthreads();
    for (int buf = 0; cw.it < cw.hi; cw.it += cw.step, buf ^= 1) {
        const int64_t left = n_cells - cw.it * CPT;
        const int nc = (int)(left < CPT ? left : CPT);
        const int* const cells = s_cell[buf];
        const Role me = role();
        const int slot = me.slot, lc = me.lc, fp = me.fp, code = face_code(slot), axis = code >> 1;
        const bool on = me.in && lc < nc;
        const bool inner = bc == BC_INTERIOR, have = on && row >= 0;
        if (me.in && slot == 0 && fp == 0) s_cell[buf ^ 1][lc] = next_cell;
        real A[3];
        bool fb = false;
        real pn[VISC ? kPack : 5], po[NP];
#pragma unroll
        for (int q = 0; q < NP; ++q) po[q] = real(0);
        if constexpr (MMA) {
            constexpr int KS = FR<P>::KS;
            const int t = tid & 63, ln = t & 15, lk = t >> 4;
            double* const st = s_a + (tid >> 6) * (16 * 17);   // the results' place is free until the distribution
            auto point = [&](int k) { return 4 * k + lk < NS ? 4 * k + lk : NS - 1; };   // past the end: times zero
            auto put = [&](d4 x) {   // product -> [flux point][value]
#pragma unroll
                for (int e = 0; e < 4; ++e) st[(4 * e + lk) * 17 + ln] = x[e];
                wave_sync();
            };
#pragma unroll
            for (int q = 0; q < kPack; ++q) pn[q] = 0.0;
#pragma unroll 1
            for (int c = 0; c < nc; ++c) {
                // sources of this cell's slot: one, or two where a face meets two cells
                uint64_t todo = __ballot(have && lc == c);
                double xa[KS], xb[KS];
                int s_nb = 0, s_blk = 0;
                auto fetch = [&]() {
                    const int lead = __builtin_amdgcn_readfirstlane(__ffsll((unsigned long long)todo) - 1);
                    s_nb = __builtin_amdgcn_readlane(nb, lead);
                    s_blk = __builtin_amdgcn_readlane((row - fp) / NFP, lead);
                    Args* a = fresh();
                    GlobalPtr<double> wf = (GlobalPtr<double>)a->work + (int64_t)s_blk * (KS * 64);
                    GlobalPtr<double> pk = (GlobalPtr<double>)a->pack + (int64_t)s_nb * (NS * kPack);
#pragma unroll
                    for (int k = 0; k < KS; ++k) {
                        xa[k] = wf[k * 64 + t];
                        xb[k] = pk[point(k) * kPack + ln];
                    }
                };
                if (todo) fetch();
                d4 x = {0, 0, 0, 0};
                const double* own = s_own + c * NS * PS + ln;
#pragma unroll
                for (int k = 0; k < KS; ++k) x = mma(fe[k], own[point(k) * PS], x);
                put(x);
                if (on && lc == c) {
#pragma unroll
                    for (int q = 0; q < NP; ++q) po[q] = st[fp * 17 + q];
                }
                wave_sync();
                while (todo) {
                    x = (d4){0, 0, 0, 0};
#pragma unroll
                    for (int k = 0; k < KS; ++k) x = mma(xa[k], xb[k], x);
                    put(x);
                    const bool mine = (todo >> t & 1) && nb == s_nb && (row - fp) / NFP == s_blk;
                    if (mine) {
#pragma unroll
                        for (int q = 0; q < NP; ++q) pn[q] = st[fp * 17 + q];
                    }
                    todo &= ~__ballot(mine);
                    wave_sync();
                    if (todo) fetch();
                }
            }
            Args* a = fresh();
            const Idx sidx = times<BIG>(cell, 5) + slot;
            const Idx ai = (sidx * NFP + fp) * 3;
#pragma unroll
            for (int q = 0; q < 3; ++q) A[q] = at<BIG>(a->slot_adjrow, ai + q);
            if constexpr (INV) fb = (at<BIG>(a->slot_fb, sidx) >> fp) & 1;
            // a product also takes the points that a row does not name, with weights of zero: where the trace
            // is not finite, it is summed over its row's own points
            real size = 0;
#pragma unroll
            for (int q = 0; q < NP; ++q) size += fabs(pn[q]);
            if (have && !(size < __builtin_huge_val())) {
#pragma unroll
                for (int q = 0; q < NP; ++q) pn[q] = real(0);
                const int nnz = at<BIG>(a->rows_nnz, (Idx)row);
#pragma unroll 1
                for (int k = 0; k < nnz; ++k) {
                    const Idx e = (Idx)row * KMAX + k;
                    const real w = at<BIG>(a->rows_w, e);
                    const int64_t p = ((int64_t)nb * NS + at<BIG>(a->rows_idx, e)) * kPack;
#pragma unroll
                    for (int q = 0; q < NP; ++q) pn[q] += w * ((GlobalPtr<real>)a->pack)[p + q];
                }
            }
        } else {
            Args* a = fresh();
            const Idx sidx = times<BIG>(cell, 5) + slot;
            const Idx ai = (sidx * NFP + fp) * 3;
#pragma unroll
            for (int q = 0; q < 3; ++q) A[q] = at<BIG>(a->slot_adjrow, ai + q);
            if constexpr (INV) fb = (at<BIG>(a->slot_fb, sidx) >> fp) & 1;
            // 1. the other side's trace (the rows hold their non-zeros first); lanes without a source join the
            //    loads of their quad with the first row and weights of zero (chosen after the loads: chosen by a
            //    branch around them, a mixed P1 evaluation took 270 us, 265 so)
            const int r = have ? row : 0;
            const Idx p0 = times<BIG>(have ? nb : 0, NS);
            const int qi = tid & 3;
            auto row_entry = [&](int kk, int& i, real& w) {
                if (rows_lds) {
                    i = s_ri[r * KMAX + kk];
                    w = s_rw[r * KMAX + kk];
                } else {
                    i = at<BIG>(a->rows_idx, (Idx)r * KMAX + kk);
                    w = at<BIG>(a->rows_w, (Idx)r * KMAX + kk);
                }
            };
            v4 acc[4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
            if constexpr (!VISC) {
#pragma unroll
                for (int q = 0; q < 5; ++q) pn[q] = real(0);
            }
            bool wide = false;    // more than N1 non-zeros (known with the first terms; rows of prism sources)
            auto terms = [&](int k0, auto first) {
                Idx pt[N1];
                real w[N1];
#pragma unroll
                for (int k = 0; k < N1; ++k) {
                    const int kk = KMAX % N1 == 0 || k0 + k < KMAX ? k0 + k : KMAX - 1;
                    int i;
                    row_entry(kk, i, w[k]);
                    if (decltype(first)::value && k == 0 && KMAX == N1 * N1) {
                        wide = rows_lds ? i & 128 : have && at<BIG>(a->rows_nnz, (Idx)r) > N1;
                        if (rows_lds) i &= 127;
                    }
                    pt[k] = p0 + i;
                    if (!have || kk != k0 + k) w[k] = real(0);
                }
                if constexpr (VISC) {
                    quad_gather<N1, BIG, real>(acc, a->pack, pt, w, qi);
                } else {
#pragma unroll
                    for (int k = 0; k < N1; ++k)
#pragma unroll
                        for (int q = 0; q < 5; ++q) pn[q] += w[k] * at<BIG>(a->dQ, pt[k] * 5 + q);
                }
            };
            // A table without rows is not read.  As a branch this also keeps the loads before it out of the gather:
            // kernel on 1.1 M P2 prisms FP32 2755 -> 2435 us, 304k P1 prisms 266 -> 254
            if (n_rows > 0) terms(0, std::true_type());
            // further terms: the quads with a wide row (prism sources), or every lane up to the widest
            // row of the wave (dense rows of tet sources)
            if constexpr (KMAX == N1 * N1) {
                if ((__ballot(have && wide) >> (tid & 60)) & 15) {
#pragma unroll 1
                    for (int k0 = N1; k0 < KMAX; k0 += N1) terms(k0, std::false_type());
                }
            } else {
                const int nnz = have ? at<BIG>(a->rows_nnz, (Idx)r) : 0;
                const int kn = __any(nnz > N1 * N1) ? KMAX : (__any(nnz > N1) ? N1 * N1 : N1);
#pragma unroll 1
                for (int k0 = N1; k0 < kn; k0 += N1) terms(k0, std::false_type());
            }
            if constexpr (VISC) quad_transpose<real>(acc, pn, qi);
        }
        // 2. jumps
        if (on && bc != -2) {
            Args* a = fresh();
            if constexpr (MMA) {
            } else if constexpr (DENSE) {
                const real* own = s_own + lc * NS * PS;
                const Idx e0 = (slot * NFP + fp) * NS;
#pragma unroll 2
                for (int k = 0; k < NS; ++k) add_point<NP>(po, at<BIG>(a->E, e0 + k), own + k * PS);
            } else {
                const real* own = s_own + (lc * NS + own_base(axis, fp)) * PS;
                const real* ew = s_ew + (slot * NFP + fp) * KW;
                const int sp = own_step(axis) * PS;
#pragma unroll
                for (int k = 0; k < N1; ++k) add_point<NP>(po, ew[k], own + k * sp);
                if (axis == 1 || (CT == 1 && axis == 2)) {
#pragma unroll
                    for (int k = N1; k < KW; ++k) add_point<NP>(po, ew[k], own + k * sp);
                }
                if (CT == 1 && axis == 2) {
                    const Idx e0 = (slot * NFP + fp) * NS;
#pragma unroll 2
                    for (int k = KW; k < NS; ++k) add_point<NP>(po, at<BIG>(a->E, e0 + k), own + k * PS);
                }
            }
            real* jo = s_j + ((lc * NSLOT + slot) * NFP + fp) * JS;
            double qo[5], qn[5];
            const double side = (code & 1) ? 1.0 : -1.0;
            double tn[3] = {0, 0, 0};
            if (!inner || fb) {
                const Idx ti = (times<BIG>(cell, 5) + slot) * 3;
#pragma unroll
                for (int q = 0; q < 3; ++q) tn[q] = (double)at<BIG>(a->slot_tn, ti + q);
            }
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                qo[v] = a->qref[v] + (double)po[v];
                qn[v] = a->qref[v] + (double)pn[v];
            }
            if (!inner) {
                const double* bcp = a->bcp + (a->cell_case ? 40 * (int64_t)((GlobalPtr<int>)a->cell_case)[cell] : 0);
                ghost_state(bc, qo, tn, bcp, qn);
            }
            if constexpr (VISC) {
                // BR1: A . (G(average) - G(own)); boundary slots mirror gradients and mu_t and take
                // the interior penalty on the momenta
                const real mu = (real)a->mu, Pr = (real)a->Pr, Prt = (real)a->Prt;
                real Qo[4], Qa[4];
#pragma unroll
                for (int v = 1; v < 4; ++v) {
                    Qo[v] = (real)qo[v];
                    Qa[v] = real(0.5) * (Qo[v] + (real)qn[v]);
                }
                real ga[10], fc[4], fo[4];
#pragma unroll
                for (int q = 0; q < 10; ++q) ga[q] = real(0.5) * (po[5 + q] + (inner ? pn[5 + q] : po[5 + q]));
                visc_dot(Qa, ga, mu, Pr, Prt, A, fc);
                visc_dot(Qo, po + 5, mu, Pr, Prt, A, fo);
#pragma unroll
                for (int v = 0; v < 4; ++v) fc[v] -= fo[v];
                if (!inner) {
                    real sum = 0;
                    for (int q = 0; q < NS; ++q) sum += at<BIG>(a->det, times<BIG>(cell, NS) + q);
                    real h = (real)cbrt((double)(sum / real(NS)));
                    h = h > Tiny<real>::v ? h : Tiny<real>::v;
                    const real mag = sqrt(A[0] * A[0] + A[1] * A[1] + A[2] * A[2]);
                    const real scale = real(4.0) * (mu + po[14]) / h * mag * (real)side;
#pragma unroll
                    for (int v = 1; v < 4; ++v) fc[v - 1] -= scale * (Qo[v] - (real)qn[v]);
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) jo[NI + v] = fc[v];
            }
            if constexpr (INV) {
                const double Av[3] = {(double)A[0], (double)A[1], (double)A[2]};
                double mag = sqrt_r(Av[0] * Av[0] + Av[1] * Av[1] + Av[2] * Av[2]);
                mag = mag > 1e-300 ? mag : 1e-300;
                const double im = side * recip(mag);
                double d[3], F[5], FA[5];
#pragma unroll
                for (int q = 0; q < 3; ++q) d[q] = fb ? tn[q] : Av[q] * im;
                euler_flux_dir(qo, Av, FA);
                ausm_up(qo, qn, d, F);
                const double sc = mag * side;
#pragma unroll
                for (int v = 0; v < 5; ++v) jo[v] = (real)(F[v] * sc - FA[v]);
            }
        } else if (on) {
#pragma unroll
            for (int v = 0; v < NR; ++v) s_j[((lc * NSLOT + slot) * NFP + fp) * JS + v] = real(0);
        }
        // the volume terms of this thread's solution point, in flight across the barrier
        const int dc = dist_bits & 255, ds = dist_bits >> 8;
        const bool dist = dc < nc;
        real vi[5], idet = real(0);
        v4 vv = {0, 0, 0, 0};
        if (dist) {
            Args* a = fresh();
            const Idx pt = times<BIG>(cells[dc], NS) + ds;
            idet = at<BIG>(a->det, pt);
            if constexpr (INV) {
#pragma unroll
                for (int v = 0; v < 5; ++v) vi[v] = at<BIG>(a->R, pt * 5 + v);
            }
            if constexpr (VISC) vv = at<BIG>((const v4*)a->rvisc, pt);
        }
        __syncthreads();
        // the next tile's slot table and own points (its cells are known), the cells of the tile after it
        cell = next_cell;
        const Slot next = load_slot(cell, role().slot);
        next_cell = cell_at((cw.it + 2 * cw.step) * CPT + role().lc);
        load_own(s_cell[buf ^ 1]);
        // 3. distribution at the solution points, / det
        if (dist) {
            Args* a = fresh();
            const int di = ds / (N1 * N1), dj = (ds / N1) % N1, dk = ds % N1;
            real acc[NR];
#pragma unroll
            for (int v = 0; v < NR; ++v) acc[v] = 0;
#pragma unroll
            for (int l = 0; l < NSLOT; ++l) {
                const int lcode = l < 3 ? l : l + 1, lax = lcode >> 1;
                const int x = lax == 0 ? di : (lax == 1 ? dj : dk);
                const int f = lax == 0 ? dj * N1 + dk : (lax == 1 ? di * N1 + dk : di * N1 + dj);
                const real g = at<BIG>((lcode & 1) ? a->gR : a->gL, (Idx)x);
                const real* jv = s_j + ((dc * NSLOT + l) * NFP + f) * JS;
#pragma unroll
                for (int v = 0; v < NR; ++v) acc[v] += g * jv[v];
            }
            idet = recip(idet);
            real* r = s_a + tid * NR;
            if constexpr (INV) {
#pragma unroll
                for (int v = 0; v < 5; ++v) r[v] = -(vi[v] + acc[v]) * idet;
            }
            if constexpr (VISC) {
#pragma unroll
                for (int v = 0; v < 4; ++v) r[NI + v] = (vv[v] + acc[NI + v]) * idet;
            }
        }
        __syncthreads();
        // 4. outlier zeroing (troubled_cell.py:339-408, see afr_outlier.hpp): with M = max_s |R| and at
        //    most (NS-1)/2 values below 1.0001e-4 M no value can exceed 1e4 times the median; only where
        //    that fails is the median selected, by rank counting
        if (fresh()->suppress) {
            constexpr int k1 = (NS - 1) / 2, k2 = NS / 2;
            for (int q = tid; q < nc * NR; q += NT) {
                const real* x = s_a + (q / NR) * NS * NR + q % NR;
                real mx = 0;
#pragma unroll 9
                for (int s = 0; s < NS; ++s) {
                    const real v = fabs(x[s * NR]);
                    mx = v > mx ? v : mx;
                }
                const real tt = mx * real(1.0001e-4);
                int cnt = 0;
#pragma unroll 9
                for (int s = 0; s < NS; ++s) cnt += fabs(x[s * NR]) < tt;
                if (cnt > k1) {
                    s_list[atomicAdd(&s_bad, 1)] = q;
                    s_med[0][q] = s_med[1][q] = real(-1);
                }
            }
            __syncthreads();
            if (const int n_bad = s_bad; n_bad > 0) {
                // the values of the listed columns over the whole workgroup: rank of each, and |U| of
                // its point for the field mean.  The value at a median position (all lanes that hold it
                // write the same) stays -1 when no finite value holds it (NaN median: nothing is zeroed).
                Args* a = fresh();
                for (int q = tid; q < n_bad * NS; q += NT) {
                    const int col = s_list[q / NS], c = col / NR, v = col % NR, s = q % NS;
                    const real* r = s_a + c * NS * NR + v;
                    const real x = fabs(r[s * NR]);
                    int lt = 0, le = 0;
#pragma unroll(NS % 9 == 0 ? 9 : 8)
                    for (int s2 = 0; s2 < NS; ++s2) {
                        const real y = fabs(r[s2 * NR]);
                        lt += y < x;
                        le += y <= x;
                    }
                    if (lt <= k1 && k1 < le) s_med[0][col] = x;
                    if (lt <= k2 && k2 < le) s_med[1][col] = x;
                    if (!a->umean) {   // of the absolute state; the own points' place is free by now
                        const int var = v < NI ? v : v - NI + 1;
                        const int64_t cell_no = cells[c];
                        double off = 0.0;
                        if (a->so.mode == 1) off = a->so.one[var];
                        if (a->so.mode == 2)
                            off = ((GlobalPtr<double>)a->so.table)[5 * (int64_t)(a->so.cell_case ? ((GlobalPtr<int>)a->so.cell_case)[cell_no] : 0) + var];
                        const double u = (double)((GlobalPtr<real>)a->U)[(cell_no * NS + s) * 5 + var];
                        s_own[q] = (real)fabs(a->so.mode ? u + off : u);
                    }
                }
                __syncthreads();
                for (int q = tid; q < n_bad; q += NT) {   // threshold of the column (in s_med[0]), -1: none
                    const int col = s_list[q], v = col % NR;
                    const real m1 = s_med[0][col], m2 = s_med[1][col];
                    real thr = real(-1);
                    if (!(m1 < real(0) || ((NS % 2) == 0 && m2 < real(0)))) {
                        real um;
                        if (a->umean) {
                            um = ((GlobalPtr<real>)a->umean)[(int64_t)cells[col / NR] * 5 + (v < NI ? v : v - NI + 1)];
                        } else {
                            real acc = 0;
#pragma unroll(NS % 9 == 0 ? 9 : 8)
                            for (int s2 = 0; s2 < NS; ++s2) acc += s_own[q * NS + s2];
                            um = acc / real(NS);
                        }
                        const real med = (NS % 2) ? m1 : real(0.5) * (m1 + m2);
                        thr = real(1e4) * nan_max(nan_max(med, real(1e-9) * um), Tiny<real>::v);
                    }
                    s_med[0][col] = thr;
                }
                __syncthreads();
                for (int q = tid; q < n_bad * NS; q += NT) {
                    const int col = s_list[q / NS];
                    real* r = s_a + (col / NR * NS + q % NS) * NR + col % NR;
                    const real thr = s_med[0][col];
                    if (thr >= real(0) && fabs(*r) > thr) *r = real(0);
                }
                __syncthreads();
                if (tid == 0) s_bad = 0;
            }
        }
        // 5. R, consecutive threads consecutive values
        {
            Args* a = fresh();
            typedef __attribute__((address_space(1))) real GlobalReal;
#pragma unroll
            for (int q = 0; q < (CPT * NS * 5 + NT - 1) / NT; ++q) {
                const int o = lane_fresh(tid) + q * NT, p = o / 5, v = o % 5, c = p / NS;
                if (c < nc) {
                    const real* r = s_a + p * NR;
                    real x = INV ? r[v] : real(0);
                    if (VISC && v > 0) x += r[NI + v - 1];
                    const Idx oi = times<BIG>(cells[c], NS * 5) + (o - c * (NS * 5));
                    GlobalReal* out;
                    if constexpr (BIG) out = (GlobalReal*)a->R + oi;
                    else out = (GlobalReal*)((__attribute__((address_space(1))) char*)a->R + (uint32_t)(oi * (uint32_t)sizeof(real)));
                    *out = (!INV && a->accumulate) ? *out + x : x;
                }
            }
        }
        take_slot(next, role().fp);
        store_own();
        __syncthreads();
    }
}

template <int P, int CT, int KMAX, typename real, bool INV, bool VISC>
int launch_iface_t(const MeanArgs<real>& a, hipStream_t st) {
    using L = IF<P, CT, real, INV, VISC>;
    const int64_t tiles = (a.n_cells + L::CPT - 1) / L::CPT;
    // 2048 workgroups, twice what is resident, up to some 50 tiles each; 4096 for larger meshes.  Whole
    // mean-flow residual, us, 2048 against 4096: P2 prisms FP32 13k tiles 289 / 296, 35k 752 / 753, 70k 1504 /
    // 1502, 100k 2140 / 2123, 150k 3185 / 3156, 220k 4749 / 4691; P1 prisms 25k 466 / 473, 99k 1812 / 1812, 222k
    // 4112 / 4110; P3 tets 41k 4159 / 4177, 96k 9577 / 9581
    const int grid = walk_grid(tiles, 1, a.grid_cap > 0 ? a.grid_cap : (tiles <= 100000 ? 2048 : 4096));
    // 32-bit byte offsets while the pack of all cells (the largest array by cells) and the table of
    // distinct interpolation rows stay under 4 GiB
    const bool big = a.n_cells_mesh * L::NS * kPack * (int64_t)sizeof(real) >= ((int64_t)1 << 32) ||
                     (int64_t)a.n_rows * KMAX * 8 >= ((int64_t)1 << 32);
    if constexpr (CT == 1 && P >= 2 && VISC && sizeof(real) == 8) {
        // matrix products wherever the fragments of the rows fit the scratch array: the rows depend on how two
        // faces meet, not on their shape (6 blocks for any box of tets), so that only meshes of a few cells have
        // more blocks than cells' scratch.  24.6k P3 tets 327 us, 700 by vector FMAs; 10.3k P2 tets 55 (81).
        // The sums are the same, term by term.
        const int64_t blocks = (a.n_rows + L::NFP - 1) / L::NFP, n = blocks * FR<P>::KS * 64;
        if (n <= a.work_len && n < ((int64_t)1 << 30)) {
            if (n > 0)
                hipLaunchKernelGGL((k_row_fragments<P>), dim3((unsigned)(blocks < 1024 ? blocks : 1024)), dim3(256), 0, st,
                                   a.rows_nnz, a.rows_idx, a.rows_w, a.knz, a.n_rows, a.work);
            if (big)
                hipLaunchKernelGGL((k_iface<P, CT, KMAX, real, INV, VISC, true, true>), dim3(grid), dim3(L::NT), 0, st, a);
            else
                hipLaunchKernelGGL((k_iface<P, CT, KMAX, real, INV, VISC, false, true>), dim3(grid), dim3(L::NT), 0, st, a);
            return hipGetLastError() == hipSuccess ? 0 : -1;
        }
    }
    if (big)
        hipLaunchKernelGGL((k_iface<P, CT, KMAX, real, INV, VISC, true, false>), dim3(grid), dim3(L::NT), 0, st, a);
    else
        hipLaunchKernelGGL((k_iface<P, CT, KMAX, real, INV, VISC, false, false>), dim3(grid), dim3(L::NT), 0, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int P, int CT, typename real>
int launch_iface(const MeanArgs<real>& a, bool inv, bool visc, hipStream_t st) {
    constexpr int NS = (P + 1) * (P + 1) * (P + 1), KS = (P + 1) * (P + 1);
    if (a.n_cells <= 0) return 0;
    if (a.knz == KS)
        return inv ? (visc ? launch_iface_t<P, CT, KS, real, true, true>(a, st)
                           : launch_iface_t<P, CT, KS, real, true, false>(a, st))
                   : launch_iface_t<P, CT, KS, real, false, true>(a, st);
    if (a.knz == NS)
        return inv ? (visc ? launch_iface_t<P, CT, NS, real, true, true>(a, st)
                           : launch_iface_t<P, CT, NS, real, true, false>(a, st))
                   : launch_iface_t<P, CT, NS, real, false, true>(a, st);
    return -1;
}

#define AFR_IF_INST(P, CT, T) template int launch_iface<P, CT, T>(const MeanArgs<T>&, bool, bool, hipStream_t);
AFR_IF_INST(1, 0, float)
AFR_IF_INST(2, 0, float)
AFR_IF_INST(1, 0, double)
AFR_IF_INST(2, 0, double)
AFR_IF_INST(1, 1, float)
AFR_IF_INST(2, 1, float)
AFR_IF_INST(1, 1, double)
AFR_IF_INST(2, 1, double)
AFR_IF_INST(3, 1, double)

}  // namespace afr_mean
