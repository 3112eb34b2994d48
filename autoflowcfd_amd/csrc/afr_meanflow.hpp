// Shared declarations of the mean-flow residual kernels (volume terms, interface terms).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "afr_physics.hpp"

namespace afr_mean {

// Per-point pack of the viscous terms, written by the viscous volume kernel and read by the
// interface kernel: dQ (5), the symmetric velocity gradient S = grad u + (grad u)^T as xx, yy, zz,
// xy, xz, yz (6: the stress needs no more of it), grad T (3), mu_t (1), pad (1).  16 values: one
// point is 64 bytes in FP32 (128 in FP64), aligned, read by four 16-byte loads.
constexpr int kPack = 16;
constexpr int kPackUsed = 15;

template <typename real>
struct MeanArgs {
    int64_t cell_begin, n_cells;   // cells [cell_begin, cell_begin + n_cells) of one type
    int64_t n_cells_mesh;          // cells of both types
    const int* schedule;           // null, or the locality order of the cells of this type
    int grid_cap;                  // workgroups (0: built-in default)
    const real* U;                 // (C, NS, 5) conserved (offset from so's table when it has one)
    afr::StateOff so;
    const real* dQ;                // (C, NS, 5) prepared primitive perturbation (kernels fed from it)
    const real* umean;             // (C, 5) mean |U| (null: taken from U where it is needed)
    const real* mu_t;              // (C, NS) or null
    real* dQ_out;                  // (C, NS, 5), (C, 5): written by the viscous volume kernel when
    real* umean_out;               //                     not null (callers that prepare the state)
    real* pack;                    // (C, NS, kPack)
    real* rvisc;                   // (C, NS, 4) viscous volume divergence of the momenta and energy
    real* R;                       // (C, NS, 5) inviscid volume divergence in, residual out
    const real* det;
    const real* adj;               // (C, NS, 3, 3)
    const real* adjf;              // (C, NF, 3, 3)
    const real* gcl;               // (C, NS, 3)
    const real* D;                 // (3, NS, NS) of the cell type
    const real* E;                 // (5, NFP, NS) of the cell type, slot order
    const real* c2f;               // (NF, NS) of the cell type (tets)
    const real* op;                // (NS, 3 NF) of the cell type (tets)
    const real* tab;               // packed prism factors
    const int* slot_nb;
    const int* slot_blk;
    const int* slot_mask;
    const int* slot_bc;
    const int* slot_fb;
    const real* slot_tn;
    const real* slot_adjrow;
    const int* rows_nnz;
    const int* rows_idx;
    const real* rows_w;
    int knz, n_rows;
    const real* gL;
    const real* gR;
    const double* bcp;
    const int* cell_case;          // null: one case
    double qref[5];                // primitive reference state, its flux F(qref)[i][v]
    double fref[15];
    double mu, Pr, Prt;
    real* work;                    // scratch for the interpolation rows as matrix fragments (FP64 tets)
    int64_t work_len;
    int suppress;
    int accumulate;                // viscous-only interface: R += result instead of R = result
};

// viscous volume term: pack, rvisc (and dQ_out, umean_out) from U
template <int P, int CT, typename real>
int launch_visc_volume(const MeanArgs<real>& a, hipStream_t st);

// inviscid volume divergence (over-integrated) from U into R
template <int P, int CT, typename real>
int launch_inv_volume(const MeanArgs<real>& a, hipStream_t st);

// interface terms: AUSM+up jumps (inv) and BR1 jumps (visc) of every slot, distribution, / det,
// outlier zeroing of each part, R
template <int P, int CT, typename real>
int launch_iface(const MeanArgs<real>& a, bool inv, bool visc, hipStream_t st);

// ------------------------------------------------------------------ device helpers
template <typename real> struct V4;
template <> struct V4<float> { typedef float type __attribute__((ext_vector_type(4))); };
template <> struct V4<double> { typedef double type __attribute__((ext_vector_type(4))); };
template <typename real>
__device__ __forceinline__ typename V4<real>::type ld4(const real* p) {
    return *reinterpret_cast<const typename V4<real>::type*>(p);
}
template <typename real>
__device__ __forceinline__ void st4(real* p, typename V4<real>::type v) {
    *reinterpret_cast<typename V4<real>::type*>(p) = v;
}

// ------------------------------------------------------------------ matrix cores, FP64 16 x 16 x 4
// D += A B: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and D[4 i + l / 16][l % 16], i = 0 .. 3.
typedef V4<double>::type d4;
__device__ __forceinline__ d4 mma(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

template <typename T> using GlobalPtr = const __attribute__((address_space(1))) T*;

// table values that every lane of the wavefront takes alike: scalar loads, no LDS, no VGPR
typedef const __attribute__((address_space(4))) float* UniF;
typedef const __attribute__((address_space(4))) double* UniD;
template <typename real> struct Uni;
template <> struct Uni<float> { typedef UniF type; };
template <> struct Uni<double> { typedef UniD type; };

// LDS operations of one wavefront execute in program order: a compiler barrier separates stages
// whose lanes exchange data through LDS
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The lane index redefined by an empty asm: index arithmetic on it is not hoisted out of a loop,
// where it would hold registers for the whole kernel
__device__ __forceinline__ int lane_fresh(int t) {
    asm volatile("" : "+v"(t));
    return t;
}

}  // namespace afr_mean
