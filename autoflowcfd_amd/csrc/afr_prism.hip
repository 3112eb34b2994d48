// Preparation of the primitive state: dQ = primitive(U) - Q_ref and the mean |U| of every cell
// (src/autoflowcfd/core/fr_residual/inviscid.py:38-47, the outlier reference of
// src/autoflowcfd/core/fr_operators/troubled_cell.py:371-380).
#include <hip/hip_runtime.h>

#include "../../include/afr.h"
#include "afr_physics.hpp"
#include "afr_prism.hpp"

using namespace afr;

namespace afr_prism {

// dQ = primitive(U) - ref and umean[c][v] = mean_s |U[c][s][v]| (outlier field reference)
template <int NS, typename real>
__global__ void __launch_bounds__(256) k_prim_umean(const real* __restrict__ U, real* __restrict__ dQ,
                                                    real* __restrict__ umean, int64_t n_cells, Ref5 ref,
                                                    StateOff so) {
    constexpr int CPB = 256 / NS;
    __shared__ real s_abs[CPB * NS * 5];
    const int t = threadIdx.x;
    for (int64_t c0 = (int64_t)blockIdx.x * CPB; c0 < n_cells; c0 += (int64_t)gridDim.x * CPB) {
        const int c = t / NS, s = t % NS;
        const bool ok = (t < CPB * NS) && (c0 + c < n_cells);
        if (ok) {
            const int64_t i = (c0 + c) * NS + s;
            double u[5], q[5];
            load_state(U, i, so, c0 + c, u);
            cons2prim(u, q);
#pragma unroll
            for (int v = 0; v < 5; ++v) {
                dQ[i * 5 + v] = (real)(q[v] - ref.q[v]);
                const real x = (real)u[v];
                s_abs[(c * NS + s) * 5 + v] = x < real(0) ? -x : x;
            }
        }
        __syncthreads();
        if (t < CPB * 5) {
            const int cc = t / 5, v = t % 5;
            if (c0 + cc < n_cells) {
                real acc = 0;
                for (int s2 = 0; s2 < NS; ++s2) acc += s_abs[(cc * NS + s2) * 5 + v];
                umean[(c0 + cc) * 5 + v] = acc / real(NS);
            }
        }
        __syncthreads();
    }
}

template <int NS, typename real>
int launch_prim_umean(const real* U, real* dQ, real* umean, int64_t n, const double* ref, StateOff so,
                      hipStream_t st) {
    Ref5 r;
    for (int v = 0; v < 5; ++v) r.q[v] = ref ? ref[v] : 0.0;
    constexpr int CPB = 256 / NS;
    int64_t blocks = (n + CPB - 1) / CPB;
    int grid = (int)(blocks < 65536 ? (blocks > 0 ? blocks : 1) : 65536);
    hipLaunchKernelGGL((k_prim_umean<NS, real>), dim3(grid), dim3(256), 0, st, U, dQ, umean, n, r, so);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template int launch_prim_umean<8, float>(const float*, float*, float*, int64_t, const double*, StateOff,
                                                 hipStream_t);
template int launch_prim_umean<27, float>(const float*, float*, float*, int64_t, const double*, StateOff,
                                                 hipStream_t);
template int launch_prim_umean<64, float>(const float*, float*, float*, int64_t, const double*, StateOff,
                                                 hipStream_t);
template int launch_prim_umean<8, double>(const double*, double*, double*, int64_t, const double*, StateOff,
                                                 hipStream_t);
template int launch_prim_umean<27, double>(const double*, double*, double*, int64_t, const double*, StateOff,
                                                 hipStream_t);
template int launch_prim_umean<64, double>(const double*, double*, double*, int64_t, const double*, StateOff,
                                                 hipStream_t);

}  // namespace afr_prism
