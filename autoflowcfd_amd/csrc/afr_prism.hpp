// Shared declarations of the prism (Kronecker-factored) kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "afr_physics.hpp"

struct Ref5 {
    double q[5];
};

namespace afr_prism {

template <int P> struct PK {
    static constexpr int N1 = P + 1;
    static constexpr int NAB = N1 * N1;
    static constexpr int OV = (2 * P < 3 ? 2 * P : 3);
    static constexpr int NF1 = OV + 1;
    static constexpr int NABF = NF1 * NF1;
    static constexpr int NF = NABF * NF1;
    static constexpr int NS = NAB * N1;
    static constexpr int NFP = N1 * N1;
    // packed factor table (autoflowcfd_amd/fr_tables.py PrismFactors.packed order)
    static constexpr int O_C2FAB = 0;
    static constexpr int O_C2FC = O_C2FAB + NABF * NAB;
    static constexpr int O_AA = O_C2FC + NF1 * N1;
    static constexpr int O_AB = O_AA + NAB * NABF;
    static constexpr int O_BC = O_AB + NAB * NABF;
    static constexpr int O_F2CC = O_BC + N1 * NF1;
    static constexpr int O_F2CAB = O_F2CC + N1 * NF1;
    static constexpr int O_EAB = O_F2CAB + NAB * NABF;
    static constexpr int O_EC = O_EAB + 3 * N1 * NAB;
    static constexpr int O_DAB = O_EC + 2 * N1;
    static constexpr int O_DC = O_DAB + 2 * NAB * NAB;
    static constexpr int TABN = O_DC + N1 * N1;
};

template <int NS, typename real>
int launch_prim_umean(const real* U, real* dQ, real* umean, int64_t n, const double* ref, afr::StateOff so,
                      hipStream_t st);

}  // namespace afr_prism
