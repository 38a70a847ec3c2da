// bosonic.hpp -- the bosonic drift of one site (update.hip, onchip.hip).
#pragma once
#include "ycn_device.hpp"

namespace ycn {

// drift += phi (m2 + lambda/6 phi^2) - (sum_nbr phi - 4 phi)
__device__ __forceinline__ double bosonic_drift(const double *__restrict__ ph, int s, int Nt, int Nx, double m2,
                                                double lam6) {
    const int t = s / Nx, x = s - t * Nx;
    const Nbr n = neighbours(t, x, Nt, Nx);
    const double f = ph[s];
    const double pot = f * (m2 + lam6 * (f * f));
    const double lap = (ph[n.tf] + ph[n.tb] + ph[n.xf] + ph[n.xb]) - 4.0 * f;
    return pot - lap;
}

}  // namespace ycn
