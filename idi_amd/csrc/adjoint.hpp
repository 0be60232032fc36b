// Shared by the adjoint kernels (adjoint.hip, adjoint_sep.hip).
#pragma once
#include "device_util.hpp"

namespace idisim {

constexpr int kAdjTile = 256;  // pixels per 16 x 16 tile (of the loss, and of k_adjoint's pixel table)

// The weight w'_p = G_p conj(E_p) e^{2 pi i Phi_p} (times 1/R_p with "scale") of pixel idx, from its
// complex64 field value E, its frame f and (nf) its pixel_phasor (cs, sn).
// target == nullptr: G_p = dLdI[p].  Otherwise the squared-intensity loss L = sum_p (I_p - T_p)^2:
// G_p = 2 (I_p - T_p) with I_p = |E_p|^2 in FP64, and res2 = (I_p - T_p)^2.
__device__ inline void adj_pixel_weight(const Geom& g, const Frame& f, double cs, double sn, float2 E, size_t idx,
                                        const float* __restrict__ dLdI, const float* __restrict__ target, double& wr,
                                        double& wi, double& res2)
{
    double G;
    if (target != nullptr) {
        const double res = (double)E.x * (double)E.x + (double)E.y * (double)E.y - (double)target[idx];
        res2 = res * res;
        G = 2.0 * res;
    } else {
        G = (double)dLdI[idx];
    }
    wr = G * (double)E.x, wi = -G * (double)E.y;
    if (g.nf) {
        const double r2 = wr * cs - wi * sn;
        wi = wr * sn + wi * cs;
        wr = r2;
    }
    if (g.scale) {  // the per-pixel factor 1/R_p of the "scale" amplitude R_c/(D_cj R_p)
        wr /= f.R;
        wi /= f.R;
    }
}

// <x^4> / <x^2> over the T pixel centres of a square's side, x in units of T / 2 pixels.
__host__ __device__ constexpr double adj_x4(int T) { return (3.0 * T * T - 7.0) / 20.0 * 4.0 / ((double)T * T); }

}  // namespace idisim
