// ndf_flux.hpp -- the diffusion fluxes of NDF (diffusion.hip, ndf2d.hip).
#pragma once
#include "common.hpp"

namespace cilreg {

// The penalty's flux for a neighbour difference d (Diffusion_core.c:166-231);
// powf(x, 2) is x * x.  PEN is the penalty (0 linear), a template argument so
// each kernel holds one straight-line flux.
template <int PEN>
__device__ inline float ndf_flux(float d, float sigma) {
    const float ad = fabsf(d);
    const float sg = (float)((d > 0.f) - (d < 0.f));
    if constexpr (PEN == 1) return ad > sigma ? sg : d / sigma;
    if constexpr (PEN == 2) {
        const float q = d / sigma;
        return d / (1.0f + q * q);
    }
    if constexpr (PEN == 3) {
        if (ad <= sigma) {
            const float q = d / sigma;
            const float t = 1.0f - q * q;
            return d * (t * t);
        }
        return 0.0f;
    }
    if constexpr (PEN == 4) return ad > sigma ? 0.0f : d;
    if constexpr (PEN == 5) return ad <= 2.0f * sigma ? (ad > sigma ? sg : d / sigma) : 0.0f;
    return d;   // linear diffusion
}

// g(dw) from F = g(D), the flux a neighbour computed for its own difference
// D across the shared edge (penalty PEN >= 1, sigma > 0).  dw = -D exactly
// unless both are +0 (a - b = -(b - a) in round-to-nearest, except equal
// operands, which give +0 both ways), and every penalty is odd except where
// it returns the literal 0: there g(dw) = 0, on zero g(dw) = dw, elsewhere
// g(dw) = -F, bit for bit (NaN operands included: the literal-zero tests are
// written as the penalty's own).
template <int PEN>
__device__ inline float ndf_flux_mirror(float dw, float F, float sigma) {
    if (dw == 0.f) return dw;
    const float ad = fabsf(dw);
    if constexpr (PEN == 3) {
        if (!(ad <= sigma)) return 0.0f;
    }
    if constexpr (PEN == 4) {
        if (ad > sigma) return 0.0f;
    }
    if constexpr (PEN == 5) {
        if (!(ad <= 2.0f * sigma)) return 0.0f;
    }
    return -F;
}

}  // namespace cilreg
