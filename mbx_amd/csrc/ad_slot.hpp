// The fitted coefficients' linear map to the polynomials' slots, and its transpose, for the differentiated
// polynomials (adjoint.hip), which take the coefficients from device memory at every call.
#pragma once

#include <hip/hip_runtime.h>

namespace mbxg {

// Slot q of the symmetry-adapted polynomial's coefficients (gen/sym_<name>.inc): products and sum are
// carried with their rounding errors (a weight such as 3/8 rounds the product too), so slots at or past
// nrow get what rounding left of slot low[q - nrow].
__device__ __forceinline__ double ad_slot(const int* row, const unsigned short* k, const double* w,
                                          const unsigned short* low, int nrow, int q,
                                          const double* __restrict__ coef) {
    const int r = q < nrow ? q : low[q - nrow];
    double s = 0.0, err = 0.0;
    for (int i = row[r]; i < row[r + 1]; ++i) {
        const double p = coef[k[i]] * w[i];
        const double t = s + p, z = t - s;
        err += ((s - (t - z)) + (p - z)) + __fma_rn(coef[k[i]], w[i], -p);
        s = t;
    }
    const double b = s + err;
    return q < nrow ? b : err - (b - s);
}

// Entry k of the transposed map: the fitted coefficient's gradient from the slots' (row[q]).
__device__ __forceinline__ double ad_coef_adjoint(const int* start, const unsigned short* slot, const double* w, int k,
                                                  const double* __restrict__ row) {
    double s = 0.0;
    for (int i = start[k]; i < start[k + 1]; ++i) s = __fma_rn(row[slot[i]], w[i], s);
    return s;
}

}  // namespace mbxg
