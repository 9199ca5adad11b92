// cf_pcg_state.hpp -- the PCG scalars' transitions on the device.
#pragma once

#include <hip/hip_runtime.h>

#include "cf_kernels.hpp"

namespace cfmi
{

__device__ __forceinline__ void init_state(PcgState* st, double rz, double nn,
                                           double tol, int maxit)
{
    const double norm = sqrt(nn);
    st->bnorm = norm;
    st->tol = tol;
    st->maxit = maxit;
    st->iter = 0;
    st->rho = rz;
    st->alpha = 0.0;
    st->beta = 0.0;
    st->alpha_lag = 0.0;
    const bool zero = norm == 0.0;
    // a NaN or Inf in the right-hand side stops the solve before it starts
    const bool bad = !isfinite(norm);
    st->done = zero || bad ? 1 : (maxit <= 0 ? 1 : 0);
    st->converged = zero ? 1 : 0;
    st->res = zero ? 0.0 : (bad ? norm : 1.0);
    st->mg = 0;
    st->nonfinite = bad ? 1 : 0;
    st->stalled = 0;
}

// Scalars after an update: iteration count, relative residual, the stop
// test, and (Jacobi-PCG) beta and rho.  A residual that is not finite stops
// the solve at once (the stop test alone would read false and run to maxit).
__device__ __forceinline__ void finish_update(PcgState* st, double rr, double rz)
{
    const int it = st->iter + 1;
    st->iter = it;
    const double res = sqrt(rr) / st->bnorm;
    const double beta = rz / st->rho; // beside the residual's chain; used if the solve goes on
    st->res = res;
    if (!isfinite(res)) {
        st->done = 1;
        st->nonfinite = 1;
    } else if (res < st->tol) {
        st->done = 1;
        st->converged = 1;
    } else if (it >= st->maxit) {
        st->done = 1;
    } else {
        if (!st->mg) { // MG-PCG: beta and rho follow the V-cycle
            st->beta = beta;
            st->rho = rz;
        }
    }
}

} // namespace cfmi
