// The CG direction step of the mixed-precision Poisson solve in one launch.
#pragma once
#include "kernels.h"

namespace gpaw {

// What the step reads and writes.  S: the solver's device scalars, alpha at
// S[ia] and the previous d.z at S[idz]; zq: nzq partials of z.q; hist: where
// the ndd partials of |d|^2 at dd are summed to (nullptr: not summed).
struct CgStep {
    const double* p_in;
    double* p_out;        // not p_in
    double* q;
    double* phi;          // nullptr: no pending step to subtract
    const double* S;
    int ia, idz;
    const double* zq;
    int nzq;
    const double* dd;
    int ndd;
    double* hist;
    double* partial;      // p.q, one partial per block
};

// Whether launch_cg_dir runs on this operator; its partials then number
// *npartial, at most stencil_partials().
bool cg_dir_ok(const Stencil& s, const Geom& g, int* npartial);
// z: the preconditioned residual, FP32 or FP64 (zdtype)
hipError_t launch_cg_dir(const Stencil& s, const Geom& g, const CgStep& a, const void* z,
                         int zdtype, hipStream_t st);

}  // namespace gpaw
