// Plan of the fused coarse-level V-cycle kernel.
#pragma once
#include "transfer_common.h"

namespace gpaw {

#define GPAW_COARSE_LEVELS 4      // levels one launch runs, at most
#define GPAW_COARSE_POINTS 2048   // points of the first level, at most (two per
                                  // thread); the others have at most 1024

struct CoarseLevel {
    int n[3], per[3];
    int off;              // LDS offset (doubles) of the level's phi pair
    int pre, post;        // smoothing counts
    double c[7];          // 7-point star: centre, z+, z-, y+, y-, x+, x-
    double w;             // Jacobi weight
    int rlo[3];           // restriction from this level: Transfer::lo
    int ilo[3], iskip[3]; // interpolation into this level: lo and skip
};

// Passed to the kernel by value.
struct CoarsePlan {
    int nlev = 0;
    CoarseLevel lev[GPAW_COARSE_LEVELS];
    const void* rho = nullptr;   // first level: right-hand side and solution,
    void* out = nullptr;         // double, or float inside an FP32 V-cycle
};

TrArgs make_trargs(const Transfer& tr);
hipError_t launch_coarse_vcycle(const CoarsePlan& plan, int dtype, hipStream_t st);

}  // namespace gpaw
