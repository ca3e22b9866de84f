// Restriction / interpolation instantiations for double grid functions.
#include "transfer_impl.h"

namespace gpaw {

hipError_t transfer_launch_f64(const Transfer& t, int mode, const void* in, void* out,
                             void* zero_out, const Phases& ph, int nin, hipStream_t st)
{
    return tr_dispatch<double>(t, mode, in, out, zero_out, ph, nin, st);
}

hipError_t launch_interp_sums(const Transfer& t, const void* in, void* out, const Phases& ph,
                              int nin, double* sums, int* nsums, hipStream_t st)
{
    *nsums = 0;
    return tr_dispatch<double>(t, TR_STORE, in, out, nullptr, ph, nin, st, sums, nsums);
}

}  // namespace gpaw
