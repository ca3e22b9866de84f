// k_star_pair instantiations for float2 grid functions.
#include "stencil_pair_impl.h"

namespace gpaw {

hipError_t pair_launch_c64(const Stencil& s, int mode, const void* in, void* out, const void* aux,
                         const Geom& g, const Phases& ph, double w, int TZ, const TileShape& sh,
                         hipStream_t st)
{
    return pair_dispatch<float2>(s, mode, in, out, aux, g, ph, w, TZ, sh, st);
}

}  // namespace gpaw
