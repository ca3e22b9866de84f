// k_star_pair instantiations for float grid functions.
#include "stencil_pair_impl.h"

namespace gpaw {

hipError_t pair_launch_f32(const Stencil& s, int mode, const void* in, void* out, const void* aux,
                         const Geom& g, const Phases& ph, double w, int TZ, const TileShape& sh,
                         hipStream_t st)
{
    return pair_dispatch<float>(s, mode, in, out, aux, g, ph, w, TZ, sh, st);
}

}  // namespace gpaw
