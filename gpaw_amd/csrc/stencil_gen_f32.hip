// stencil_gen.h instantiations for float grid functions.
#include "stencil_gen_impl.h"

namespace gpaw {

hipError_t gen_launch_f32(const Stencil& s, int mode, const void* in, void* out, const void* aux,
                        const Geom& g, const Phases& ph, int nin, double w, hipStream_t st,
                        bool* handled)
{
    return gen_launch<float>(s, mode, in, out, aux, g, ph, nin, w, st, handled);
}

}  // namespace gpaw
