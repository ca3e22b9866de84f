// Host launcher of k_star_pair for one storage type (stencil_pair_<type>.hip).
#pragma once
#include "stencil_pair.h"

namespace gpaw {

template <class V, int R, int TZ, int MODE>
hipError_t pair_go(const Stencil& s, const void* in, void* out, const void* aux, const Geom& g,
                   const Phases& ph, double w, const TileShape& sh, hipStream_t st)
{
    TileCoefs sc;
    for (int c = 0; c < 6 * R + 1; c++) sc.c[c] = s.coefs[c];
    return launch_kernel((k_star_pair<V, R, TZ, MODE>), dim3(sh.nblocks), dim3(TZ, PAIR_TY), 0, st,
                         (const V*)in, (V*)out, (const V*)aux, g, ph, sc, w, sh,
                         (i64)g.n[0] * g.n[1] * g.n[2]);
}

template <class V, int R, int TZ>
hipError_t pair_mode(const Stencil& s, int mode, const void* in, void* out, const void* aux,
                     const Geom& g, const Phases& ph, double w, const TileShape& sh,
                     hipStream_t st)
{
    if (mode == ST_APPLY) return pair_go<V, R, TZ, ST_APPLY>(s, in, out, aux, g, ph, w, sh, st);
    if constexpr (st_mode_ok<V, ST_HPSI>())
        if (mode == ST_HPSI) return pair_go<V, R, TZ, ST_HPSI>(s, in, out, aux, g, ph, w, sh, st);
    return hipErrorInvalidValue;
}

template <class V, int R>
hipError_t pair_tz(const Stencil& s, int mode, const void* in, void* out, const void* aux,
                   const Geom& g, const Phases& ph, double w, int TZ, const TileShape& sh,
                   hipStream_t st)
{
    switch (TZ) {
    case 32: return pair_mode<V, R, 32>(s, mode, in, out, aux, g, ph, w, sh, st);
    case 48: return pair_mode<V, R, 48>(s, mode, in, out, aux, g, ph, w, sh, st);
    case 64: return pair_mode<V, R, 64>(s, mode, in, out, aux, g, ph, w, sh, st);
    case 96:
        if constexpr (sizeof(V) < 16)
            return pair_mode<V, R, 96>(s, mode, in, out, aux, g, ph, w, sh, st);
    }
    return hipErrorInvalidValue;
}

template <class V>
hipError_t pair_dispatch(const Stencil& s, int mode, const void* in, void* out, const void* aux,
                         const Geom& g, const Phases& ph, double w, int TZ, const TileShape& sh,
                         hipStream_t st)
{
    switch (s.star_r) {
    case 1: return pair_tz<V, 1>(s, mode, in, out, aux, g, ph, w, TZ, sh, st);
    case 2: return pair_tz<V, 2>(s, mode, in, out, aux, g, ph, w, TZ, sh, st);
    case 3: return pair_tz<V, 3>(s, mode, in, out, aux, g, ph, w, TZ, sh, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace gpaw
