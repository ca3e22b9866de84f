// Launch rules of stencil_gen.h, instantiated once per storage type in
// stencil_gen_<type>.hip.
#pragma once
#include "stencil_gen.h"

namespace gpaw {

inline bool gen_shape(const Stencil& s, const Geom& g, int esize, int nin, GenShape& sh)
{
    const int* r = s.reach;
    const int R = s.gen_r;
    // every coordinate a tile touches lies within one period of the grid
    for (int a = 0; a < 3; a++)
        if (g.n[a] < r[a]) return false;
    if ((long)g.n[1] * g.n[2] >= PLANE_REF_MAX) return false;
    for (int a = 0; a < 3; a++) sh.r[a] = r[a];
    // Tile of up to 256 threads: the width with the least lanes and LDS cells
    // over the plane (a 72-point row is 3 tiles of 24, not 3 of 32).  Rows of
    // 16-byte elements are padded so that a wave's lanes, which run over
    // several rows, fall on distinct banks (158 against 171 us on the case
    // above; for 8-byte elements the longer rows cost more blocks per CU than
    // the conflicts do: 80 against 90 us).
    long best = -1;
    const int P = 16;
    for (int tz = 16; tz <= 64; tz++) {
        int ty = 256 / tz;
        const int row = tz + 2 * r[2], lw = esize == 16 && tz % P ? tz + (2 * r[2] + P - 1) / P * P : row;
        const int ntz = (g.n[2] + tz - 1) / tz;
        while (ty > 1 && ((ty + 2 * r[1]) * lw > gen_cells(R) ||
                          (ty + 2 * r[1]) * row > 256 * GEN_NC))
            ty--;
        const int nty = (g.n[1] + ty - 1) / ty;
        const int cells = (ty + 2 * r[1]) * row;
        if ((ty + 2 * r[1]) * lw > gen_cells(R) || cells > 256 * GEN_NC) continue;
        if (ntz * tz + r[2] > 2 * g.n[2] || nty * ty + r[1] > 2 * g.n[1]) continue;
        const long cost = (long)ntz * nty * (256 + cells);
        if (best < 0 || cost < best) {
            best = cost;
            sh.tz = tz;
            sh.lw = lw;
            sh.ty = ty;
            sh.ntz = ntz;
            sh.nty = nty;
        }
    }
    if (best < 0) return false;
    // i0 runs split until there are 2048 blocks (float64, 960 tiles: 80 us
    // against 84 for 512 blocks; the 2 r0 planes that a run reads twice cost
    // more on shorter runs)
    const long tiles = (long)sh.ntz * sh.nty * nin;
    long nch = (2048 + tiles - 1) / tiles;
    const long maxch = (g.n[0] + GEN_PL - 1) / GEN_PL;
    if (nch > maxch) nch = maxch;
    sh.q = (int)((g.n[0] + nch - 1) / nch);
    sh.q = (sh.q + GEN_PL - 1) / GEN_PL * GEN_PL;
    sh.nchunk = (g.n[0] + sh.q - 1) / sh.q;
    if (tiles * sh.nchunk > 0x7fffffffL) return false;
    sh.nblocks = (int)(tiles * sh.nchunk);
    return true;
}

template <class V, int R>
hipError_t gen_mode(const Stencil& s, int mode, const void* in, void* out, const void* aux,
                    const Geom& g, const Phases& ph, double w, const GenShape& sh, hipStream_t st,
                    bool* handled)
{
    const i64 ng = (i64)g.n[0] * g.n[1] * g.n[2];
    const dim3 grid(sh.nblocks), block(256);
#define GPAW_GEN_MODE(M)                                                                        \
    case M:                                                                                     \
        if constexpr (st_mode_ok<V, M>()) {                                                     \
            *handled = true;                                                                    \
            return launch_kernel((k_gen_sweep<V, R, M>), grid, block, 0, st, (const V*)in,      \
                                 (V*)out, (const V*)aux, g, ph, sh, (const GenTerm*)s.d_terms,  \
                                 s.nc, w, ng);                                                  \
        }                                                                                       \
        return hipSuccess;
    switch (mode) {
        GPAW_GEN_MODE(ST_APPLY)
        GPAW_GEN_MODE(ST_RESID)
        GPAW_GEN_MODE(ST_JACOBI)
        GPAW_GEN_MODE(ST_PCUPD)
        GPAW_GEN_MODE(ST_PCFIN)
        GPAW_GEN_MODE(ST_HPSI)
    }
#undef GPAW_GEN_MODE
    return hipSuccess;
}

template <class V, int R, int AXIS, int Q>
hipError_t axis_go(const Stencil& s, const void* in, void* out, const Geom& g, const Phases& ph,
                   int nin, hipStream_t st)
{
    AxisCoefs sc;
    for (int c = 0; c < 2 * R; c++) sc.c[c] = s.coefs[c];
    const i64 ng = (i64)g.n[0] * g.n[1] * g.n[2];
    const int n = g.n[AXIS == 1 ? 1 : 0];
    const i64 ncol = ng / n;
    return launch_kernel((k_axis<V, R, AXIS, Q>),
                         dim3((unsigned)((ncol + 255) / 256), (n + Q - 1) / Q, nin), dim3(256), 0,
                         st, (const V*)in, (V*)out, g, ph, sc, (int)ncol, ng);
}

template <class V, int R>
hipError_t axis2_go(const Stencil& s, const void* in, void* out, const Geom& g, const Phases& ph,
                    int nin, hipStream_t st)
{
    AxisCoefs sc;
    for (int c = 0; c < 2 * R; c++) sc.c[c] = s.coefs[c];
    const int n = g.n[2], rows = g.n[0] * g.n[1] * nin, nr = AXIS2_PTS / n;
    const size_t lds = (size_t)nr * (n + 2 * R) * sizeof(V);
    const unsigned magic = (unsigned)(((1ULL << 32) + n - 1) / n);   // exact below 2^32 / n
    return launch_kernel((k_axis2<V, R>), dim3((unsigned)((rows + nr - 1) / nr)), dim3(256), lds,
                         st, (const V*)in, (V*)out, g, ph, sc, nr, rows, magic);
}

template <class V, int R>
hipError_t axis_launch(const Stencil& s, const void* in, void* out, const Geom& g,
                       const Phases& ph, int nin, hipStream_t st)
{
    // 4 points per thread: 1 / 2 / 4 / 8 measured 22 / 17 / 12.5 / 12 us along axis
    // 0 and 17.4 / 16.5 / 16.5 / 18 us along axis 2 on 2 x 127^3 float64
    switch (s.axis) {
    case 0: return axis_go<V, R, 0, 4>(s, in, out, g, ph, nin, st);
    case 1: return axis_go<V, R, 1, 4>(s, in, out, g, ph, nin, st);
    case 2:
        // whole rows of 16 .. 1024 points in LDS: shorter ones would be mostly
        // ghosts, longer ones do not fit (127: 12.5 against 16.5 us)
        if (g.n[2] >= 16 && g.n[2] <= AXIS2_PTS && (long)g.n[0] * g.n[1] * nin < 0x7fffffffL)
            return axis2_go<V, R>(s, in, out, g, ph, nin, st);
        return axis_go<V, R, 2, 4>(s, in, out, g, ph, nin, st);
    }
    return hipErrorInvalidValue;
}

template <class V>
hipError_t gen_launch(const Stencil& s, int mode, const void* in, void* out, const void* aux,
                      const Geom& g, const Phases& ph, int nin, double w, hipStream_t st,
                      bool* handled)
{
    *handled = false;
    if (s.axis >= 0 && mode == ST_APPLY && g.n[s.axis] >= s.gen_r &&
        (long)g.n[1] * g.n[2] < PLANE_REF_MAX && (long)g.n[0] * g.n[2] < PLANE_REF_MAX &&
        g.n[0] <= 65535 && g.n[1] <= 65535) {
        *handled = true;
        switch (s.gen_r) {
        case 1: return axis_launch<V, 1>(s, in, out, g, ph, nin, st);
        case 2: return axis_launch<V, 2>(s, in, out, g, ph, nin, st);
        case 3: return axis_launch<V, 3>(s, in, out, g, ph, nin, st);
        case 4: return axis_launch<V, 4>(s, in, out, g, ph, nin, st);
        }
        return hipErrorInvalidValue;
    }
    GenShape sh;
    if (!s.d_terms || !gen_shape(s, g, (int)sizeof(V), nin, sh)) return hipSuccess;
    switch (s.gen_r) {
    case 1: return gen_mode<V, 1>(s, mode, in, out, aux, g, ph, w, sh, st, handled);
    case 2: return gen_mode<V, 2>(s, mode, in, out, aux, g, ph, w, sh, st, handled);
    case 3: return gen_mode<V, 3>(s, mode, in, out, aux, g, ph, w, sh, st, handled);
    case 4: return gen_mode<V, 4>(s, mode, in, out, aux, g, ph, w, sh, st, handled);
    }
    return hipSuccess;
}

}  // namespace gpaw
