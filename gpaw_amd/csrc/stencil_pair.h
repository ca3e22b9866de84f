// Star stencils of large band sets, two planes per step (gfx950).
//
// k_star_tile (stencil_tile.h) takes one barrier, one wait for memory and a
// shift of its register queue per plane, and its 32-column tiles cut a grid's
// rows into segments that are not whole cache lines where the row length is
// odd.  Here a block of TZ x 8 threads, TZ up to the whole row, sweeps its tile
// two planes at a time: whole planes with their halo sit in a ring of R + 2
// LDS slots, loaded R planes ahead (so halo rows are read while the
// neighbouring tile's own rows are still in the L2), the next two in flight in
// registers while the current two are summed.  The planes behind are needed at
// a thread's own point only and stay in R registers.
// Terms in k_star_tile's order with the same epilogue: bit-identical.
//
// HBM bound.  R = 3, where the launch rule (large_cfg, stencil.hip) takes it:
// float64 256 x 64^3 264 us with k_star_tile, 240 here (4.5 TB/s); 96 x 79x87x95
// 290 and 264, 128 x 79x87x63 252 and 206; with the potential 128 x 63^3 176 and
// 152; float32 256 x 64^3 182 and 149.  Rings of R + 4 slots (one barrier per pair)
// and tiles of 16 or 32 rows leave fewer blocks per CU and were no faster; two or
// four bands per block, to share the potential, were slower (96 x 79x87x95 327 ->
// 357 us), and so was running the bands of one tile together.
#pragma once
#include "stencil_tile.h"

namespace gpaw {

constexpr int PAIR_TY = 8;   // rows per tile

template <class V, int R, int TZ, int MODE>
__global__ __launch_bounds__(TZ * PAIR_TY) void k_star_pair(const V* __restrict__ in,
                                                       V* __restrict__ out,
                                                       const V* __restrict__ aux, Geom g,
                                                       Phases phases, TileCoefs sc, double w,
                                                       TileShape sh, i64 ng)
{
    typedef typename VT<V>::R RT;
    constexpr int TY = PAIR_TY, NT = TZ * TY, NP = R + 2, LW = TZ + 2 * R, LH = TY + 2 * R, PS = LH * LW;
    constexpr int NC = (PS + NT - 1) / NT;
    __shared__ V ring[NP * PS];
    const Phases ph = scalar_phases<V>(phases);
    const int t = xcd_tile(blockIdx.x, sh.nblocks);
    const int tzi = t % sh.ntz;
    int rest = t / sh.ntz;
    const int tyb = rest % sh.nty;
    rest /= sh.nty;
    const int i0s = rest % sh.nchunk * sh.q, i0e = min(i0s + sh.q, g.n[0]);
    const i64 band = rest / sh.nchunk;
    const i64 boff = band * ng;
    const V* __restrict__ a = in + boff;
    V* __restrict__ o = out + boff;
    const V* __restrict__ sa = (aux && MODE != ST_HPSI) ? aux + boff : aux;
    const int tx = threadIdx.x, tyi = threadIdx.y, tid = tx + TZ * tyi;
    const int n0 = g.n[0];
    const i64 plane = (i64)g.n[1] * g.n[2];
    const int z0 = tzi * TZ, y0 = tyb * TY;
    const bool own = y0 + tyi < g.n[1] && z0 + tx < g.n[2];
    const unsigned poff = own ? (unsigned)((y0 + tyi) * g.n[2] + z0 + tx) : 0u;
    const int lbase = (R + tyi) * LW + R + tx;

    // this thread's cells of a plane: byte offset, wrap flags (bits 0..3), LDS
    // index (-1: none, or beyond a zero boundary, where the ring stays zero)
    unsigned co[NC];
    int cf[NC], cl[NC];
#pragma unroll
    for (int k = 0; k < NC; k++) {
        const int c = tid + NT * k;
        const PlaneRef r = c < PS ? plane_ref(y0 + c / LW - R, z0 + c % LW - R, g) : PREF_ZERO;
        const bool ok = (r & 3) != 3 && (r >> 2 & 3) != 3;
        co[k] = ok ? (unsigned)pref_off(r) * (unsigned)sizeof(V) : 0u;
        cf[k] = ok ? r & 15 : 0;
        cl[k] = ok ? c : -1;
    }
    auto at = [](const V* p, unsigned bytes) -> V {
        return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(p) + bytes);
    };
    auto pflag = [&](int p, i64& base) -> int {
        const int f = p < n0 + R ? wrap_index(p, n0, g.per[0]) : 3;
        base = f == 3 ? 0 : (i64)p * plane;
        return f;
    };
    auto load = [&](int p, V* v) -> int {
        i64 base;
        const int f = pflag(p, base);
        const V* q = a + base;
#pragma unroll
        for (int k = 0; k < NC; k++) v[k] = at(q, co[k]);
        return f;
    };
    // ghost corrections in axis order (ghost_fix); f0 is uniform
    auto fix = [&](V v, int f0, int fl) -> V {
        if constexpr (VT<V>::cplx) {
            if (f0) v = pside<true>(v, ph, 0, f0);
            if (fl) {
                asm volatile("");   // a branch, not selects
                if (fl & 3) v = pside<true>(v, ph, 1, fl & 3);
                if (fl >> 2) v = pside<true>(v, ph, 2, fl >> 2);
            }
        }
        return v;
    };
    auto put = [&](int slot, const V* v, int f) {
        V* B = ring + slot * PS;
#pragma unroll
        for (int k = 0; k < NC; k++) {
            const V x = f == 3 ? vzero<V>() : fix(v[k], f, cf[k]);
            if (cl[k] >= 0) B[cl[k]] = x;
        }
    };
    if (!g.per[1] || !g.per[2]) {   // cells beyond a zero boundary stay zero
        for (int i = tid; i < NP * PS; i += NT) ring[i] = vzero<V>();
        __syncthreads();
    }
    // planes i0s - R .. i0s - 1 at this point, i0s .. i0s + R - 1 into slots
    // 0 .. R - 1, the next two in flight
    V prev[R], pre[2][NC], sn[2], res[2];
    int pf[2];
    auto load_aux = [&](int i0) {
        if (MODE != ST_APPLY) {
#pragma unroll
            for (int u = 0; u < 2; u++)
                sn[u] = aux_value<MODE>(sa, 0, (i64)min(i0 + u, n0 - 1) * plane + poff);
        }
    };
    {
        V fill[R][NC];
        int ff[R], fp[R];
        const PlaneRef qr = plane_ref(y0 + tyi, z0 + tx, g);
#pragma unroll
        for (int k = 0; k < R; k++) {
            i64 base;
            fp[k] = pflag(i0s - R + k, base);
            prev[k] = a[base + pref_off(qr)];
        }
#pragma unroll
        for (int k = 0; k < R; k++) ff[k] = load(i0s + k, fill[k]);
#pragma unroll
        for (int u = 0; u < 2; u++) pf[u] = load(i0s + R + u, pre[u]);
        load_aux(i0s);
#pragma unroll
        for (int k = 0; k < R; k++) prev[k] = ghost_fix(prev[k], fp[k], qr, ph);
#pragma unroll
        for (int k = 0; k < R; k++) put(k, fill[k], ff[k]);
    }
    auto store = [&](int i0) {
#pragma unroll
        for (int u = 0; u < 2; u++)
            if (own && i0 + u < i0e) tile_store<true>(o + (i64)(i0 + u) * plane + poff, res[u]);
    };
    auto wrap = [](int s) { return s >= NP ? s - NP : s; };
    int rs = 0;   // slot of plane i0
    for (int i0 = i0s; i0 < i0e; i0 += 2) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
#pragma unroll
            for (int k = 0; k < NC; k++) vtouch(pre[u][k]);
            if (MODE != ST_APPLY) vtouch(sn[u]);
        }
        if (i0 > i0s) __syncthreads();   // the slots written next were read in the last step
        put(wrap(rs + R), pre[0], pf[0]);
        put(wrap(rs + R + 1), pre[1], pf[1]);
        V s[2];
        if (MODE != ST_APPLY) {
            s[0] = sn[0];
            s[1] = sn[1];
        }
        if (i0 > i0s) store(i0 - 2);
        if (i0 + 2 < i0e) {
#pragma unroll
            for (int u = 0; u < 2; u++) pf[u] = load(i0 + 2 + R + u, pre[u]);
            load_aux(i0 + 2);
        }
        __syncthreads();
        const V* pl[R + 2];   // plane i0 + j at this thread's point
        V col[2 * R + 2];     // its values at planes i0 - R .. i0 + R + 1
#pragma unroll
        for (int j = 0; j < R + 2; j++) pl[j] = ring + wrap(rs + j) * PS + lbase;
#pragma unroll
        for (int j = 0; j < R; j++) col[j] = prev[j];
#pragma unroll
        for (int j = 0; j < R + 2; j++) col[R + j] = pl[j][0];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const V* row = pl[u];
            V x = vzero<V>();
            if (MODE != ST_JACOBI) x = vmac(x, col[R + u], (RT)sc.c[0]);
#pragma unroll
            for (int k = 1; k <= R; k++) x = vmac(x, row[k], (RT)sc.c[k]);
#pragma unroll
            for (int k = 1; k <= R; k++) x = vmac(x, row[-k], (RT)sc.c[R + k]);
#pragma unroll
            for (int k = 1; k <= R; k++) x = vmac(x, row[k * LW], (RT)sc.c[2 * R + k]);
#pragma unroll
            for (int k = 1; k <= R; k++) x = vmac(x, row[-k * LW], (RT)sc.c[3 * R + k]);
#pragma unroll
            for (int k = 1; k <= R; k++) x = vmac(x, col[R + u + k], (RT)sc.c[4 * R + k]);
#pragma unroll
            for (int k = 1; k <= R; k++) x = vmac(x, col[R + u - k], (RT)sc.c[5 * R + k]);
            res[u] = st_epilogue<MODE>(x, col[R + u], MODE == ST_APPLY ? vzero<V>() : s[u], (RT)w,
                                       (RT)sc.c[0]);
        }
#pragma unroll
        for (int j = 0; j < R; j++) prev[j] = col[j + 2];
        rs = wrap(rs + 2);
    }
    if (i0e > i0s) store(i0s + (i0e - i0s - 1) / 2 * 2);
}

}  // namespace gpaw
