// Stencils other than the orthogonal-cell Laplacian: non-orthogonal cells,
// Mehrstellen, gradients (gfx950).
//
// k_generic (stencil.hip) looks up every term of every point through the
// caches with its own wrap tests, which bounds it at 15-25 % of the bandwidth
// a copy reaches.  Two kernels replace it wherever a grid and stencil allow
// (gen_launch); the sums run in coefficient order (c/bmgs/fd.c:41-44) with
// the same epilogue, so results are bit-identical to it.
//
// k_gen_sweep: any offsets of up to 4 points.  A block of 256 threads owns a
// TY x TZ tile of the (i1, i2) plane and sweeps a run of i0 planes two at a
// time; the planes that the terms reach (with an r1 x r2 halo, ghost-indexed)
// are held in a ring of 2 R + 2 LDS slots, the next two are in flight in
// registers while the current two are summed.  A term is one LDS read and
// five (complex: seven) vector instructions per point, which bounds it: 25
// terms of a hexagonal cell, 64 complex128 bands of 48 x 48 x 72, 430 -> 158 us
// (2.1 TB/s), float64 341 -> 80 us; Mehrstellen on 127^3 57 -> 17.5 us.  Blocks
// of 512 and 1024 threads sharing a deeper ring measured 166 and 149 us there
// and lost on 9 terms (82 -> 92 and 102 us).
//
// k_axis: stencils along one axis in the order -R..-1, +1..+R (Gradient,
// gpaw/fd_operators.py:123-144).  One thread per in-plane point and Q planes,
// every load issued at once, no LDS: the neighbours along axes 0 and 1 come
// from the thread's own column of Q + 2 R points, along axis 2 through the L1.
// HBM bound: 2 x 127^3 float64, R = 3, 43 -> 12.5 us (16.5 us along axis 2, where
// k_axis2 takes over for rows that fit a block).
#pragma once
#include "kernels.h"

namespace gpaw {

constexpr int GEN_PL = 2;      // planes per thread and step
constexpr int GEN_NC = 3;      // LDS cells per thread and plane
constexpr int GEN_MAXR = 4;
// LDS slots, and LDS cells of one plane (640 at range 3 keep two complex128
// blocks per CU)
constexpr int gen_planes(int R) { return 2 * R + GEN_PL; }
constexpr int gen_cells(int R) { return R == 3 ? 640 : 256 * GEN_NC; }

struct GenShape {
    int tz, ty, ntz, nty;      // tile, tiles along i2 / i1
    int lw;                    // LDS row length
    int q, nchunk, nblocks;    // planes per block, chunks along i0
    int r[3];                  // reach of the stencil per axis
};

template <class V, int R, int MODE>
__global__ __launch_bounds__(256) void k_gen_sweep(const V* __restrict__ in, V* __restrict__ out,
                                                   const V* __restrict__ aux, Geom g, Phases ph,
                                                   GenShape sh, const GenTerm* __restrict__ terms,
                                                   int nc, double w, i64 ng)
{
    typedef typename VT<V>::R RT;
    constexpr int PL = GEN_PL, NC = GEN_NC, NP = gen_planes(R), CELLS = gen_cells(R);
    __shared__ V lds[NP * CELLS];
    const int t = xcd_tile(blockIdx.x, sh.nblocks);
    const int tzi = t % sh.ntz;
    int rest = t / sh.ntz;
    const int tyb = rest % sh.nty;
    rest /= sh.nty;
    const int ch = rest % sh.nchunk;
    const i64 boff = (i64)(rest / sh.nchunk) * ng;
    const V* __restrict__ a = in + boff;
    V* __restrict__ o = out + boff;
    const V* __restrict__ sa = (aux && MODE != ST_HPSI) ? aux + boff : aux;

    const int tid = threadIdx.x;
    const int r0 = sh.r[0], r1 = sh.r[1], r2 = sh.r[2];
    const int LW = sh.lw, row = sh.tz + 2 * r2, cells = row * (sh.ty + 2 * r1);
    const int n0 = g.n[0];
    const i64 plane = (i64)g.n[1] * g.n[2];
    const int z0 = tzi * sh.tz, y0 = tyb * sh.ty;
    const int ly = tid / sh.tz, lz = tid - ly * sh.tz;
    const int i1 = y0 + ly, i2 = z0 + lz;
    const bool own = ly < sh.ty && i1 < g.n[1] && i2 < g.n[2];
    // threads without a point read the tile's first one
    const int base = own ? (r1 + ly) * LW + r2 + lz : r1 * LW + r2;
    const int poff = own ? i1 * g.n[2] + i2 : 0;
    const int i0s = ch * sh.q, i0e = min(i0s + sh.q, n0);

    PlaneRef cr[NC];
    int cl[NC];   // LDS index, -1: no cell
#pragma unroll
    for (int k = 0; k < NC; k++) {
        const int c = tid + 256 * k, lr = c / row, lc = c - lr * row;
        cr[k] = c < cells ? plane_ref(y0 + lr - r1, z0 + lc - r2, g) : PREF_ZERO;
        cl[k] = c < cells ? lr * LW + lc : -1;
    }
    // plane p of the cells, raw; planes no term reaches are not loaded
    auto load = [&](int p, V* v) -> int {
        const int f = p < n0 + r0 ? wrap_index(p, n0, g.per[0]) : 3;
        const i64 b = f == 3 ? 0 : (i64)p * plane;
#pragma unroll
        for (int k = 0; k < NC; k++) v[k] = a[b + pref_off(cr[k])];
        return f;
    };
    auto put = [&](int slot, const V* v, int f) {
        V* B = lds + slot * CELLS;
#pragma unroll
        for (int k = 0; k < NC; k++)
            if (cl[k] >= 0) B[cl[k]] = ghost_fix(v[k], f, cr[k], ph);
    };
    auto wrap = [](int slot) { return slot >= NP ? slot - NP : slot; };
    V pre[PL][NC];
    int pf[PL];
    {   // planes i0s - r0 .. i0s + r0 - 1 into slots 0 .. 2 r0 - 1
        V fill[2 * R][NC];
        int ff[2 * R];
#pragma unroll
        for (int k = 0; k < 2 * R; k++)
            if (k < 2 * r0) ff[k] = load(i0s - r0 + k, fill[k]);
#pragma unroll
        for (int u = 0; u < PL; u++) pf[u] = load(i0s + r0 + u, pre[u]);
#pragma unroll
        for (int k = 0; k < 2 * R; k++)
            if (k < 2 * r0) put(k, fill[k], ff[k]);
    }
    // Terms c0 .. c0 + 63 in the lanes of every wave: coefficient, in-plane LDS
    // offset and plane offset; read back as uniform values lane by lane
    // (scalar loads in the term loop cost their latency every few terms).
    const int lane = tid & 63;
    double tc;
    int toff, td0;
    auto fetch = [&](int c0) {
        const GenTerm tm = terms[min(c0 + lane, nc - 1)];
        tc = tm.c;
        toff = tm.d[1] * LW + tm.d[2];
        td0 = tm.d[0];
    };
    auto uniform = [](double v, int l) -> double {
        const long long b = __builtin_bit_cast(long long, v);
        const int lo = __builtin_amdgcn_readlane((int)b, l);
        const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
        return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
    };
    fetch(0);
    const double c00 = uniform(tc, 0);
    int rs = 0;   // slot of plane i0 - r0
    V res[PL];
    auto store = [&](int i0) {
#pragma unroll
        for (int u = 0; u < PL; u++)
            if (own && i0 + u < i0e) o[(i64)(i0 + u) * plane + poff] = res[u];
    };
    for (int i0 = i0s; i0 < i0e; i0 += PL) {
#pragma unroll
        for (int u = 0; u < PL; u++)
#pragma unroll
            for (int k = 0; k < NC; k++) vtouch(pre[u][k]);
        // the slots written here are those of planes i0 - r0 - PL .., which
        // the previous step read
        if (i0 > i0s) __syncthreads();
#pragma unroll
        for (int u = 0; u < PL; u++) put(wrap(rs + 2 * r0 + u), pre[u], pf[u]);
        if (i0 > i0s) store(i0 - PL);
        if (i0 + PL < i0e) {
#pragma unroll
            for (int u = 0; u < PL; u++) pf[u] = load(i0 + PL + r0 + u, pre[u]);
        }
        V s[PL];
        if (MODE != ST_APPLY) {
#pragma unroll
            for (int u = 0; u < PL; u++)
                s[u] = aux_value<MODE>(sa, 0, own && i0 + u < i0e ? (i64)(i0 + u) * plane + poff : 0);
        }
        __syncthreads();
        V x[PL];
#pragma unroll
        for (int u = 0; u < PL; u++) x[u] = vzero<V>();
        const int rc = rs + r0;   // slot of plane i0, before its wrap
        for (int c0 = 0; c0 < nc; c0 += 64) {
            if (nc > 64) fetch(c0);
            int at[PL];   // LDS index of each lane's term, plane by plane
#pragma unroll
            for (int u = 0; u < PL; u++) at[u] = wrap(rc + u + td0) * CELLS + toff;
            // groups of terms, whose LDS reads go out together
            constexpr int U = sizeof(V) == 16 ? 4 : 8;
            auto term = [&](int c) {
                const RT k = (RT)uniform(tc, c);
#pragma unroll
                for (int u = 0; u < PL; u++)
                    x[u] = vmac(x[u], lds[__builtin_amdgcn_readlane(at[u], c) + base], k);
            };
            const int ce = min(64, nc - c0);
#pragma unroll
            for (int c = 0; c < 64; c += U) {
                if (c + U <= ce) {
#pragma unroll
                    for (int i = 0; i < U; i++)
                        if (!(MODE == ST_JACOBI && c + i == 0) || c0 > 0) term(c + i);
                } else {
#pragma unroll
                    for (int i = 0; i < U - 1; i++)
                        if (c + i < ce && (!(MODE == ST_JACOBI && c + i == 0) || c0 > 0)) term(c + i);
                    break;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < PL; u++) {
            const V f = MODE == ST_APPLY || MODE == ST_RESID ? vzero<V>()
                                                             : lds[wrap(rc + u) * CELLS + base];
            res[u] = st_epilogue<MODE>(x[u], f, MODE == ST_APPLY ? vzero<V>() : s[u], (RT)w,
                                       (RT)c00);
        }
        rs = wrap(rs + PL);
    }
    if (i0e > i0s) store(i0s + (i0e - i0s - 1) / PL * PL);
}

struct AxisCoefs {
    double c[2 * GEN_MAXR];
};

template <class V, int R, int AXIS, int Q>
__global__ __launch_bounds__(256) void k_axis(const V* __restrict__ in, V* __restrict__ out,
                                              Geom g, Phases ph, AxisCoefs sc, int ncol, i64 ng)
{
    typedef typename VT<V>::R RT;
    // a thread owns Q points of a column along QA: the stencil's axis, or for
    // axis 2, whose neighbours are other lanes' points, axis 0
    constexpr int QA = AXIS == 1 ? 1 : 0;
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= ncol) return;
    const int n = g.n[QA], s0 = blockIdx.y * Q;
    const i64 plane = (i64)g.n[1] * g.n[2];
    const i64 st = QA == 1 ? g.n[2] : plane;   // stride along QA
    const i64 b = (i64)blockIdx.z * ng + (QA == 1 ? j / g.n[2] * plane + j % g.n[2] : j);
    const V* __restrict__ a = in + b;
    V* __restrict__ o = out + b;
    // offsets -R..-1, 1..R of terms 0 .. 2 R - 1
    auto offset = [](int m) { return m < R ? m - R : m - R + 1; };
    V v[AXIS < 2 ? Q + 2 * R : Q * 2 * R];
    int f[AXIS < 2 ? Q + 2 * R : 2 * R];
    if (AXIS < 2) {
#pragma unroll
        for (int k = 0; k < Q + 2 * R; k++) {
            int p = s0 - R + k;
            f[k] = p < n + R ? wrap_index(p, n, g.per[QA]) : 3;
            v[k] = a[f[k] == 3 ? 0 : p * st];
        }
    } else {
        const int i = j % g.n[2];
#pragma unroll
        for (int m = 0; m < 2 * R; m++) {
            int k = i + offset(m);
            f[m] = wrap_index(k, g.n[2], g.per[2]);
            const int d = f[m] == 3 ? 0 : k - i;
#pragma unroll
            for (int u = 0; u < Q; u++) v[u * 2 * R + m] = a[min(s0 + u, n - 1) * st + d];
        }
    }
    auto fix = [&](V x, int fl) -> V {
        if (fl == 3) return vzero<V>();
        if (VT<V>::cplx && fl) x = pside<true>(x, ph, AXIS, fl);
        return x;
    };
#pragma unroll
    for (int u = 0; u < Q; u++) {
        if (s0 + u >= n) break;
        V x = vzero<V>();
#pragma unroll
        for (int m = 0; m < 2 * R; m++) {
            const V y = AXIS < 2 ? fix(v[u + R + offset(m)], f[u + R + offset(m)])
                                 : fix(v[u * 2 * R + m], f[m]);
            x = vmac(x, y, (RT)sc.c[m]);
        }
        o[(s0 + u) * st] = x;
    }
}

// The same along axis 2 for rows of up to AXIS2_PTS points: a block takes whole
// rows, up to AXIS2_PTS points in all, which are contiguous in memory; they go
// to LDS once, with R ghosts on either side of each row, and a point reads its
// 2 R neighbours there instead of through the L1 (2 x 127^3 float64, R = 3:
// 16.5 -> 12.5 us).
constexpr int AXIS2_PTS = 1024;

template <class V, int R>
__global__ __launch_bounds__(256) void k_axis2(const V* __restrict__ in, V* __restrict__ out,
                                               Geom g, Phases ph, AxisCoefs sc, int nr, int rows,
                                               unsigned magic)
{
    typedef typename VT<V>::R RT;
    constexpr int PT = AXIS2_PTS / 256;
    extern __shared__ __align__(16) char axis2_lds[];
    V* __restrict__ L = (V*)axis2_lds;
    const int n = g.n[2], LW = n + 2 * R;
    const int row0 = blockIdx.x * nr, mine = min(nr, rows - row0), pts = mine * n;
    const V* __restrict__ a = in + (i64)row0 * n;
    V* __restrict__ o = out + (i64)row0 * n;
    V v[PT];
    int at[PT];
#pragma unroll
    for (int k = 0; k < PT; k++) {
        const int el = threadIdx.x + 256 * k;
        v[k] = a[el < pts ? el : 0];
        const int r = __umulhi((unsigned)el, magic);   // el / n
        at[k] = el < pts ? r * LW + R + el - r * n : -1;
    }
    // ghosts: cell c of a row is at -R + c, or for c >= R at n + c - R
    for (int h = threadIdx.x; h < mine * 2 * R; h += 256) {
        const int r = h / (2 * R), c = h % (2 * R), pos = c < R ? c - R : n + c - R;
        int p = pos;
        const int f = wrap_index(p, n, g.per[2]);
        V x = vzero<V>();
        if (f != 3) {
            x = a[r * n + p];
            if (VT<V>::cplx && f) x = pside<true>(x, ph, 2, f);
        }
        L[r * LW + R + pos] = x;
    }
#pragma unroll
    for (int k = 0; k < PT; k++)
        if (at[k] >= 0) L[at[k]] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PT; k++) {
        if (at[k] < 0) continue;
        const V* __restrict__ c = L + at[k];
        V x = vzero<V>();
#pragma unroll
        for (int m = 0; m < 2 * R; m++) x = vmac(x, c[m < R ? m - R : m - R + 1], (RT)sc.c[m]);
        o[threadIdx.x + 256 * k] = x;
    }
}

// Launch one of the kernels above if it can run this pass (*handled says
// whether it did): grids whose halo wraps at most once, no partial sums.
template <class V>
hipError_t gen_launch(const Stencil& s, int mode, const void* in, void* out, const void* aux,
                      const Geom& g, const Phases& ph, int nin, double w, hipStream_t st,
                      bool* handled);

}  // namespace gpaw
