// Stencil passes of the preconditioner over fields that are never stored
// (gfx950).
//
// The preconditioner (precond.hip) applies its stencils to scaled residuals
// and to interpolations of the coarser level.  These kernels form those fields
// on the way into the stencil instead of reading what another launch wrote:
//   k_pc_scaled  F = c b                (d1 = 4 s r1, d2 = 16 s r2)
//   k_pc_interp  F = I e                (d0 = I1(d1), up to its sign)
//                F = c b - I e          (BASE: d1 -= I2(d2))
// with b a field of this level and I the K = 2 interpolation of e from the
// coarser one, every step rounded as the separate launches round it: the
// interpolation's z, y, x passes on ghost-indexed coarse values, the scaling,
// the difference, and the Bloch phases of F's own halo last.
#pragma once
#include "stencil_tile.h"
#include "transfer_common.h"

namespace gpaw {

// F = c b: the register queue and LDS plane of k_star_tile, each loaded value
// scaled before its ghost phase.  HBM bound: 256 complex128 bands of 32^3 in
// 51 us (5.2 TB/s), where the scaling and the stencil launch took 61 + 86.
template <class V, int R, int MODE, int NT, int TZ>
__global__ __launch_bounds__(NT) void k_pc_scaled(const V* __restrict__ in, V* __restrict__ out,
                                                  Geom g, Phases ph, TileCoefs sc, double cb,
                                                  double w, TileShape sh, i64 ng)
{
    typedef typename VT<V>::R RT;
    constexpr int TY = NT / TZ;
    constexpr int LW = TZ + 2 * R, LH = TY + 2 * R, NHALO = 2 * R * (TZ + TY);
    static_assert(NHALO <= NT, "one halo cell per thread");
    __shared__ V lds[2 * LH * LW];
    const int t = xcd_tile(blockIdx.x, sh.nblocks);
    const int tzi = t % sh.ntz;
    int rest = t / sh.ntz;
    const int tyb = rest % sh.nty;
    rest /= sh.nty;
    const int i0s = rest % sh.nchunk * sh.q, i0e = min(i0s + sh.q, g.n[0]);
    const i64 band = rest / sh.nchunk;
    const V* __restrict__ b = in + band * ng;
    V* __restrict__ o = out + band * ng;
    const int tx = threadIdx.x, tyi = threadIdx.y, tid = tx + TZ * tyi;
    const int n0 = g.n[0];
    const i64 plane = (i64)g.n[1] * g.n[2];
    const int z0 = tzi * TZ, y0 = tyb * TY;
    const bool own = y0 + tyi < g.n[1] && z0 + tx < g.n[2];
    const PlaneRef qr = plane_ref(y0 + tyi, z0 + tx, g);
    int hy, hz;
    if (tid < 2 * R * TZ) {
        const int yr = tid / TZ;
        hz = R + tid % TZ;
        hy = yr < R ? yr : TY + yr;
    } else {
        const int hh = tid - 2 * R * TZ, zc = hh % (2 * R);
        hy = R + hh / (2 * R);
        hz = zc < R ? zc : TZ + zc;
    }
    const bool halo = tid < NHALO;
    const PlaneRef hr = halo ? plane_ref(y0 + hy - R, z0 + hz - R, g) : PREF_ZERO;
    auto pflag = [&](int p, i64& base) -> int {
        const int f = p < n0 + R ? wrap_index(p, n0, g.per[0]) : 3;
        base = f == 3 ? 0 : (i64)p * plane;
        return f;
    };
    // bq: raw values of planes i0 .. i0 + R (the residual's b); q: F of planes
    // i0 - R .. i0 + R
    V q[2 * R + 1], bq[R + 1], bpre, hpre;
    i64 base;
#pragma unroll
    for (int k = 0; k < 2 * R; k++) {
        const int f = pflag(i0s - R + k, base);
        const V v = b[base + pref_off(qr)];
        q[k] = ghost_fix(vmul(v, (RT)cb), f, qr, ph);
        if (k >= R) bq[k - R] = v;
    }
    int hf = pflag(i0s, base);
    hpre = b[base + pref_off(hr)];
    int qf = pflag(i0s + R, base);
    bpre = b[base + pref_off(qr)];
    V rp;
    for (int i0 = i0s; i0 < i0e; i0++) {
        V* B = lds + ((i0 - i0s) & 1) * (LH * LW);
        vtouch(bpre);
        vtouch(hpre);
        bq[R] = bpre;
        q[2 * R] = ghost_fix(vmul(bpre, (RT)cb), qf, qr, ph);
        B[(R + tyi) * LW + R + tx] = q[R];
        if (halo) B[hy * LW + hz] = ghost_fix(vmul(hpre, (RT)cb), hf, hr, ph);
        if (i0 > i0s && own) o[(i64)(i0 - 1) * plane + pref_off(qr)] = rp;
        if (i0 + 1 < i0e) {
            qf = pflag(i0 + 1 + R, base);
            bpre = b[base + pref_off(qr)];
            hf = pflag(i0 + 1, base);
            hpre = b[base + pref_off(hr)];
        }
        __syncthreads();
        const V* row = B + (R + tyi) * LW + R + tx;
        V x = vmac(vzero<V>(), q[R], (RT)sc.c[0]);
#pragma unroll
        for (int k = 1; k <= R; k++) x = vmac(x, row[k], (RT)sc.c[k]);
#pragma unroll
        for (int k = 1; k <= R; k++) x = vmac(x, row[-k], (RT)sc.c[R + k]);
#pragma unroll
        for (int k = 1; k <= R; k++) x = vmac(x, row[k * LW], (RT)sc.c[2 * R + k]);
#pragma unroll
        for (int k = 1; k <= R; k++) x = vmac(x, row[-k * LW], (RT)sc.c[3 * R + k]);
#pragma unroll
        for (int k = 1; k <= R; k++) x = vmac(x, q[R + k], (RT)sc.c[4 * R + k]);
#pragma unroll
        for (int k = 1; k <= R; k++) x = vmac(x, q[R - k], (RT)sc.c[5 * R + k]);
        rp = st_epilogue<MODE>(x, q[R], bq[0], (RT)w, (RT)sc.c[0]);
#pragma unroll
        for (int k = 0; k < 2 * R; k++) q[k] = q[k + 1];
#pragma unroll
        for (int k = 0; k < R; k++) bq[k] = bq[k + 1];
    }
    if (i0e > i0s && own) o[(i64)(i0e - 1) * plane + pref_off(qr)] = rp;
}

struct PcCoarse {          // the K = 2 interpolation onto this level
    int nc[3];             // coarse extent
    int skip[3], lo[3];
};

// F = I e or c b - I e.  A block of 32 x TY threads sweeps its tile two planes
// at a time, an odd and an even one (in interpolation parity): together they
// need one new coarse plane.  Its raw values under the tile and halo go to
// LDS; one thread per coarse cell forms the z and y passes of the cell's
// 2 x 2 fine columns, keeps them for the next x pass and writes both planes of
// F to a ring of R + 2 LDS planes (i0 .. i0 + R + 1; the R planes before i0 are
// needed at a thread's own point only and stay in registers).
// Bound by instruction issue and its two barriers per pair next to HBM: the
// last pass of 256 complex128 bands of 64^3 reads r and the coarse field and
// writes the result, 2.28 GB; interpolation and stencil launch took 1015 us
// for 4.4 GB.  A first version with the passes of every thread's column and
// halo cell in register queues needed 206 vector and 160 scalar instructions a
// point and took 801 us.
template <class V, int R, bool BASE, int MODE, int TY>
__global__ __launch_bounds__(32 * TY) void k_pc_interp(const V* __restrict__ bin,
                                                       const V* __restrict__ ein,
                                                       V* __restrict__ out,
                                                       const V* __restrict__ aux, Geom g,
                                                       Phases phases, PcCoarse pc, TileCoefs sc,
                                                       double cb, double w, TileShape sh, i64 ng,
                                                       i64 ngc)
{
    typedef typename VT<V>::R RT;
    constexpr int TZ = 32, NT = TZ * TY;
    constexpr int LW = TZ + 2 * R, LH = TY + 2 * R, NP = R + 2, PS = LH * LW;
    constexpr int CW = LW / 2 + 2, CH = LH / 2 + 2;   // raw coarse values
    constexpr int EW = CW - 1, EH = CH - 1;           // cells: 2 x 2 fine columns
    static_assert(CW * CH <= NT, "one coarse value per thread");
    __shared__ V ring[NP * PS];
    const Phases ph = scalar_phases<V>(phases);
    __shared__ V C[CH * CW];
    const int t = xcd_tile(blockIdx.x, sh.nblocks);
    const int tzi = t % sh.ntz;
    int rest = t / sh.ntz;
    const int tyb = rest % sh.nty;
    rest /= sh.nty;
    const int i0s = rest % sh.nchunk * sh.q, i0e = min(i0s + sh.q, g.n[0]);
    const i64 band = rest / sh.nchunk;
    const V* __restrict__ b = BASE ? bin + band * ng : nullptr;
    const V* __restrict__ e = ein + band * ngc;
    const V* __restrict__ sa = aux + band * ng;
    V* __restrict__ o = out + band * ng;

    const int tx = threadIdx.x, tyi = threadIdx.y, tid = tx + TZ * tyi;
    const int n0 = g.n[0];
    const i64 plane = (i64)g.n[1] * g.n[2], cplane = (i64)pc.nc[1] * pc.nc[2];
    const int z0 = tzi * TZ, y0 = tyb * TY;
    const bool own = y0 + tyi < g.n[1] && z0 + tx < g.n[2];
    const int poff = own ? (y0 + tyi) * g.n[2] + z0 + tx : 0;
    const int lbase = (R + tyi) * LW + R + tx;

    // first fine pair of rows / columns (parity index P = fine + skip, P / 2)
    const int A1 = (y0 - R + pc.skip[1]) >> 1, A2 = (z0 - R + pc.skip[2]) >> 1;
    // this thread's raw coarse value: offset in a coarse plane, -1: zero
    int coff = -1;
    if (tid < CW * CH) {
        int ky = A1 - pc.lo[1] + tid / CW, kz = A2 - pc.lo[2] + tid % CW;
        if (g.per[1]) ky = ky < 0 ? ky + pc.nc[1] : ky >= pc.nc[1] ? ky - pc.nc[1] : ky;
        if (g.per[2]) kz = kz < 0 ? kz + pc.nc[2] : kz >= pc.nc[2] ? kz - pc.nc[2] : kz;
        if (ky >= 0 && ky < pc.nc[1] && kz >= 0 && kz < pc.nc[2]) coff = ky * pc.nc[2] + kz;
    }
    // this thread's cell: its fine columns' LDS offsets (-1: outside the tile,
    // or beyond a zero boundary, where the ring stays zero) and in-plane
    // offsets; wrap flags of the cell, the same for its columns (a periodic
    // axis has an even number of points); whether its second corner row /
    // column is a periodic ghost
    const bool cell = tid < EW * EH;
    const int ca = tid / EW, cz = tid % EW;
    int el[2][2], eo[2][2];
    int f1 = 0, f2 = 0;
    bool g1 = false, g2 = false;
#pragma unroll
    for (int d1 = 0; d1 < 2; d1++)
#pragma unroll
        for (int d2 = 0; d2 < 2; d2++) {
            const int j1 = 2 * (A1 + ca) + d1 - pc.skip[1], j2 = 2 * (A2 + cz) + d2 - pc.skip[2];
            const int ly = j1 - y0 + R, lz = j2 - z0 + R;
            const bool in = cell && ly >= 0 && ly < LH && lz >= 0 && lz < LW;
            const PlaneRef r = in ? plane_ref(j1, j2, g) : PREF_ZERO;
            const bool ok = (r & 3) != 3 && (r >> 2 & 3) != 3;
            el[d1][d2] = ok ? ly * LW + lz : -1;
            eo[d1][d2] = ok ? pref_off(r) : 0;
            if (ok) {
                f1 = r & 3;
                f2 = r >> 2 & 3;
            }
        }
    if (cell) {
        if (g.per[1]) {   // skip = lo = 0, fine extent 2 nc
            const int k = A1 + ca;
            g1 = (k < 0 ? k + pc.nc[1] : k >= pc.nc[1] ? k - pc.nc[1] : k) + 1 == pc.nc[1];
        }
        if (g.per[2]) {
            const int k = A2 + cz;
            g2 = (k < 0 ? k + pc.nc[2] : k >= pc.nc[2] ? k - pc.nc[2] : k) + 1 == pc.nc[2];
        }
    }
    // z and y passes of the cell from the staged plane; f0: the plane is the
    // ghost behind the last one of a periodic axis
    auto yz = [&](bool f0, V y[2][2]) {
        V v[2][2];
#pragma unroll
        for (int d1 = 0; d1 < 2; d1++)
#pragma unroll
            for (int d2 = 0; d2 < 2; d2++) v[d1][d2] = C[(ca + d1) * CW + cz + d2];
        if constexpr (VT<V>::cplx) {   // ghost corners: phases in axis order
            if (f0) {
#pragma unroll
                for (int d1 = 0; d1 < 2; d1++)
#pragma unroll
                    for (int d2 = 0; d2 < 2; d2++) v[d1][d2] = pmul(v[d1][d2], ph.re[0][0], ph.im[0][0]);
            }
            if (g1) {
                asm volatile("");   // branches: few cells have ghost corners
                v[1][0] = pmul(v[1][0], ph.re[1][0], ph.im[1][0]);
                v[1][1] = pmul(v[1][1], ph.re[1][0], ph.im[1][0]);
            }
            if (g2) {
                asm volatile("");
                v[0][1] = pmul(v[0][1], ph.re[2][0], ph.im[2][0]);
                v[1][1] = pmul(v[1][1], ph.re[2][0], ph.im[2][0]);
            }
        }
        const RT h = (RT)0.5;
#pragma unroll
        for (int d1 = 0; d1 < 2; d1++) v[d1][1] = vmul(vadd(v[d1][0], v[d1][1]), h);
#pragma unroll
        for (int d2 = 0; d2 < 2; d2++) {
            y[0][d2] = v[0][d2];
            y[1][d2] = vmul(vadd(v[0][d2], v[1][d2]), h);
        }
    };

    // The pair (p, p + 1), P = p + skip odd: wrap flags of both planes; the
    // coarse plane behind p and before p + 1, its staged index, and whether it
    // is the periodic ghost for p.
    struct Pair {
        int f[2], k;
        bool ghost, zero;
        i64 at[2];
    };
    auto pair_of = [&](int p) -> Pair {
        Pair s;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            int q = p + u;
            s.f[u] = q >= -n0 && q < n0 + R ? wrap_index(q, n0, g.per[0]) : 3;
            s.at[u] = s.f[u] == 3 ? 0 : (i64)q * plane;
        }
        s.k = ((p + 1 + pc.skip[0]) >> 1) - pc.lo[0];
        s.ghost = false;
        if (g.per[0]) {
            // p's own period decides: p = n0 - 1 or -1 reads the ghost of plane 0
            s.ghost = s.k == pc.nc[0] || s.k == 0;
            s.k = s.k < 0 ? s.k + pc.nc[0] : s.k >= pc.nc[0] ? s.k - pc.nc[0] : s.k;
        }
        s.zero = s.k < 0 || s.k >= pc.nc[0];
        return s;
    };
    V Y[2][2];
#pragma unroll
    for (int d1 = 0; d1 < 2; d1++)
#pragma unroll
        for (int d2 = 0; d2 < 2; d2++) Y[d1][d2] = vzero<V>();
    V bpre[2][2][2];
    auto load_base = [&](const Pair& s) {
        if (BASE && cell) {
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int d1 = 0; d1 < 2; d1++)
#pragma unroll
                    for (int d2 = 0; d2 < 2; d2++)
                        bpre[u][d1][d2] = b[s.at[u] + eo[d1][d2]];
        }
    };
    // F of the pair from the staged plane into ring slots s0, s1
    auto make = [&](const Pair& s, int s0, int s1) {
        if (!cell) return;
        V y[2][2], yo[2][2];
        yz(false, y);
        if (VT<V>::cplx && s.ghost) {
            yz(true, yo);
        } else {
#pragma unroll
            for (int d1 = 0; d1 < 2; d1++)
#pragma unroll
                for (int d2 = 0; d2 < 2; d2++) yo[d1][d2] = y[d1][d2];
        }
        V f[2][2][2];
#pragma unroll
        for (int d1 = 0; d1 < 2; d1++)
#pragma unroll
            for (int d2 = 0; d2 < 2; d2++) {
                f[0][d1][d2] = vmul(vadd(Y[d1][d2], yo[d1][d2]), (RT)0.5);
                f[1][d1][d2] = Y[d1][d2] = y[d1][d2];
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    if (BASE) f[u][d1][d2] = vsub(vmul(bpre[u][d1][d2], (RT)cb), f[u][d1][d2]);
                    if (s.f[u] == 3) f[u][d1][d2] = vzero<V>();
                }
            }
        if constexpr (VT<V>::cplx) {   // F's own ghosts: phases in axis order
            auto phase = [&](int u, int axis, int fl) {
                const double pr = fl == 1 ? ph.re[axis][0] : ph.re[axis][1];
                const double pi = fl == 1 ? ph.im[axis][0] : ph.im[axis][1];
#pragma unroll
                for (int d1 = 0; d1 < 2; d1++)
#pragma unroll
                    for (int d2 = 0; d2 < 2; d2++) f[u][d1][d2] = pmul(f[u][d1][d2], pr, pi);
            };
#pragma unroll
            for (int u = 0; u < 2; u++)
                if (s.f[u] == 1 || s.f[u] == 2) phase(u, 0, s.f[u]);
            if (f1) {
                asm volatile("");
                phase(0, 1, f1);
                phase(1, 1, f1);
            }
            if (f2) {
                asm volatile("");
                phase(0, 2, f2);
                phase(1, 2, f2);
            }
        }
#pragma unroll
        for (int d1 = 0; d1 < 2; d1++)
#pragma unroll
            for (int d2 = 0; d2 < 2; d2++)
                if (el[d1][d2] >= 0) {
                    ring[s0 * PS + el[d1][d2]] = f[0][d1][d2];
                    ring[s1 * PS + el[d1][d2]] = f[1][d1][d2];
                }
    };
    auto stage = [&](const Pair& s, V raw) {
        if (tid < CW * CH) C[tid] = (coff < 0 || s.zero) ? vzero<V>() : raw;
    };
    auto raw_of = [&](const Pair& s) -> V {
        return e[coff < 0 || s.zero ? 0 : s.k * cplane + coff];
    };
    if (!g.per[1] || !g.per[2]) {   // cells beyond a zero boundary stay zero
        for (int i = tid; i < NP * PS; i += NT) ring[i] = vzero<V>();
        __syncthreads();
    }
    // the first pair of planes whose stencil this block evaluates (it may
    // begin one plane early) and the planes before it: R pairs, behind one
    // coarse plane whose passes only start Y.  Plane ib - R + j goes to slot
    // j % NP; the own values of the first R planes stay in prev.
    const int ib = i0s - ((i0s + R + pc.skip[0] + 1) & 1);
    V prev[R];
    {
        V raw[R + 1];
        Pair s[R + 1];
#pragma unroll
        for (int m = 0; m <= R; m++) {
            s[m] = pair_of(ib - R - 2 + 2 * m);
            raw[m] = raw_of(s[m]);
        }
#pragma unroll
        for (int m = 0; m <= R; m++) {
            if (m > 0) load_base(s[m]);
            stage(s[m], raw[m]);
            __syncthreads();
            if (m == 0) {
                if (cell) yz(false, Y);
            } else {
                make(s[m], (2 * m - 2) % NP, (2 * m - 1) % NP);
            }
            __syncthreads();
            if (m > 0) {
#pragma unroll
                for (int j = 2 * m - 2; j < 2 * m; j++)
                    if (j < R) prev[j] = ring[j % NP * PS + lbase];
            }
        }
    }
    Pair pr = pair_of(ib + R);
    V raw = raw_of(pr), res[2], sn[2];
    load_base(pr);
    auto load_aux = [&](int i0) {
#pragma unroll
        for (int u = 0; u < 2; u++)
            sn[u] = sa[i0 + u >= 0 && i0 + u < n0 ? (i64)(i0 + u) * plane + poff : 0];
    };
    load_aux(ib);
    auto store = [&](int i0) {
#pragma unroll
        for (int u = 0; u < 2; u++)
            if (own && i0 + u >= i0s && i0 + u < i0e) o[(i64)(i0 + u) * plane + poff] = res[u];
    };
    auto wrap = [](int s) { return s >= NP ? s - NP : s; };
    int rs = R % NP;   // slot of plane i0
    for (int i0 = ib; i0 < i0e; i0 += 2) {
        vtouch(raw);
        vtouch(sn[0]);
        vtouch(sn[1]);
        if (BASE) {
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int d1 = 0; d1 < 2; d1++)
#pragma unroll
                    for (int d2 = 0; d2 < 2; d2++) vtouch(bpre[u][d1][d2]);
        }
        const V s[2] = {sn[0], sn[1]};
        stage(pr, raw);
        if (i0 > ib) store(i0 - 2);
        const Pair cur = pr;
        if (!BASE && i0 + 2 < i0e) {
            pr = pair_of(i0 + 2 + R);
            raw = raw_of(pr);
            load_aux(i0 + 2);
        }
        __syncthreads();   // the staged plane; everyone is done with the slots written next
        make(cur, wrap(rs + R), wrap(rs + R + 1));
        if (BASE && i0 + 2 < i0e) {   // the pair's base values were consumed by make
            pr = pair_of(i0 + 2 + R);
            raw = raw_of(pr);
            load_base(pr);
            load_aux(i0 + 2);
        }
        __syncthreads();
        const V* pl[NP];   // plane i0 + j at this thread's point
        V col[2 * R + 2];  // its values at planes i0 - R .. i0 + R + 1
#pragma unroll
        for (int j = 0; j < NP; j++) pl[j] = ring + wrap(rs + j) * PS + lbase;
#pragma unroll
        for (int j = 0; j < R; j++) col[j] = prev[j];
#pragma unroll
        for (int j = 0; j < NP; j++) col[R + j] = pl[j][0];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const V* row = pl[u];
            V x = vmac(vzero<V>(), col[R + u], (RT)sc.c[0]);
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
            res[u] = st_epilogue<MODE>(x, col[R + u], s[u], (RT)w, (RT)sc.c[0]);
        }
#pragma unroll
        for (int j = 0; j < R; j++) prev[j] = col[j + 2];
        rs = wrap(rs + 2);
    }
    if (i0e > i0s) store(ib + (i0e - 1 - ib) / 2 * 2);
}

}  // namespace gpaw
