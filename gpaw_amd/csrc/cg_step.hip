// CG direction step of the mixed-precision Poisson solve (gfx950):
//   phi -= alpha p          (the step the previous iteration left pending)
//   p'   = z + beta p       (beta: Polak-Ribiere, as in k_p_update)
//   q    = L p'             with the partials of p'.q
// for a star operator, in the one-shot box kernel's form (stencil_box.h): a
// block of 32 x TY threads owns a tile of Q planes, loads p and z over its
// column and in-plane halo and forms p' there.  p' goes to another array, as
// the neighbours still read p.
//
// Bound by memory: on 159^3 (32 MB a field) p and phi are read once and
// phi, p', q written, 176 MB with the FP32 z; the separate launches also read p
// once more for phi and p' once more for the operator (16.7 + 21.8 us and
// 14 us of the update that subtracted alpha p).  Each point is rounded as in the
// separate launches; z.q is summed by 512 threads in the larger tiles and p.q over
// other blocks, so beta and alpha can differ from theirs in the last bits.
#include "cg_step.h"
#include "stencil_box.h"

namespace gpaw {

namespace {

template <int R, int Q, int TY>
struct CgGeom {
    static constexpr int TZ = BOX_TZ, NT = TZ * TY;
    static constexpr int LW = TZ + 2 * R, LH = TY + 2 * R;
    static constexpr int NHALO = 2 * R * (TZ + TY), NH = (NHALO + NT - 1) / NT;
    static constexpr int LDS = Q * LH * LW;
};

// Tiles of 32 x 16 x 8 points where there is one for every CU, else 32 x 8 x 4:
// the larger one reads 2.3 instead of 3.4 values per point of p and z (from the
// L2 beyond the first).  159^3, a solve of 11 steps: 2574 us with 32 x 16 x 8,
// 2594 with 32 x 8 x 8, 2623 with 32 x 16 x 4, 2630 with 32 x 8 x 4; 127^3 1663
// against 1701, 111^3 1427 against 1429, 95^3 (216 of the larger) 1168 both.
bool cg_shape(const Geom& g, int R, int& Q, int& TY, TileShape& sh)
{
    const long tz = (g.n[2] + BOX_TZ - 1) / BOX_TZ;
    const bool large = tz * ((g.n[1] + 15) / 16) * ((g.n[0] + 7) / 8) >= 256;
    Q = large ? 8 : 4;
    TY = large ? 16 : 8;
    if (!box_geometry(g, R, 1, Q, sh)) return false;
    sh.nty = (g.n[1] + TY - 1) / TY;
    sh.nblocks = sh.ntz * sh.nty * sh.nchunk;
    return sh.nty * TY + R <= 2 * g.n[1];   // one wrap, for the taller tile too
}

// sum_partials of the solver, for a block of 32 x TY threads (in k_red1's order
// with 8 rows)
template <int NT>
__device__ __forceinline__ double sum_tid(const double* __restrict__ p, int n, int tid, double* red)
{
    double t = 0.0;
    for (int i = tid; i < n; i += NT) t += p[i];
    return block_sum<NT>(t, red);
}

template <class T, int R, bool UPD, int Q, int TY>
__global__ __launch_bounds__(32 * TY) void k_cg_dir(CgStep s, const T* __restrict__ z, Geom g,
                                                   TileCoefs sc, TileShape sh)
{
    typedef CgGeom<R, Q, TY> BG;
    constexpr int TZ = BG::TZ, NT = BG::NT, LW = BG::LW, LH = BG::LH, NHALO = BG::NHALO,
                  NH = BG::NH;
    __shared__ double lds[BG::LDS];
    __shared__ double red[NT];
    const double* __restrict__ a = s.p_in;
    double* __restrict__ pn = s.p_out;
    double* __restrict__ o = s.q;
    double* __restrict__ phi = s.phi;

    const int b = blockIdx.x;
    const int t = xcd_tile(b, sh.nblocks);
    const int tzi = t % sh.ntz;
    int rest = t / sh.ntz;
    const int tyb = rest % sh.nty;
    const int ch = rest / sh.nty;
    const int tx = threadIdx.x, tyi = threadIdx.y;
    const int tid = tx + TZ * tyi;
    const int n0 = g.n[0];
    const i64 plane = (i64)g.n[1] * g.n[2];
    const int z0 = tzi * TZ, y0 = tyb * TY;
    const int i0s = ch * Q;
    const bool inr = (y0 + tyi < g.n[1]) && (z0 + tx < g.n[2]);
    const PlaneRef qr = plane_ref(y0 + tyi, z0 + tx, g);

    int hoff[NH];
    PlaneRef hr[NH];
#pragma unroll
    for (int k = 0; k < NH; k++) {
        const int h = tid + NT * k;
        int lr, lc;
        if (h < 2 * R * TZ) {
            const int yr = h / TZ;
            lc = R + h % TZ;
            lr = yr < R ? yr : TY + yr;
        } else {
            const int hh = h - 2 * R * TZ;
            const int zc = hh % (2 * R);
            lr = R + hh / (2 * R);
            lc = zc < R ? zc : TZ + zc;
        }
        hoff[k] = (h < NHALO) ? lr * LW + lc : -1;
        hr[k] = (h < NHALO) ? plane_ref(y0 + lr - R, z0 + lc - R, g) : 0;
    }

    // every load first (planes past the grid load a valid address)
    double q[Q + 2 * R], hq[Q][NH], pv[Q], own[Q];
    T zq[Q + 2 * R], hz[Q][NH];
    int qf[Q + 2 * R];
#pragma unroll
    for (int p = 0; p < Q + 2 * R; p++) {
        int j = i0s - R + p;
        qf[p] = wrap_index(j, n0, g.per[0]);
        const i64 at = (qf[p] == 3 ? 0 : (i64)j * plane) + pref_off(qr);
        q[p] = a[at];
        zq[p] = z[at];
    }
#pragma unroll
    for (int p = 0; p < Q; p++) {
        const i64 base = qf[R + p] == 3 ? 0 : (i64)(i0s + p - (qf[R + p] == 1 ? n0 : 0)) * plane;
#pragma unroll
        for (int k = 0; k < NH; k++) {
            hq[p][k] = a[base + pref_off(hr[k])];
            hz[p][k] = z[base + pref_off(hr[k])];
        }
        if (UPD) {
            const bool ok = inr && i0s + p < n0;
            pv[p] = phi[ok ? (i64)(i0s + p) * plane + pref_off(qr) : 0];
        }
    }
    // the scalars, while the loads are in flight
    if (s.hist && b == 0) {
        const double v = sum_tid<NT>(s.dd, s.ndd, tid, red);
        if (tid == 0) *s.hist = v;
    }
    const double dzo = s.S[s.idz], alpha = s.S[s.ia];
    const bool f = dzo == 0.0;   // a (re)start: p' = z
    const double zqs = f ? 0.0 : sum_tid<NT>(s.zq, s.nzq, tid, red);
    const double beta = f ? 0.0 : -alpha * zqs / dzo;
#pragma unroll
    for (int p = 0; p < Q; p++) own[p] = q[R + p];
    auto dir = [&](double pe, T ze, int fl, PlaneRef r) -> double {
        const double v = f ? (double)ze : (double)ze + beta * pe;
        return ghost_fix(v, fl, r, Phases{});
    };
#pragma unroll
    for (int p = 0; p < Q + 2 * R; p++) q[p] = dir(q[p], zq[p], qf[p], qr);
#pragma unroll
    for (int p = 0; p < Q; p++) {
        double* B = lds + p * (LH * LW);
        B[(R + tyi) * LW + R + tx] = q[R + p];
#pragma unroll
        for (int k = 0; k < NH; k++)
            if (hoff[k] >= 0) B[hoff[k]] = dir(hq[p][k], hz[p][k], qf[R + p], hr[k]);
    }
    __syncthreads();

    double acc = 0.0;
#pragma unroll
    for (int p = 0; p < Q; p++) {
        const double* row = lds + p * (LH * LW) + (R + tyi) * LW + R + tx;
        const double fv = q[R + p];
        double x = vmac(0.0, fv, sc.c[0]);
#pragma unroll
        for (int k = 1; k <= R; k++) x = vmac(x, row[k], sc.c[k]);
#pragma unroll
        for (int k = 1; k <= R; k++) x = vmac(x, row[-k], sc.c[R + k]);
#pragma unroll
        for (int k = 1; k <= R; k++) x = vmac(x, row[k * LW], sc.c[2 * R + k]);
#pragma unroll
        for (int k = 1; k <= R; k++) x = vmac(x, row[-k * LW], sc.c[3 * R + k]);
#pragma unroll
        for (int k = 1; k <= R; k++) x = vmac(x, q[R + p + k], sc.c[4 * R + k]);
#pragma unroll
        for (int k = 1; k <= R; k++) x = vmac(x, q[R + p - k], sc.c[5 * R + k]);
        if (inr && i0s + p < n0) {
            const i64 at = (i64)(i0s + p) * plane + pref_off(qr);
            o[at] = x;
            pn[at] = fv;
            if (UPD) phi[at] = pv[p] - alpha * own[p];
            acc += tdot(fv, x);
        }
    }
    const double sum = block_sum<NT>(acc, red);
    if (tid == 0) s.partial[b] = sum;
}

template <class T, int R, bool UPD>
hipError_t cg_go(const Stencil& st_, const Geom& g, const CgStep& a, const void* z,
                 hipStream_t st)
{
    TileCoefs sc;
    for (int c = 0; c < 6 * R + 1; c++) sc.c[c] = st_.coefs[c];
    TileShape sh;
    int Q = 0, TY = 0;
    if (!cg_shape(g, R, Q, TY, sh)) return hipErrorInvalidValue;
    if (TY == 16)
        launch_kernel((k_cg_dir<T, R, UPD, 8, 16>), dim3(sh.nblocks), dim3(BOX_TZ, 16), 0, st, a,
                      (const T*)z, g, sc, sh);
    else
        launch_kernel((k_cg_dir<T, R, UPD, 4, 8>), dim3(sh.nblocks), dim3(BOX_TZ, 8), 0, st, a,
                      (const T*)z, g, sc, sh);
    return launch_error();
}

template <class T, bool UPD>
hipError_t cg_r(const Stencil& s, const Geom& g, const CgStep& a, const void* z, hipStream_t st)
{
    switch (s.star_r) {
    case 1: return cg_go<T, 1, UPD>(s, g, a, z, st);
    case 2: return cg_go<T, 2, UPD>(s, g, a, z, st);
    case 3: return cg_go<T, 3, UPD>(s, g, a, z, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace

bool cg_dir_ok(const Stencil& s, const Geom& g, int* npartial)
{
    TileShape sh;
    int Q = 0, TY = 0;
    if (s.star_r < 1 || s.star_r > 3 || !cg_shape(g, s.star_r, Q, TY, sh)) return false;
    *npartial = sh.nblocks;
    return sh.nblocks <= stencil_partials(s, g, 1);
}

hipError_t launch_cg_dir(const Stencil& s, const Geom& g, const CgStep& a, const void* z,
                         int zdtype, hipStream_t st)
{
    int np = 0;
    if (!cg_dir_ok(s, g, &np) || a.p_in == a.p_out) return hipErrorInvalidValue;
    if (zdtype == DT_F32)
        return a.phi ? cg_r<float, true>(s, g, a, z, st) : cg_r<float, false>(s, g, a, z, st);
    if (zdtype == DT_F64)
        return a.phi ? cg_r<double, true>(s, g, a, z, st) : cg_r<double, false>(s, g, a, z, st);
    return hipErrorInvalidValue;
}

}  // namespace gpaw
