// Multigrid preconditioner of the finite-difference eigensolvers
// (gpaw/preconditioner.py:13-70) as one stream-ordered sequence of launches
// over all bands at once.
//
// The reference evaluates, per call (r = residuals, s = step):
//   r1 = R0(-r);  d1 = 4s r1;  q1 = L1 d1 - r1
//   r2 = R1(q1);  d2 = 16s r2; q2 = L2 d2 - r2;  d2 -= 16s q2
//   d1 -= I2(d2); q1 = L1 d1 - r1;  d1 -= 4s q1
//   d0 = I1(-d1); q0 = L0 d0 - r;   d0 += -s q0;  d0 *= -1
// Restriction, interpolation and the stencils are linear and round
// symmetrically, so R0(-r) == -R0(r) and I1(-d1) == -I1(d1) bit for bit.
// With e0 = I1(d1) = -d0 the last line becomes e0 - s (L0 e0 + r), which is
// one fused stencil pass (ST_PCFIN); the two "d -= w (L d - r)" updates are
// ST_PCUPD passes and "d1 -= I2(d2)" is the subtracting interpolation.
// Every value is rounded exactly where the reference's numpy / BLAS steps
// round it (BLAS axpy evaluated as y + (a x), without a fused multiply-add).
//
// Six launches where the levels allow it (pc_scaled, pc_interp): d1 = 4s r1, d2 = 16s r2,
// d1 - I2(d2) and e0 = I1(d1) are formed inside the stencil passes that read
// them (precond_sweep.h), so E0, D1 and D2 are never stored; 4.2 instead of
// 7.4 GB on 256 complex128 bands of 64^3.  A pass that cannot be fused runs
// its steps one by one.
//
// Buffers (caller's workspace, one slice per band, 256-byte aligned):
//   level 0: E0;  level 1: R1, D1, Q1;  level 2: R2, D2, X2.
#include "capi_internal.h"
#include "precond_sweep.h"

namespace gpaw {

// d = c * r over n doubles (complex data counted as pairs)
__global__ __launch_bounds__(256) void k_pc_scale(const double* __restrict__ r,
                                                  double* __restrict__ d, double c, i64 n)
{
    const i64 i = (i64)blockIdx.x * 256 + threadIdx.x;
    if (i < n) d[i] = c * r[i];
}

namespace {

// Runs of the whole i0 axis, split towards 1024 blocks where there are too few
// tiles, each of at least `run` planes: a small set waits on a block's serial
// planes, but a run reads 2 R more and one of k_pc_interp starts with R + 1
// coarse planes of two barriers each.  2 planes for k_pc_scaled, 4 for
// k_pc_interp with b and 8 without: real 3 bands of 79 x 63 x 71, a call in
// 40.7 us, with 8 planes in all three 50.4, 4 / 8 / 8 44.7, 2 / 2 / 8 42.5;
// complex128 24 x 64^3 145, 149, 147, 150; 16 x 32^3 54, 56, 54, 56; 6 or 4
// planes without b: 59 or 54.5, real 8 x 64^3 48.6 or 47.3 instead of 45.
bool pc_shape(const Geom& g, int R, int esize, int nin, int nt, int run, TileShape* sh,
              int TZ = 32)
{
    if (!tile_geometry(g, R, esize, nin, TZ, g.n[0], *sh, nt)) return false;
    long nch = (1024L + sh->nblocks - 1) / sh->nblocks;
    const long maxch = g.n[0] / run > 1 ? g.n[0] / run : 1;
    if (nch > maxch) nch = maxch;
    return tile_geometry(g, R, esize, nin, TZ, (int)((g.n[0] + nch - 1) / nch), *sh, nt);
}

TileCoefs pc_coefs(const Stencil& s)
{
    TileCoefs sc{};
    for (int c = 0; c < 6 * s.star_r + 1; c++) sc.c[c] = s.coefs[c];
    return sc;
}

i64 pc_points(const int n[3]) { return (i64)n[0] * n[1] * n[2]; }

// out = mode(L F, aux b) with F = c b; hipErrorNotSupported (nothing launched)
// where k_pc_scaled does not run: it takes range-1 stars whose halo wraps once,
// complex data from 2^15 points in all (below, one tile's serial planes take
// longer than the two short launches: 8 bands of 13 x 11 x 17, a call of 50
// instead of 46 us).
template <class V, int TZ>
hipError_t pc_scaled_go(const gpaw_operator* L, int mode, const void* b, void* out,
                        const Phases& ph, double cb, double w, const TileShape& sh, hipStream_t st)
{
    const dim3 grid(sh.nblocks), block(TZ, TILE_NT / TZ);
    const TileCoefs sc = pc_coefs(L->st);
    const i64 ng = pc_points(L->g.n);
    if (mode == ST_RESID)
        return launch_kernel((k_pc_scaled<V, 1, ST_RESID, TILE_NT, TZ>), grid, block, 0, st,
                             (const V*)b, (V*)out, L->g, ph, sc, cb, w, sh, ng);
    return launch_kernel((k_pc_scaled<V, 1, ST_PCUPD, TILE_NT, TZ>), grid, block, 0, st,
                         (const V*)b, (V*)out, L->g, ph, sc, cb, w, sh, ng);
}

template <class V>
hipError_t pc_scaled(const gpaw_operator* L, int mode, const void* b, void* out, int nin,
                     const Phases& ph, double cb, double w, hipStream_t st)
{
    TileShape sh;
    if (VT<V>::cplx && nin * pc_points(L->g.n) < 1 << 15) return hipErrorNotSupported;
    if (L->st.star_r != 1) return hipErrorNotSupported;
    // rows of up to 16 points (level 2 of a 64^3 grid) in tiles of 16 x 16: a tile
    // of 32 would wrap twice, and the two separate launches took 21 us on 256
    // complex128 bands of 16^3, now 10 (a call 934 -> 923; 2 real bands of 48 x 64 x
    // 40 32.5 -> 29.5)
    if (L->g.n[2] <= 16 && pc_shape(L->g, 1, (int)sizeof(V), nin, TILE_NT, 2, &sh, 16))
        return pc_scaled_go<V, 16>(L, mode, b, out, ph, cb, w, sh, st);
    if (pc_shape(L->g, 1, (int)sizeof(V), nin, TILE_NT, 2, &sh))
        return pc_scaled_go<V, 32>(L, mode, b, out, ph, cb, w, sh, st);
    return hipErrorNotSupported;
}

// out = mode(L F, aux) with F = I e (b null) or c b - I e; hipErrorNotSupported
// where k_pc_interp cannot run: it takes K = 2, stars of range 1 .. 3 (1 with
// b), halos that wrap once, and on periodic axes grids twice the coarser one.
template <class V, int R, bool BASE, int MODE, int TY>
hipError_t pc_interp_go(const gpaw_operator* L, const Transfer& t, const void* b, const void* e,
                        void* out, const void* aux, int nin, const Phases& ph, double cb, double w,
                        hipStream_t st)
{
    const Geom& g = L->g;
    TileShape sh;
    if (!pc_shape(g, R, (int)sizeof(V), nin, 32 * TY, BASE ? 4 : 8, &sh)) return hipErrorNotSupported;
    PcCoarse pc;
    for (int a = 0; a < 3; a++) {
        pc.nc[a] = t.gin.n[a];
        pc.skip[a] = t.skip[a][0];
        pc.lo[a] = t.lo[a];
    }
    return launch_kernel((k_pc_interp<V, R, BASE, MODE, TY>), dim3(sh.nblocks), dim3(32, TY), 0, st,
                         (const V*)b, (const V*)e, (V*)out, (const V*)aux, g, ph, pc,
                         pc_coefs(L->st), cb, w, sh, pc_points(g.n), pc_points(pc.nc));
}

template <class V>
hipError_t pc_interp(const gpaw_operator* L, const Transfer& t, const void* b, const void* e,
                     void* out, const void* aux, int nin, const Phases& ph, double cb, double w,
                     hipStream_t st)
{
    const Geom& g = L->g;
    const int R = L->st.star_r;
    if (t.K != 2 || R < 1 || R > (b ? 1 : 3)) return hipErrorNotSupported;
    for (int a = 0; a < 3; a++) {
        if (t.nout[a] != g.n[a] || t.gin.per[a] != g.per[a] || g.n[a] < 2 * R + 2)
            return hipErrorNotSupported;
        if (g.per[a] && (t.nout[a] != 2 * t.gin.n[a] || t.skip[a][0] || t.lo[a]))
            return hipErrorNotSupported;
    }
    const i64 points = nin * pc_points(g.n);
    // complex bands below 2^18 points in all: every launch is a few us there, and
    // a block's serial planes cost what the launch saved (1 / 4 / 16 bands of
    // 32^3: 49 / 51 / 54 us fused, 47 / 50 / 58 in steps); real bands gain on most
    // grids (3 bands of 79 x 63 x 71: 38 us instead of 41, one of 96^3: 33 instead
    // of 37)
    if (VT<V>::cplx && points < 1 << 18) return hipErrorNotSupported;
    // the level-0 pass of wider stencils where there is little to read: real rows
    // of one tile (7 bands of 23 x 27 x 27: 32.6 us a call in steps, 36.9 fused; 24
    // such grids 4 % slower fused), complex bands between walls (12 bands of
    // 47 x 19 x 59: 52.5 and 55; 11 such grids 2 %; from 2^21 points fused is faster)
    if (!b && !VT<V>::cplx && R > 1 && g.n[2] <= 32 && points < 1 << 18) return hipErrorNotSupported;
    if (!b && VT<V>::cplx && R > 2 && !g.per[0] && points < 1 << 21) return hipErrorNotSupported;
    // 16 rows per block on large sets where they pad no more rows than 8 do
    // (complex128, 256 x 64^3: 1075 us a call with 8, 1001 with 16, 1009 with 32
    // rows; 64 x 32^3: 90 with 8, 82 with 16; real 16 x 48^3: 47 with 8, 50 with 16)
    const bool tall = points >= 1 << 21 && (g.n[1] + 15) / 16 * 2 == (g.n[1] + 7) / 8;
    hipError_t r = hipErrorNotSupported;
#define GPAW_PC_INTERP(RR, B, M)                                                                  \
    if (tall) r = pc_interp_go<V, RR, B, M, 16>(L, t, b, e, out, aux, nin, ph, cb, w, st);        \
    if (r == hipErrorNotSupported)                                                                \
        r = pc_interp_go<V, RR, B, M, 8>(L, t, b, e, out, aux, nin, ph, cb, w, st);
    if (b) {
        GPAW_PC_INTERP(1, true, ST_PCUPD)
    } else if (R == 1) {
        GPAW_PC_INTERP(1, false, ST_PCFIN)
    } else if (R == 2) {
        GPAW_PC_INTERP(2, false, ST_PCFIN)
    } else {
        GPAW_PC_INTERP(3, false, ST_PCFIN)
    }
#undef GPAW_PC_INTERP
    return r;
}

}  // namespace

}  // namespace gpaw

using namespace gpaw;

struct gpaw_preconditioner {
    gpaw_operator* kin[3];
    gpaw_transformer* rst[2];   // level 0 -> 1, 1 -> 2
    gpaw_transformer* ip[2];    // level 2 -> 1, 1 -> 0
    double step;
    i64 ng[3];
};

static i64 npts(const int n[3]) { return (i64)n[0] * n[1] * n[2]; }

static bool same(const int a[3], const int b[3])
{
    return a[0] == b[0] && a[1] == b[1] && a[2] == b[2];
}

extern "C" int gpaw_preconditioner_new(gpaw_operator* kin0, gpaw_operator* kin1,
                                       gpaw_operator* kin2, gpaw_transformer* restrictor0,
                                       gpaw_transformer* restrictor1,
                                       gpaw_transformer* interpolator2,
                                       gpaw_transformer* interpolator1,
                                       gpaw_preconditioner** out)
{
    if (!out) return gpaw_fail(GPAW_EINVAL, "preconditioner: NULL argument");
    *out = nullptr;
    if (!kin0 || !kin1 || !kin2 || !restrictor0 || !restrictor1 || !interpolator2 ||
        !interpolator1)
        return gpaw_fail(GPAW_EINVAL, "preconditioner: NULL operator or transformer");
    const Transfer &r0 = restrictor0->t, &r1 = restrictor1->t;
    const Transfer &i2 = interpolator2->t, &i1 = interpolator1->t;
    if (r0.interpolate || r1.interpolate || !i2.interpolate || !i1.interpolate)
        return gpaw_fail(GPAW_EINVAL,
                         "preconditioner: expects two restrictions and two interpolations");
    if (!same(kin0->g.n, r0.gin.n) || !same(r0.nout, kin1->g.n) || !same(kin1->g.n, r1.gin.n) ||
        !same(r1.nout, kin2->g.n) || !same(kin2->g.n, i2.gin.n) || !same(i2.nout, kin1->g.n) ||
        !same(kin1->g.n, i1.gin.n) || !same(i1.nout, kin0->g.n))
        return gpaw_fail(GPAW_EINVAL, "preconditioner: grid sizes of the levels do not chain");
    const int real = kin0->real;
    if (kin1->real != real || kin2->real != real || restrictor0->real != real ||
        restrictor1->real != real || interpolator2->real != real || interpolator1->real != real)
        return gpaw_fail(GPAW_EINVAL, "preconditioner: mixed real and complex objects");
    if (kin0->diag == 0.0)
        return gpaw_fail(GPAW_EINVAL, "preconditioner: kin0 has no diagonal element");
    gpaw_preconditioner* pc = new gpaw_preconditioner();
    pc->kin[0] = kin0;
    pc->kin[1] = kin1;
    pc->kin[2] = kin2;
    pc->rst[0] = restrictor0;
    pc->rst[1] = restrictor1;
    pc->ip[0] = interpolator2;
    pc->ip[1] = interpolator1;
    pc->step = 0.66666666 / kin0->diag;   // gpaw/preconditioner.py:24
    for (int l = 0; l < 3; l++) pc->ng[l] = npts(pc->kin[l]->g.n);
    *out = pc;
    return GPAW_OK;
}

extern "C" double gpaw_preconditioner_step(const gpaw_preconditioner* pc)
{
    return pc ? pc->step : 0.0;
}

static size_t slice_bytes(i64 n, long nin, int dtype)
{
    const size_t b = (size_t)n * (size_t)nin * (size_t)dtype_size(dtype);
    return (b + 255) & ~(size_t)255;
}

static size_t workspace_bytes(const gpaw_preconditioner* pc, long nin, int dtype)
{
    return slice_bytes(pc->ng[0], nin, dtype) + 3 * slice_bytes(pc->ng[1], nin, dtype) +
           3 * slice_bytes(pc->ng[2], nin, dtype);
}

static int check_args(const gpaw_preconditioner* pc, long nin, int dtype)
{
    if (!pc) return gpaw_fail(GPAW_EINVAL, "preconditioner: NULL handle");
    if (dtype != GPAW_F64 && dtype != GPAW_C128)
        return gpaw_fail(GPAW_EUNSUPPORTED, "preconditioner: float64 or complex128 data only");
    int rc = gpaw_check_dtype(pc->kin[0]->real, dtype);
    if (rc) return rc;
    if (nin < 0 || nin > 65535) return gpaw_fail(GPAW_EINVAL, "preconditioner: nin = %ld", nin);
    return GPAW_OK;
}

extern "C" int gpaw_preconditioner_workspace(const gpaw_preconditioner* pc, long nin, int dtype,
                                             long* bytes)
{
    int rc = check_args(pc, nin, dtype);
    if (rc) return rc;
    if (!bytes) return gpaw_fail(GPAW_EINVAL, "preconditioner: NULL bytes");
    *bytes = (long)workspace_bytes(pc, nin, dtype);
    return GPAW_OK;
}

extern "C" int gpaw_preconditioner_apply(gpaw_preconditioner* pc, const void* residuals,
                                         void* out, long nin, int dtype, const double* phases,
                                         void* work, long work_bytes, void* stream)
{
    int rc = check_args(pc, nin, dtype);
    if (rc) return rc;
    if (nin == 0) return GPAW_OK;
    if (!residuals || !out || !work) return gpaw_fail(GPAW_EINVAL, "preconditioner: NULL array");
    if (residuals == out) return gpaw_fail(GPAW_EINVAL, "preconditioner: out must differ from residuals");
    if (work_bytes < 0 || (size_t)work_bytes < workspace_bytes(pc, nin, dtype))
        return gpaw_fail(GPAW_EINVAL, "preconditioner: workspace of %ld bytes, %zu needed",
                         work_bytes, workspace_bytes(pc, nin, dtype));
    if ((reinterpret_cast<uintptr_t>(work) & 255) != 0)
        return gpaw_fail(GPAW_EINVAL, "preconditioner: workspace must be 256-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    Phases ph;
    gpaw_phases(phases, ph);
    const int nb = (int)nin;
    char* free_ = (char*)work;
    auto take = [&](int l) {
        void* p = free_;
        free_ += slice_bytes(pc->ng[l], nin, dtype);
        return p;
    };
    void* E0 = take(0);
    void* R1 = take(1);
    void* D1 = take(1);
    void* Q1 = take(1);
    void* R2 = take(2);
    void* D2 = take(2);
    void* X2 = take(2);
    const int dpp = dtype_complex(dtype) ? 2 : 1;   // doubles per point
    const i64 n1 = pc->ng[1] * nin * dpp, n2 = pc->ng[2] * nin * dpp;
    const double s = pc->step, c1 = 4 * s, c2 = 16 * s;
    gpaw_operator *L0 = pc->kin[0], *L1 = pc->kin[1], *L2 = pc->kin[2];

    hipError_t e;
    auto scale = [&](const void* r, void* d, double c, i64 n) {
        return launch_kernel(k_pc_scale, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                             (const double*)r, (double*)d, c, n);
    };
    auto stencil = [&](const gpaw_operator* L, int mode, const void* in, void* o, const void* aux,
                       double c) {
        return launch_stencil(L->st, dtype, mode, in, o, aux, L->g, ph, nb, c, nullptr, nullptr,
                              true, st);
    };
    auto transfer = [&](const Transfer& t, int mode, const void* in, void* o) {
        return launch_transfer(t, dtype, mode, in, o, nullptr, ph, nb, st);
    };
    // the passes in one launch each or, where those kernels cannot run one
    // (hipErrorNotSupported, nothing launched), in its separate steps
    const bool real = !dtype_complex(dtype);
    auto scaled = [&](const gpaw_operator* L, int mode, const void* b, void* o, double c) {
        return real ? pc_scaled<double>(L, mode, b, o, nb, ph, c, c, st)
                    : pc_scaled<double2>(L, mode, b, o, nb, ph, c, c, st);
    };
    auto interp = [&](const gpaw_operator* L, const Transfer& t, const void* b, const void* x,
                      void* o, const void* aux, double c, double w) {
        return real ? pc_interp<double>(L, t, b, x, o, aux, nb, ph, c, w, st)
                    : pc_interp<double2>(L, t, b, x, o, aux, nb, ph, c, w, st);
    };
    bool d1 = false;   // D1 = 4s r1
    Transfer rneg = pc->rst[0]->t;
    rneg.negate = 1;
    e = transfer(rneg, TR_STORE, residuals, R1);   // r1 = -R0(r)
    if (e == hipSuccess) {   // q1 = L1 d1 - r1, d1 = 4s r1
        e = scaled(L1, ST_RESID, R1, Q1, c1);
        if (e == hipErrorNotSupported) {
            d1 = true;
            e = scale(R1, D1, c1, n1);
            if (e == hipSuccess) e = stencil(L1, ST_RESID, D1, Q1, R1, 0.0);
        }
    }
    if (e == hipSuccess) e = transfer(pc->rst[1]->t, TR_STORE, Q1, R2);   // r2 = R1(q1)
    if (e == hipSuccess) {   // x2 = d2 - 16s (L2 d2 - r2), d2 = 16s r2
        e = scaled(L2, ST_PCUPD, R2, X2, c2);
        if (e == hipErrorNotSupported) {
            e = scale(R2, D2, c2, n2);
            if (e == hipSuccess) e = stencil(L2, ST_PCUPD, D2, X2, R2, c2);
        }
    }
    if (e == hipSuccess) {   // q = d1 - 4s (L1 d1 - r1), d1 = 4s r1 - I2(x2)
        e = interp(L1, pc->ip[0]->t, R1, X2, Q1, R1, c1, c1);
        if (e == hipErrorNotSupported) {
            e = d1 ? hipSuccess : scale(R1, D1, c1, n1);
            if (e == hipSuccess) e = transfer(pc->ip[0]->t, TR_SUBTRACT, X2, D1);
            if (e == hipSuccess) e = stencil(L1, ST_PCUPD, D1, Q1, R1, c1);
        }
    }
    if (e == hipSuccess) {   // e0 - s (L0 e0 + r), e0 = I1(q) = -d0
        e = interp(L0, pc->ip[1]->t, nullptr, Q1, out, residuals, 0.0, s);
        if (e == hipErrorNotSupported) {
            e = transfer(pc->ip[1]->t, TR_STORE, Q1, E0);
            if (e == hipSuccess) e = stencil(L0, ST_PCFIN, E0, out, residuals, s);
        }
    }
    return gpaw_check(e, "preconditioner apply");
}

extern "C" void gpaw_preconditioner_free(gpaw_preconditioner* pc) { delete pc; }
