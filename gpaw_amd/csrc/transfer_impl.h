// Restriction / interpolation kernels and their launchers, instantiated
// once per storage type in transfer_<type>.hip.
//
// One thread produces one output point of one band; the arithmetic is the
// point-wise separable evaluation of transfer_common.h, bit-identical to the
// reference's three-sweep bmgs_restrict / bmgs_interpolate
// (c/bmgs/restrict.c:137-154, c/bmgs/interpolate.c:141-168).
// TR_SUBTRACT fuses the multigrid correction phi -= interpolate(e)
// (gpaw/poisson.py:263-264), and restriction can zero the next level's phi
// in the same pass (gpaw/poisson.py:259-261).
#pragma once
#include <cstdlib>
#include "kernels.h"
#include "transfer_common.h"
#include "transfer_tile.h"

namespace gpaw {

TrArgs make_trargs(const Transfer& tr);

template <class V, int K>
__global__ __launch_bounds__(256) void k_restrict(const V* __restrict__ in, V* __restrict__ out,
                                                  V* __restrict__ zero_out, TrArgs t, Phases ph)
{
    const i64 idx = (i64)blockIdx.x * 256 + threadIdx.x;
    if (idx >= t.ngout) return;
    const int o2 = (int)(idx % t.nout[2]);
    const int o1 = (int)((idx / t.nout[2]) % t.nout[1]);
    const int o0 = (int)(idx / ((i64)t.nout[1] * t.nout[2]));
    const V* __restrict__ a = in + (i64)blockIdx.y * t.ngin;
    const i64 o = (i64)blockIdx.y * t.ngout + idx;
    out[o] = neg_if(restrict_point<V, K>(a, o0, o1, o2, t, ph), t.negate);
    if (zero_out) zero_out[o] = vzero<V>();
}

template <class V, int K, int MODE>
__global__ __launch_bounds__(256) void k_interpolate(const V* __restrict__ in, V* __restrict__ out,
                                                     TrArgs t, Phases ph)
{
    const i64 idx = (i64)blockIdx.x * 256 + threadIdx.x;
    if (idx >= t.ngout) return;
    const int o2 = (int)(idx % t.nout[2]);
    const int o1 = (int)((idx / t.nout[2]) % t.nout[1]);
    const int o0 = (int)(idx / ((i64)t.nout[1] * t.nout[2]));
    const V* __restrict__ a = in + (i64)blockIdx.y * t.ngin;
    const V r = interp_point<V, K>(a, o0, o1, o2, t, ph);
    const i64 o = (i64)blockIdx.y * t.ngout + idx;
    if (MODE == TR_SUBTRACT)
        out[o] = vsub(out[o], r);
    else
        out[o] = r;
}

// K = 2 interpolation, one thread per coarse cell (interp2_cell).
template <class V, int MODE>
__global__ __launch_bounds__(256) void k_interp2(const V* __restrict__ in, V* __restrict__ out,
                                                 TrArgs t, int nc0, int nc1, int nc2, Phases ph)
{
    const i64 idx = (i64)blockIdx.x * 256 + threadIdx.x;
    const i64 ncell = (i64)nc0 * nc1 * nc2;
    if (idx >= ncell) return;
    const int k2 = (int)(idx % nc2);
    const int k1 = (int)((idx / nc2) % nc1);
    const int k0 = (int)(idx / ((i64)nc1 * nc2));
    interp2_cell<V, MODE>(in + (i64)blockIdx.y * t.ngin, out + (i64)blockIdx.y * t.ngout, t, k0,
                          k1, k2, ph);
}

// Tiles and i0 chunks of the tile kernels.  A block's planes are a serial
// chain of about 1 us each, so few bands on one chunk leave the chip idle:
// 2 x 127^3 -> 63^3 K = 6 is 32 blocks of 135 planes.  The axis is split, but every
// chunk sweeps 2 K - 3 (restriction; K - 1) planes again.
// Interpolation: until there are TR_BLOCKS_INTERP blocks (four per CU); 1 / 256 /
// 512 / 1024 / 2048 blocks on 2 x 63^3 -> 127^3, K = 6: 54 / 31 / 21 / 18.5 / 20 us.
// Restriction: until there are TR_BLOCKS_RESTRICT blocks (121 / 27 / 25 / 36 / 54 us on
// 2 x 127^3 -> 63^3), unless whole axes are estimated to take no longer; complex128,
// whose blocks fill the chip at 512, by the estimate alone.  On 2500 drawn
// grids of 40 .. 700 blocks complex128 loses 2 % to the best of 1 .. 8 chunks and never
// to whole axes; splitting it until there are 512 blocks lost 12 %, and on 156 of
// 974 to whole axes, for a few blocks more than a round (29 x 111x121x95 ->
// 55x59x47, 464 blocks: 178 us, in two chunks 220).  Other types lose 5 .. 7 %.
constexpr i64 TR_BLOCKS_RESTRICT = 512, TR_BLOCKS_INTERP = 1024;

// planes a restriction in chunks of cq sweeps one after another: rounds of
// `slots` blocks, the last one half as a whole one and half by its share
inline double restrict_planes(int n0, int cq, int K, i64 base, int slots, double more)
{
    const i64 b = base * ((n0 + cq - 1) / cq);
    const double rounds = 0.5 * ((double)((b + slots - 1) / slots) + (double)b / slots) + more;
    return (rounds > 1.0 ? rounds : 1.0) * (2 * cq + 2 * K - 3);
}

inline i64 restrict_chunks(int n0, int K, i64 base, bool c128)
{
    if (!c128) {
        i64 nch = (TR_BLOCKS_RESTRICT + base - 1) / base;
        if (nch > n0) nch = n0;
        const bool split = nch > 1 && restrict_planes(n0, (int)((n0 + nch - 1) / nch), K, base, 768, 0.25) <
                                          restrict_planes(n0, n0, K, base, 768, 0.25);
        return split ? nch : 1;
    }
    const double whole = restrict_planes(n0, n0, K, base, 512, 0.0);
    double least = 0.95 * whole;
    i64 best = 1;
    // each chunk length once, while there are at most four rounds
    for (int cq = n0; cq > 1;) {
        const int next = (n0 + cq - 2) / (cq - 1);
        cq = (n0 + next - 1) / next;
        const i64 nch = (n0 + cq - 1) / cq;
        if (base * nch > 2048) break;
        const double planes = restrict_planes(n0, cq, K, base, 512, 0.0);
        if (planes < least) {
            least = 0.97 * planes;
            best = nch;
        }
    }
    return best;
}

inline TileTr tile_tr(const TrArgs& t, bool interpolate, int nin, int K, bool c128)
{
    TileTr tt;
    tt.nt1 = (t.nout[1] + 7) / 8;
    tt.nt2 = (t.nout[2] + 31) / 32;
    const int n0 = interpolate ? interp2_cells(t, 0) : t.nout[0];   // outputs or centres
    const i64 base = (i64)tt.nt1 * tt.nt2 * nin;
    i64 nch = interpolate ? (TR_BLOCKS_INTERP + base - 1) / base
                          : restrict_chunks(n0, K, base, c128);
    if (nch > n0) nch = n0;
    tt.cq = (int)((n0 + nch - 1) / nch);
    tt.nch = (n0 + tt.cq - 1) / tt.cq;
    return tt;
}

template <class V, int K>
hipError_t tr_launch(const Transfer& tr, int mode, const void* in, void* out, void* zero_out,
                     const Phases& ph, int nin, hipStream_t st, double* sums = nullptr,
                     int* nsums = nullptr)
{
    const TrArgs t = make_trargs(tr);
    dim3 grid((unsigned)((t.ngout + 255) / 256), nin, 1);
    if (K == 2 && tr.interpolate) {
        // coarse cells covering every output: i from skip_lo/2 to (nout-1+skip_lo)/2
        int nc[3];
        for (int a = 0; a < 3; a++) nc[a] = interp2_cells(t, a);
        const i64 ncell = (i64)nc[0] * nc[1] * nc[2];
        dim3 g2((unsigned)((ncell + 255) / 256), nin, 1);
        if (mode == TR_SUBTRACT)
            launch_kernel((k_interp2<V, TR_SUBTRACT>), g2, dim3(256), 0, st, (const V*)in,
                               (V*)out, t, nc[0], nc[1], nc[2], ph);
        else
            launch_kernel((k_interp2<V, TR_STORE>), g2, dim3(256), 0, st, (const V*)in,
                               (V*)out, t, nc[0], nc[1], nc[2], ph);
        return launch_error();
    }
    // wide transfers on large planes, and K = 2 restrictions of many points
    // (band sets: the point-wise kernel reads each input up to 8 times through
    // the caches): LDS-tiled plane sweep (8 x 32 tiles)
    const bool big2 = K == 2 && !tr.interpolate && t.ngout * nin >= (1 << 20);
    if ((K >= 4 || big2) && t.nout[1] >= 4 && t.nout[2] >= 16 &&
        (long)t.gin.n[1] * t.gin.n[2] < PLANE_REF_MAX && !getenv("GPAW_AMD_POINTWISE_TRANSFER")) {
        const TileTr tt = tile_tr(t, tr.interpolate, nin, K, sizeof(V) == 16);
        const dim3 gt((unsigned)(tt.nt1 * tt.nt2 * tt.nch * nin));
        // chunked real restrictions (few blocks per CU) take two planes per
        // step: 25 us against 27 on 2 x 127^3 -> 63^3, K = 6; one plane is
        // faster where blocks hide each other's waits (256 x 64^3: 174 us
        // against 181), and complex slabs have no registers for two
        constexpr int PL2 = VT<V>::cplx ? 1 : 2;
        if (!tr.interpolate && tt.nch > 1)
            launch_kernel((k_restrict_tile<V, K, 8, 32, PL2>), gt, dim3(256), 0, st,
                               (const V*)in, (V*)out, t, tt, ph);
        else if (!tr.interpolate)
            launch_kernel((k_restrict_tile<V, K, 8, 32, 1>), gt, dim3(256), 0, st, (const V*)in,
                               (V*)out, t, tt, ph);
        else if (mode == TR_SUBTRACT)
            launch_kernel((k_interp_tile<V, K, 8, 32, TR_SUBTRACT>), gt, dim3(256), 0, st,
                               (const V*)in, (V*)out, t, tt, ph, (double*)nullptr);
        else {
            // partial sums of each function's outputs, where a row holds them
            const int np = tt.nt1 * tt.nt2 * tt.nch;
            double* s = sums && np <= SUM_PARTIALS ? sums : nullptr;
            if (s) *nsums = np;
            launch_kernel((k_interp_tile<V, K, 8, 32, TR_STORE>), gt, dim3(256), 0, st,
                               (const V*)in, (V*)out, t, tt, ph, s);
        }
        if (!tr.interpolate && zero_out) return launch_fill(zero_out, VT<V>::cplx ? (sizeof(typename VT<V>::R) == 8 ? DT_C128 : DT_C64) : (sizeof(typename VT<V>::R) == 8 ? DT_F64 : DT_F32), t.ngout * nin, st);
        return launch_error();
    }
    if (!tr.interpolate) {
        launch_kernel((k_restrict<V, K>), grid, dim3(256), 0, st, (const V*)in, (V*)out,
                           (V*)zero_out, t, ph);
    } else if (mode == TR_SUBTRACT) {
        launch_kernel((k_interpolate<V, K, TR_SUBTRACT>), grid, dim3(256), 0, st,
                           (const V*)in, (V*)out, t, ph);
    } else {
        launch_kernel((k_interpolate<V, K, TR_STORE>), grid, dim3(256), 0, st, (const V*)in,
                           (V*)out, t, ph);
    }
    return launch_error();
}

template <class V>
hipError_t tr_dispatch(const Transfer& tr, int mode, const void* in, void* out, void* zero_out,
                       const Phases& ph, int nin, hipStream_t st, double* sums = nullptr,
                       int* nsums = nullptr)
{
    switch (tr.K) {
    case 2: return tr_launch<V, 2>(tr, mode, in, out, zero_out, ph, nin, st, sums, nsums);
    case 4: return tr_launch<V, 4>(tr, mode, in, out, zero_out, ph, nin, st, sums, nsums);
    case 6: return tr_launch<V, 6>(tr, mode, in, out, zero_out, ph, nin, st, sums, nsums);
    case 8: return tr_launch<V, 8>(tr, mode, in, out, zero_out, ph, nin, st, sums, nsums);
    }
    return hipErrorInvalidValue;
}

}  // namespace gpaw
