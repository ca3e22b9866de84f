// Fused coarse-level V-cycle (gfx950): the smallest levels of the multigrid
// hierarchy are smoothed, restricted and corrected by ONE workgroup in one
// launch, with a workgroup barrier between passes instead of a kernel
// boundary.  On these grids (11^3 and below for a 95^3 problem) a separate
// launch per pass costs more than the pass itself.
//
// The passes and their arithmetic are those of iterate2
// (gpaw/poisson.py:245-270) on 7-point operators (Laplace nn=1) with K=2
// transformers, exactly as the standalone kernels evaluate them:
//   Jacobi    x = sum_{c>=1} coef_c phi[g+off_c] (order z+, z-, y+, y-, x+, x-),
//             phi' = (1-w) phi + w (rho - x) / coef_0   (c/bmgs/relax.c:47-71)
//   residual  r = sum_c coef_c phi[g+off_c] - rho       (c/bmgs/fd.c:41-44)
//   restrict / interpolate   transfer_common.h
// so the fused path is bit-identical to launching the passes one by one.
//
// Bound by latency: about 20 passes on one compute unit, each a round of LDS
// reads, a chain of some 15 dependent FP64 operations and a barrier.  So
// nothing else is left on that chain.  The plan comes as a kernel argument
// (read from memory behind a pointer, with neighbour tables behind a second
// one, the first pass waited for three round trips), each thread keeps its
// points' right-hand sides and neighbour indices in registers for all passes of
// a level, and only the phi pair of every level lives in LDS (the residual
// takes the array the last sweep read).  With 1024 threads a lane has 128
// registers: one point a thread and up to two levels of two points fit (123 at
// four levels, 103), two points on three or four levels spill 12 and 84 bytes a
// lane.  The block has no more waves than the first level needs.  11^3 + 5^3 (16
// sweeps): 17.6 us before, 12.7 now; 6 x 6 x 8 + 3 x 3 x 4: 13.0 and 7.8; 9^3 alone
// (8 sweeps): 6.6 and 5.0.
#include "kernels.h"
#include "coarse.h"
#include "transfer_common.h"

namespace gpaw {

namespace {

// index of (j0, j1, j2), each at most one period outside, in a level's array:
// wrapped on periodic axes; outside a zero boundary the array's element n, its
// zero slot, which holds 0.0 for the whole kernel
__device__ __forceinline__ int slot_of(int j0, int j1, int j2, const CoarseLevel& L, int n)
{
    const int j[3] = {j0, j1, j2};
    int w[3];
    bool out = false;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        w[a] = j[a];
        if (w[a] < 0 || w[a] >= L.n[a]) {
            if (!L.per[a]) out = true;
            w[a] = w[a] < 0 ? w[a] + L.n[a] : w[a] - L.n[a];
        }
    }
    return out ? n : (w[0] * L.n[1] + w[1]) * L.n[2] + w[2];
}

// A thread's K points of one level: flat index (-1: none), the six neighbours
// in summation order (z+, z-, y+, y-, x+, x-), right-hand side and phi.
template <int K>
struct Pts {
    int idx[K];
    int i[K][3];
    int nb[K][6];
    double rho[K], phi[K];
};

__device__ __forceinline__ int points(const CoarseLevel& L) { return L.n[0] * L.n[1] * L.n[2]; }

template <int K>
__device__ __forceinline__ void level_points(const CoarseLevel& L, Pts<K>& p)
{
    const int n = points(L);
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int idx = threadIdx.x + blockDim.x * k;
        p.idx[k] = idx < n ? idx : -1;
        const int i2 = idx % L.n[2], t = idx / L.n[2], i1 = t % L.n[1], i0 = t / L.n[1];
        p.i[k][0] = i0;
        p.i[k][1] = i1;
        p.i[k][2] = i2;
        p.rho[k] = p.phi[k] = 0.0;
#pragma unroll
        for (int m = 0; m < 6; m++) p.nb[k][m] = n;
        if (idx < n) {
            p.nb[k][0] = slot_of(i0, i1, i2 + 1, L, n);
            p.nb[k][1] = slot_of(i0, i1, i2 - 1, L, n);
            p.nb[k][2] = slot_of(i0, i1 + 1, i2, L, n);
            p.nb[k][3] = slot_of(i0, i1 - 1, i2, L, n);
            p.nb[k][4] = slot_of(i0 + 1, i1, i2, L, n);
            p.nb[k][5] = slot_of(i0 - 1, i1, i2, L, n);
        }
    }
}

// x + the six neighbour terms in summation order.  A zero neighbour adds
// 0.0 * c as the standalone kernels do.
__device__ __forceinline__ double nb_sum(const double* a, const int* nb, const double* c, double x)
{
    double v[6];
#pragma unroll
    for (int m = 0; m < 6; m++) v[m] = a[nb[m]];
#pragma unroll
    for (int m = 0; m < 6; m++) x = x + v[m] * c[m + 1];
    return x;
}

// a / d rounded to nearest, from r = 1 / d rounded to nearest: the product
// q = a r is within an ulp of a / d, its remainder a - q d is exact in one
// fma, and q + (a - q d) r rounded once is the correctly rounded quotient
// (Markstein's theorem, binary64 without overflow or underflow).  A zero
// remainder keeps q, so exact quotients and signed zeros come out as a / d
// does.  Three operations instead of the division sequence, on a pass that
// runs on one compute unit.
__device__ __forceinline__ double div_rn(double a, double d, double r)
{
    const double q = a * r;
    const double e = __builtin_fma(-q, d, a);
    return e == 0.0 ? q : __builtin_fma(e, r, q);
}

// `sweeps` Jacobi sweeps between the level's arrays, from src; src is the
// array that holds the result, dst the other one
template <int K>
__device__ __forceinline__ void jacobi_sweeps(const CoarseLevel& L, Pts<K>& p, int sweeps,
                                              double*& src, double*& dst)
{
    double c[7];
#pragma unroll
    for (int m = 0; m < 7; m++) c[m] = L.c[m];
    const double w = L.w, rc0 = 1.0 / c[0];
    for (int it = 0; it < sweeps; it++) {
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int idx = p.idx[k];
            if (idx < 0) continue;
            const double x = nb_sum(src, p.nb[k], c, 0.0);
            p.phi[k] = (1.0 - w) * p.phi[k] + div_rn(w * (p.rho[k] - x), c[0], rc0);
            dst[idx] = p.phi[k];
        }
        __syncthreads();
        double* t = src;
        src = dst;
        dst = t;
    }
}

// one restriction pass of K = 2: 0.5 * (centre + 0.5 * (plus + minus))
__device__ __forceinline__ double rst_pass(double c, double p, double m)
{
    return (c + (p + m) * 0.5) * 0.5;
}

// the restriction of `res`, an array of level L, at point i of the next one
__device__ __forceinline__ double restrict_at(const double* res, const CoarseLevel& L, const int* i)
{
    const int n = points(L);
    const int c0 = 1 + 2 * i[0] - L.rlo[0], c1 = 1 + 2 * i[1] - L.rlo[1],
              c2 = 1 + 2 * i[2] - L.rlo[2];
    double v[3][3][3];   // centre, plus, minus per axis
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
        for (int b = 0; b < 3; b++)
#pragma unroll
            for (int c = 0; c < 3; c++)
                v[a][b][c] = res[slot_of(c0 + (a == 2 ? -1 : a), c1 + (b == 2 ? -1 : b),
                                         c2 + (c == 2 ? -1 : c), L, n)];
    double y[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        double z[3];
#pragma unroll
        for (int b = 0; b < 3; b++) z[b] = rst_pass(v[a][b][0], v[a][b][1], v[a][b][2]);
        y[a] = rst_pass(z[0], z[1], z[2]);
    }
    return rst_pass(y[0], y[1], y[2]);
}

// the interpolation of `e`, an array of level N, at point i of the finer level L
__device__ __forceinline__ double interp_at(const double* e, const CoarseLevel& L,
                                            const CoarseLevel& N, const int* i)
{
    const int n = points(N);
    const int q0 = i[0] + L.iskip[0], q1 = i[1] + L.iskip[1], q2 = i[2] + L.iskip[2];
    const int l0 = (q0 >> 1) - L.ilo[0], l1 = (q1 >> 1) - L.ilo[1], l2 = (q2 >> 1) - L.ilo[2];
    double v[2][2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int c = 0; c < 2; c++) v[a][b][c] = e[slot_of(l0 + a, l1 + b, l2 + c, N, n)];
    return interp2_combine<double>([&](int a, int b, int c) { return v[a][b][c]; }, q0 & 1, q1 & 1,
                                   q2 & 1);
}

// level l down: pre-smooth, residual into the other array
template <int K>
__device__ __forceinline__ void descend(const CoarseLevel& L, Pts<K>& p, double*& cur,
                                        double*& alt)
{
    jacobi_sweeps(L, p, L.pre, cur, alt);
    double c[7];
#pragma unroll
    for (int m = 0; m < 7; m++) c[m] = L.c[m];
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int idx = p.idx[k];
        if (idx >= 0) alt[idx] = nb_sum(cur, p.nb[k], c, 0.0 + p.phi[k] * c[0]) - p.rho[k];
    }
    __syncthreads();
}

// level l up: correct from e on the coarser level N, post-smooth
template <int K>
__device__ __forceinline__ void ascend(const CoarseLevel& L, const CoarseLevel& N,
                                       Pts<K>& p, const double* e, double*& cur, double*& alt)
{
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int idx = p.idx[k];
        if (idx >= 0) {
            p.phi[k] = p.phi[k] - interp_at(e, L, N, p.i[k]);
            cur[idx] = p.phi[k];
        }
    }
    __syncthreads();
    jacobi_sweeps(L, p, L.post, cur, alt);
}

// PPT: points per thread of the first level; the others have one
template <class TB, int NL, int PPT>
__global__ __launch_bounds__(1024) void k_coarse_vcycle(const CoarsePlan P)
{
    extern __shared__ double smem[];
    // per level: the array the last pass wrote, and the other one
    double *cur[NL], *alt[NL];
    Pts<PPT> p0;
    Pts<1> p[NL];   // p[0] is not used
#pragma unroll
    for (int l = 0; l < NL; l++) {
        const int n = points(P.lev[l]);
        cur[l] = smem + P.lev[l].off;
        alt[l] = cur[l] + n + 1;
        if (threadIdx.x == 0) {   // the zero slots
            cur[l][n] = 0.0;
            alt[l][n] = 0.0;
        }
    }
    // the first level's right-hand side, on the way while indices are formed
    const int n0 = points(P.lev[0]);
    double rho0[PPT];
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        const int idx = threadIdx.x + blockDim.x * k;
        rho0[k] = (double)((const TB*)P.rho)[idx < n0 ? idx : 0];
    }
    // every level starts from phi = 0
    level_points(P.lev[0], p0);
#pragma unroll
    for (int k = 0; k < PPT; k++) {
        if (p0.idx[k] >= 0) cur[0][p0.idx[k]] = 0.0;
        p0.rho[k] = rho0[k];
    }
#pragma unroll
    for (int l = 1; l < NL; l++) {
        level_points(P.lev[l], p[l]);
        if (p[l].idx[0] >= 0) cur[l][p[l].idx[0]] = 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int l = 0; l < NL - 1; l++) {
        if (l == 0)
            descend(P.lev[0], p0, cur[0], alt[0]);
        else
            descend(P.lev[l], p[l], cur[l], alt[l]);
        if (p[l + 1].idx[0] >= 0) p[l + 1].rho[0] = restrict_at(alt[l], P.lev[l], p[l + 1].i[0]);
    }
    // bottom: post-smooth only
    if (NL == 1)
        jacobi_sweeps(P.lev[0], p0, P.lev[0].post, cur[0], alt[0]);
    else
        jacobi_sweeps(P.lev[NL - 1], p[NL - 1], P.lev[NL - 1].post, cur[NL - 1], alt[NL - 1]);
#pragma unroll
    for (int l = NL - 2; l >= 0; l--) {
        if (l == 0)
            ascend(P.lev[0], P.lev[1], p0, cur[1], cur[0], alt[0]);
        else
            ascend(P.lev[l], P.lev[l + 1], p[l], cur[l + 1], cur[l], alt[l]);
    }
#pragma unroll
    for (int k = 0; k < PPT; k++)   // each thread's own points
        if (p0.idx[k] >= 0) ((TB*)P.out)[p0.idx[k]] = (TB)p0.phi[k];
}

template <class TB, int NL>
hipError_t coarse_nl(const CoarsePlan& P, int nt, bool two, size_t lds, hipStream_t st)
{
    return two ? launch_kernel(k_coarse_vcycle<TB, NL, 2>, dim3(1), dim3(nt), lds, st, P)
               : launch_kernel(k_coarse_vcycle<TB, NL, 1>, dim3(1), dim3(nt), lds, st, P);
}

template <class TB>
hipError_t coarse_go(const CoarsePlan& P, hipStream_t st)
{
    int first = 0, rest = 1, doubles = 0;
    for (int l = 0; l < P.nlev; l++) {
        const int n = P.lev[l].n[0] * P.lev[l].n[1] * P.lev[l].n[2];
        if (n < 1 || n > (l ? 1024 : GPAW_COARSE_POINTS) || P.lev[l].off != doubles)
            return hipErrorInvalidValue;
        if (l == 0) first = n;
        if (l > 0 && n > rest) rest = n;
        doubles += 2 * (n + 1);
    }
    // no more waves at the barriers than there are points for; beyond 1024
    // points two for some threads (11^3: 13.0 us with 16 waves, 13.9 with 11)
    const bool two = first > 1024;
    const int nt = two ? 1024 : ((first > rest ? first : rest) + 63) / 64 * 64;
    const size_t lds = sizeof(double) * doubles;
    if (lds > 64 * 1024) return hipErrorInvalidValue;
    switch (P.nlev) {
    case 1: return coarse_nl<TB, 1>(P, nt, two, lds, st);
    case 2: return coarse_nl<TB, 2>(P, nt, two, lds, st);
    case 3: return coarse_nl<TB, 3>(P, nt, two, lds, st);
    case 4: return coarse_nl<TB, 4>(P, nt, two, lds, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_coarse_vcycle(const CoarsePlan& plan, int dtype, hipStream_t st)
{
    hipError_t e = dtype == DT_F32   ? coarse_go<float>(plan, st)
                   : dtype == DT_F64 ? coarse_go<double>(plan, st)
                                     : hipErrorInvalidValue;
    return e == hipSuccess ? launch_error() : e;
}

}  // namespace gpaw
