"""The fused CG direction step of the mixed-precision Poisson solve: both tile
shapes, every star range, both inner precisions, odd and even step counts per
chunk, and grids it does not take.

phi is only complete once the step each launch leaves pending is subtracted, and
p must be back in the first array after an odd number of steps: both show in
the true residual, taken here with the oracle's FP64 operator.  The solver
stops on its own FP64 evaluation of the same norm; the two differ by the
rounding of L phi, below |L|_inf |phi|_inf eps sqrt(n) / |rho| ~ 1e-13 here, so
the bound is rel_tol (1 + 1e-2) with rel_tol 1e-9.
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

I, P, S = (False,) * 3, (True,) * 3, (True, True, False)


@pytest.mark.parametrize('n,pbc,nn,inner', [
    ((16, 16, 16), I, 3, 'fp32'),        # 15^3: smallest tiles, partial everywhere
    ((16, 24, 40), P, 1, 'fp32'),
    ((24, 16, 72), S, 2, 'fp64'),        # rows of 71: a third tile of 7 columns
    ((72, 40, 32), P, 3, 'fp32'),
    ((48, 32, 16), I, 2, 'fp32'),        # rows shorter than a tile
    ((8, 8, 8), P, 3, 'fp32'),           # halo wraps more than once: separate launches
    ((32, 32, 32), I, 4, 'fp32'),        # range 4: separate launches
    ((112, 112, 80), P, 3, 'fp32'),      # 32 x 16 x 8 tiles (294)
    ((112, 96, 112), I, 1, 'fp64'),      # 32 x 16 x 8 tiles, partial (336)
])
def test_true_residual(n, pbc, nn, inner):
    torch = pytest.importorskip('torch')
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    print('case', n, pbc, nn, inner, flush=True)
    from gpaw_amd.grid_descriptor import GridDescriptor
    from gpaw_amd.poisson import MixedPoissonSolver, PoissonConvergenceError
    gd = GridDescriptor(n, np.array(n) * 0.35, pbc)
    og = O.Grid(gd.N_c, gd.cell_cv, gd.pbc_c)
    lap = O.gpaw_oracle.laplace(og, -0.25 / np.pi, nn)
    rng = np.random.default_rng(5)
    rho = rng.standard_normal(tuple(int(x) for x in gd.n_c))
    rho -= rho.mean()
    rho_g = torch.from_numpy(rho).cuda()
    tol = 1e-9

    def relres(phi_g):
        phi = phi_g.cpu().numpy()
        out = np.zeros_like(phi)
        lap.apply(phi, out)
        return np.linalg.norm(out - rho) / np.linalg.norm(rho)

    solver = MixedPoissonSolver(nn=nn, rel_tol=tol, inner_precision=inner)
    solver.set_grid_descriptor(gd)
    solver.initialize()
    steps = []
    for again in range(2):       # chunks by observed rate, then one of the last count
        phi = torch.zeros_like(rho_g)
        steps.append(solver.solve(phi, rho_g))
        assert relres(phi) <= 1.01 * tol
    for cut in (1, 2, 3):        # a last chunk of one, two or three steps
        short = MixedPoissonSolver(nn=nn, rel_tol=tol, inner_precision=inner, maxiter=cut)
        short.set_grid_descriptor(gd)
        short.initialize()
        phi = torch.zeros_like(rho_g)
        try:
            short.solve(phi, rho_g)
        except PoissonConvergenceError:
            pass
        seen = relres(phi)
        # the recursion's residual after few steps is the true one to rounding
        assert abs(seen - short.relres) <= 1e-8 * max(seen, tol)
