"""The fused coarse levels against a launch per pass (GPAW_AMD_COARSE_MAX=0, read
when the plan is made): the same V-cycle, bit for bit, for one to four fused
levels, one and two points per thread, odd and even extents, axes of one point.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

I, P, S = (False,) * 3, (True,) * 3, (True, True, False)


@pytest.mark.parametrize('n,pbc', [
    ((24, 24, 24), I),        # 11^3 (two points a thread), 5^3, 2^3
    ((16, 16, 16), P),        # 8^3, 4^3, 2^3
    ((16, 32, 64), P),        # below 16 x 32 x 64: 1024 x ..., two axes shrink first
    ((32, 32, 32), I),        # 7^3, 3^3, 1^3 below 15^3 (3375, too large)
    ((48, 48, 64), P),        # 6 x 6 x 8, 3 x 3 x 4
    ((32, 48, 16), S),        # 16 x 24 x 7 (2688, too large), 8 x 12 x 3, 4 x 6 x 1
    ((20, 20, 32), S),        # 10 x 10 x 15 (1500, two points a thread), 5 x 5 x 7
    ((20, 20, 20), P),        # 10^3 (1000), 5^3
    ((12, 20, 36), I),        # 5 x 9 x 17, 2 x 4 x 8
    ((18, 10, 26), P),        # one coarse level, 9 x 5 x 13
])
@pytest.mark.parametrize('cmax', ['2000', '600', '64'])
def test_same_cycle_as_single_launches(monkeypatch, n, pbc, cmax):
    torch = pytest.importorskip('torch')
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    print('case', n, pbc, cmax, flush=True)
    from gpaw_amd.grid_descriptor import GridDescriptor
    from gpaw_amd.poisson import PoissonSolver
    gd = GridDescriptor(n, np.array(n) * 0.35, pbc)
    rng = np.random.default_rng(9)
    rho = rng.standard_normal(tuple(int(x) for x in gd.n_c))
    rho -= rho.mean()
    rho_g = torch.from_numpy(rho).cuda()
    out = []
    for limit in (cmax, '0'):
        monkeypatch.setenv('GPAW_AMD_COARSE_MAX', limit)
        solver = PoissonSolver(nn=3)
        solver.set_grid_descriptor(gd)
        solver.initialize()
        phi = torch.zeros_like(rho_g)
        errors = solver.vcycles(phi, rho_g, 3)
        out.append((errors, phi.cpu().numpy()))
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1])
