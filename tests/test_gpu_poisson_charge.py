"""A density that is not neutral costs gpaw_poisson_solve its integral, whatever
was solved before: no V-cycle runs for it, and phi stays as it was."""
import ctypes
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N, pbc', [((64, 64, 64), True), ((96, 96, 96), False)])
def test_charged_density_runs_no_cycles(N, pbc):
    """The best of ten calls after a neutral solve each, against half the time of
    the best of those solves (8 to 11 V-cycles): the integral and the copy of phi
    take less than one V-cycle, so a single cycle of margin would do."""
    torch = pytest.importorskip('torch')
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    from gpaw_amd import _arrays, _lib
    from gpaw_amd.grid_descriptor import GridDescriptor
    from gpaw_amd.poisson import PoissonSolver
    print('case charged after neutral', N, pbc, flush=True)
    gd = GridDescriptor(N, np.array(N) * 0.35, pbc)
    solver = PoissonSolver()
    solver.set_grid_descriptor(gd)
    solver.initialize()
    rho = np.random.default_rng(2).standard_normal(tuple(int(x) for x in gd.n_c))
    rho = torch.from_numpy(rho - rho.mean()).cuda()
    charged = rho + 1.0
    phi = torch.zeros_like(rho)
    kept = torch.full_like(rho, 0.25)

    def call(target, density):
        q, e = ctypes.c_double(0.0), ctypes.c_double(0.0)
        neutral, niter = ctypes.c_int(-1), ctypes.c_int(-1)
        torch.cuda.synchronize()
        t = time.perf_counter()
        _lib.check(_lib.lib().gpaw_poisson_solve(
            solver._plan, target.data_ptr(), density.data_ptr(), 2e-10, 100, 1e-6,
            ctypes.byref(q), ctypes.byref(neutral), ctypes.byref(niter), ctypes.byref(e),
            _arrays.stream()))
        torch.cuda.synchronize()
        return time.perf_counter() - t, neutral.value, niter.value, q.value

    solves, refused = [], []
    for _ in range(12):
        phi.zero_()
        t, neutral, niter, _ = call(phi, rho)
        assert neutral == 1 and niter > 4
        solves.append(t)
        t, neutral, niter, q = call(kept, charged)
        assert neutral == 0 and niter == -1
        assert abs(q - charged.numel() * gd.dv) <= 1e-9 * abs(q)
        refused.append(t)
    assert torch.equal(kept, torch.full_like(rho, 0.25))
    assert min(refused[2:]) < 0.5 * min(solves[2:])
