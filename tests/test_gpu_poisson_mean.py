"""phi's mean on periodic grids is the one that the grid's own methods give."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = (16, 20, 24)


def descriptor(what):
    from gpaw_amd.grid_descriptor import GridDescriptor

    class Integral(GridDescriptor):   # one of two equal parts of a larger cell
        def integrate(self, a_xg, b_xg=None, global_integral=True):
            return 2.0 * GridDescriptor.integrate(self, a_xg, b_xg)

    class Size(GridDescriptor):
        def get_size_of_global_array(self):
            return GridDescriptor.get_size_of_global_array(self) * np.array((2, 1, 1))

    cls = {'integral': Integral, 'size': Size}.get(what, GridDescriptor)
    gd = cls(N, np.array(N) * 0.4, True)
    if what == 'object':
        plain = gd.integrate
        gd.integrate = lambda *a, **k: 2.0 * plain(*a, **k)
    return gd


@pytest.mark.parametrize('mixed', [False, True])
@pytest.mark.parametrize('whole', [False, True])
@pytest.mark.parametrize('what', ['plain', 'integral', 'size', 'object'])
def test_mean_of_the_grid(what, whole, mixed):
    torch = pytest.importorskip('torch')
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    from gpaw_amd import _lib, ops
    from gpaw_amd.poisson import MixedPoissonSolver, PoissonSolver
    print('case mean', what, whole, mixed, flush=True)
    gd = descriptor(what)
    solver = MixedPoissonSolver(reuse_history=False) if mixed else PoissonSolver()
    solver.set_grid_descriptor(gd)
    solver.initialize()
    gen = torch.Generator(device='cuda').manual_seed(3)
    rho = torch.randn(N, dtype=torch.float64, device='cuda', generator=gen)
    rho -= rho.mean()
    start = torch.randn(N, dtype=torch.float64, device='cuda', generator=gen) + 1.0
    phi = start.clone()
    if whole:
        solver.solve(phi, rho)
        # the density that solve goes on with
        q = ops.integrate(gd, rho)
        ops.sub_scalar(rho, rho, q / gd.dv / np.prod(N))
    else:
        solver.solve_neutral(phi, rho)

    # the solution before its mean is removed
    raw = start.clone()
    L, n, e = _lib.lib(), ctypes.c_int(0), ctypes.c_double(0.0)
    _lib.check(L.gpaw_poisson_remove_mean(solver._plan, 0))
    if mixed:
        _lib.check(L.gpaw_poisson_solve_mixed(
            solver._plan, raw.data_ptr(), rho.data_ptr(), solver.rel_tol, solver.maxiter, 1, 1,
            ctypes.byref(n), ctypes.byref(e), None))
    else:
        _lib.check(L.gpaw_poisson_solve_neutral(
            solver._plan, raw.data_ptr(), rho.data_ptr(), solver.eps, solver.maxiter,
            ctypes.byref(n), ctypes.byref(e), None))
    torch.cuda.synchronize()
    mean = gd.integrate(raw) / gd.dv / np.prod(gd.get_size_of_global_array())
    assert abs(mean) > 0.1
    ops.sub_scalar(raw, raw, mean)
    assert torch.equal(phi, raw)
