"""Solves that launch before the host has read back what decides them: the
V-cycles of a repeated solve start before the charge is known, and the solution
is stored before the errors are.  Every result must be what a new solver, which
has no earlier solve to go by, gives bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = (16, 24, 32)


@pytest.fixture(scope='module')
def torch():
    t = pytest.importorskip('torch')
    if not t.cuda.is_available():
        pytest.skip('no GPU')
    return t


def make(pbc, mixed=False, **kw):
    from gpaw_amd.grid_descriptor import GridDescriptor
    from gpaw_amd.poisson import MixedPoissonSolver, PoissonSolver
    gd = GridDescriptor(N, np.array(N) * 0.35, pbc)
    s = MixedPoissonSolver(reuse_history=False, **kw) if mixed else PoissonSolver(**kw)
    s.set_grid_descriptor(gd)
    s.initialize()
    return s


def density(torch, solver, seed, charge):
    rng = np.random.default_rng(seed)
    gd = solver.gd
    rho = rng.standard_normal(tuple(int(x) for x in gd.n_c))
    rho += charge / gd.dv / rho.size - rho.mean()
    return torch.from_numpy(rho).cuda()


def run(torch, solver, rho):
    from gpaw_amd.poisson import PoissonConvergenceError
    phi = torch.full_like(rho, 0.25)
    try:
        niter = solver.solve(phi, rho)
    except PoissonConvergenceError:
        niter = -1
    return niter, phi.cpu().numpy()


@pytest.mark.parametrize('mixed', [False, True])
@pytest.mark.parametrize('pbc', [(True,) * 3, (False,) * 3])
@pytest.mark.parametrize('relax', ['J', 'GS'])
def test_charge_changes_between_solves(torch, pbc, mixed, relax):
    if mixed and relax == 'GS':
        pytest.skip('mixed precision sweeps are Jacobi')
    print('case', pbc, mixed, relax, flush=True)
    solver = make(pbc, mixed, relax=relax)
    for step, charge in enumerate([0, 0, 1.5, 0, -2.0, -2.0, 0, 0]):
        rho = density(torch, solver, step // 2, charge)
        kept = rho.clone()
        got = run(torch, solver, rho)
        want = run(torch, make(pbc, mixed, relax=relax), rho)
        assert got[0] == want[0]
        assert np.array_equal(got[1], want[1])
        assert torch.equal(rho, kept)


def test_charged_slab_is_refused_unchanged(torch):
    solver = make((True, True, False))
    run(torch, solver, density(torch, solver, 0, 0))
    phi = torch.full(tuple(int(x) for x in solver.gd.n_c), 0.25, dtype=torch.float64,
                     device='cuda')
    with pytest.raises(NotImplementedError):
        solver.solve(phi, density(torch, solver, 1, 1.0))
    assert torch.equal(phi, torch.full_like(phi, 0.25))


@pytest.mark.parametrize('mixed', [False, True])
def test_cut_short_after_a_converged_solve(torch, mixed):
    solver = make((True,) * 3, mixed)
    rho = density(torch, solver, 3, 0)
    n, _ = run(torch, solver, rho)
    assert n > 2
    for maxiter in (n, n - 1, 1):     # n: met, but counted as not converged
        solver.maxiter = maxiter
        other = make((True,) * 3, mixed)
        other.maxiter = maxiter
        got, want = run(torch, solver, rho), run(torch, other, rho)
        assert got[0] == want[0]
        assert np.array_equal(got[1], want[1])
    solver.maxiter = 1000
    harder = density(torch, solver, 4, 0) * 1e3     # more cycles than the last solve
    got, want = run(torch, solver, harder), run(torch, make((True,) * 3, mixed), harder)
    assert got[0] == want[0] and np.array_equal(got[1], want[1])
    easier = harder * 1e-6                          # fewer
    got, want = run(torch, solver, easier), run(torch, make((True,) * 3, mixed), easier)
    assert got[0] == want[0] and np.array_equal(got[1], want[1])


@pytest.mark.parametrize('mixed', [False, True])
def test_mean_is_removed_as_integrate_and_subtract(torch, mixed):
    from gpaw_amd import _lib, ops
    solver, plain = make((True,) * 3, mixed), make((True,) * 3, mixed)
    _lib.check(_lib.lib().gpaw_poisson_remove_mean(plain._plan, 0))
    rho = density(torch, solver, 6, 0)
    for _ in range(2):
        phi, raw = torch.full_like(rho, 0.25), torch.full_like(rho, 0.25)
        solver.solve(phi, rho)
        plain.solve(raw, rho)
        mean = solver.gd.integrate(raw) / solver.gd.dv
        mean /= np.prod(solver.gd.get_size_of_global_array())
        ops.sub_scalar(raw, raw, mean)
        assert torch.equal(phi, raw)


@pytest.mark.parametrize('mixed', [False, True])
def test_first_solve_beside_a_busy_null_stream(torch, mixed):
    """A solver's first solve sets its state up; on a stream that does not wait
    for the null stream nothing of that may be left queued there."""
    want = None
    side = torch.cuda.Stream()
    a = torch.ones((4096, 4096), dtype=torch.float64, device='cuda')
    for busy in (False, True):
        solver = make((True,) * 3, mixed)
        rho = density(torch, solver, 8, 0)
        torch.cuda.synchronize()
        if busy:
            for _ in range(20):
                b = a @ a           # tens of milliseconds on the null stream
        with torch.cuda.stream(side):
            got = run(torch, solver, rho)
        torch.cuda.synchronize()
        assert got[0] > 0
        if want is not None:
            assert got[0] == want[0] and np.array_equal(got[1], want[1])
        want = got
