"""Every instance of the two-planes-per-step star kernel, forced and seen to be
the one that runs: each storage type, pass, range and tile width, on grids whose
last tile and last run are partial ones, against the column kernel on every band
and against the oracle on one (64-bit types; the 32-bit ones round as the column
kernel does, which the other tests hold against 64 bits)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

# stored points along axis 2 -> the tile width that covers them with fewest lanes
WIDTH = {29: 32, 45: 48, 61: 64, 93: 96}
TYPES = ['float64', 'complex128', 'float32', 'complex64']


def instances():
    for dtype in TYPES:
        for potential in (False, True):
            if potential and dtype in ('float32', 'complex64'):
                continue        # potentials are applied to 64-bit bands
            for R in (1, 2, 3):
                for n2, tz in WIDTH.items():
                    if tz == 96 and dtype == 'complex128':
                        continue    # 16-byte planes of that width leave one block a CU
                    yield dtype, potential, R, n2


def setup(dtype, R, N, pbc, nb):
    import torch

    from gpaw_amd.fd_operators import Laplace
    from gpaw_amd.grid_descriptor import GridDescriptor
    cell = tuple(0.3 * n for n in N)
    gd, og = GridDescriptor(N, cell, pbc), O.Grid(N, cell, pbc)
    t = complex if dtype.startswith('complex') else float
    psi = torch.randn((nb,) + tuple(int(x) for x in gd.n_c), dtype=getattr(torch, dtype),
                      device='cuda', generator=torch.Generator(device='cuda').manual_seed(5))
    ph = gd.phase_cd(np.where(gd.pbc_c, (0.15, -0.3, 0.4), 0.0)) if t is complex else None
    return Laplace(gd, -0.5, R, t), O.laplace(og, -0.5, R, dtype=t), psi, ph


def forced(kind, run, like, fill):
    import torch

    from gpaw_amd import ops
    out = torch.full_like(like, fill)
    prev = ops.stencil_kernel(kind)
    try:
        run(out)
    finally:
        ops.stencil_kernel(prev)
    return out


@pytest.mark.parametrize('pbc', [True, False, (True, False, True)])
@pytest.mark.parametrize('dtype, potential, R, n2', list(instances()))
def test_instance(dtype, potential, R, n2, pbc):
    import torch

    from gpaw_amd import ops
    print('case pair', dtype, potential, R, n2, pbc, flush=True)
    periodic = (pbc,) * 3 if isinstance(pbc, bool) else pbc
    N = [n + (not p) for n, p in zip((21, 13, n2), periodic)]   # 21 x 13 x n2 stored
    lap, ref, psi, ph = setup(dtype, R, N, pbc, 3)
    v = torch.randn(tuple(psi.shape[1:]), dtype=torch.float64, device='cuda')
    seen = []

    def run(out):
        seen.append(lap.operator.kernel(psi, potential))
        if potential:
            lap.operator.apply_potential(psi, out, v, ph)
        else:
            lap.apply(psi, out, ph)

    got = forced('pair', run, psi, 3.0)
    want = forced('queue', run, psi, 5.0)
    family, columns, planes = seen[0]
    assert (family, columns) == ('pair', WIDTH[n2]) and 0 < planes < 21 and 21 % planes
    assert seen[1] == ('queue', 0, 0)
    assert torch.equal(got, want)
    if dtype in ('float64', 'complex128'):
        a = psi[1].cpu().numpy()
        exact = np.zeros_like(a)
        ref.apply(a, exact, ph)
        if potential:
            exact = exact + a * v.cpu().numpy()
        assert np.array_equal(got[1].cpu().numpy(), exact)
    assert ops.stencil_kernel('default') == 'default'


def test_leaves_what_it_cannot_run():
    """Range 4, planes that a tile's halo would wrap around twice, and a stencil
    that is no star take their default."""
    import torch

    from gpaw_amd import ops
    from gpaw_amd.fd_operators import Gradient
    from gpaw_amd.grid_descriptor import GridDescriptor
    for R, N in ((4, (20, 20, 40)), (3, (12, 5, 40)), (3, (12, 12, 8))):
        lap, _, psi, ph = setup('complex128', R, N, True, 2)
        default = lap.operator.kernel(psi)
        seen = []

        def run(out):
            seen.append(lap.operator.kernel(psi))
            lap.apply(psi, out, ph)

        got = forced('pair', run, psi, 3.0)
        assert seen == [default] and default[0] != 'pair'
        assert torch.equal(got, forced('queue', run, psi, 5.0))
    gd = GridDescriptor((12, 12, 12), (4, 4, 4), True)
    grad = Gradient(gd, 1, n=2)
    a = torch.randn((12, 12, 12), dtype=torch.float64, device='cuda')
    prev = ops.stencil_kernel('pair')
    try:
        assert grad.operator.kernel(a)[0] == 'generic'
    finally:
        ops.stencil_kernel(prev)
