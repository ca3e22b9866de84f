"""The two-planes-per-step star kernel (large band sets) against the column
kernel on every band and against the oracle on one, at the edges of its tiles
(32, 48, 64, 96 columns, 8 rows) and runs."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

# N_c, periodic, dtype, range; enough bands that the plane-sweeping kernels run
CASES = [
    ((32, 30, 96), False, 'float64', 3), ((17, 22, 64), True, 'float64', 3),
    ((20, 27, 48), (True, False, True), 'float64', 2), ((9, 33, 110), False, 'float64', 1),
    ((24, 24, 29), True, 'float64', 3), ((21, 18, 97), (False, True, False), 'float64', 3),
    ((28, 36, 44), True, 'complex128', 3), ((15, 40, 47), (True, True, False), 'complex128', 3),
    ((16, 17, 60), False, 'complex128', 2), ((11, 9, 95), True, 'complex128', 1),
    ((56, 60, 52), (True, True, False), 'complex64', 3), ((13, 20, 33), True, 'complex64', 2),
    ((22, 31, 90), True, 'float32', 3), ((19, 16, 63), False, 'float32', 1),
]


def _setup(N, pbc, dtype, R):
    import torch

    from gpaw_amd.fd_operators import Laplace
    from gpaw_amd.grid_descriptor import GridDescriptor
    cell = tuple(0.3 * n for n in N)
    gd, og = GridDescriptor(N, cell, pbc), O.Grid(N, cell, pbc)
    cplx = dtype.startswith('complex')
    n = tuple(int(x) for x in gd.n_c)
    # real data: more than the box kernel's limit of points
    nb = 40 if cplx else (1 << 23) // int(np.prod(n)) + 3
    psi = torch.randn((nb,) + n, dtype=getattr(torch, dtype), device='cuda',
                      generator=torch.Generator(device='cuda').manual_seed(7))
    ph = gd.phase_cd(np.where(gd.pbc_c, (0.15, -0.3, 0.4), 0.0)) if cplx else None
    t = complex if cplx else float
    return Laplace(gd, -0.5, R, t), O.laplace(og, -0.5, R, dtype=t), psi, ph, cplx


def _both(run, like):
    """run(out) with the default kernel and with the column kernel."""
    import torch

    from gpaw_amd import ops
    got, want = torch.full_like(like, 3.0), torch.full_like(like, 5.0)
    run(got)
    prev = ops.stencil_kernel('queue')
    try:
        run(want)
    finally:
        ops.stencil_kernel(prev)
    assert torch.equal(got, want)
    return got


@pytest.mark.parametrize('N, pbc, dtype, R', CASES)
def test_apply(N, pbc, dtype, R):
    print('case pair apply', N, pbc, dtype, R, flush=True)
    lap, ref, psi, ph, cplx = _setup(N, pbc, dtype, R)
    got = _both(lambda out: lap.apply(psi, out, ph), psi)
    if dtype in ('float64', 'complex128'):
        band = psi.shape[0] - 1
        a = psi[band].cpu().numpy()
        want = np.zeros_like(a)
        ref.apply(a, want, ph)
        assert np.array_equal(got[band].cpu().numpy(), want)


@pytest.mark.parametrize('N, pbc, dtype, R', [c for c in CASES if c[2] in ('float64', 'complex128')])
def test_apply_with_potential(N, pbc, dtype, R):
    import torch
    print('case pair potential', N, pbc, dtype, R, flush=True)
    lap, ref, psi, ph, cplx = _setup(N, pbc, dtype, R)
    v = torch.randn(tuple(psi.shape[1:]), dtype=torch.float64, device='cuda')
    got = _both(lambda out: lap.operator.apply_potential(psi, out, v, ph), psi)
    a = psi[0].cpu().numpy()
    want = np.zeros_like(a)
    ref.apply(a, want, ph)
    want = want + a * v.cpu().numpy()
    assert np.array_equal(got[0].cpu().numpy(), want)
