"""Stencils without a star form (non-orthogonal cells, Mehrstellen, gradients,
GUC): the LDS sweep and the one-axis kernel against the generic kernel, bit
for bit, at the edges of their tiles and runs."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H = 0.38
CELLS = {
    'hex': lambda n: [[n[0] * H, 0, 0], [-n[1] * H / 2, n[1] * H * math.sqrt(3) / 2, 0],
                      [0, 0, n[2] * H]],
    'fcc': lambda n: [[0, n[0] * H, n[0] * H], [n[1] * H, 0, n[1] * H], [n[2] * H, n[2] * H, 0]],
    'ortho': lambda n: np.diag([x * H for x in n]),
}


def _operators(kind, gd, dtype):
    from gpaw_amd.fd_operators import Gradient, GUCLaplace, Laplace, LaplaceA, LaplaceB
    if kind.startswith('lap'):
        return [Laplace(gd, -0.5, int(kind[3:]), dtype)]
    if kind.startswith('guc'):
        return [GUCLaplace(gd, -0.5, int(kind[3:]), dtype)]
    if kind == 'mehrstellen':
        return [LaplaceA(gd, 0.3, dtype), LaplaceB(gd, dtype)]
    return [Gradient(gd, v, n=int(kind[4:]), dtype=dtype) for v in range(3)]


CASES = [('hex', 'lap1', (8, 8, 8)), ('hex', 'lap3', (16, 16, 36)), ('hex', 'lap4', (13, 13, 25)),
         ('hex', 'guc3', (12, 12, 17)), ('hex', 'grad2', (9, 9, 33)),
         ('fcc', 'lap2', (10, 10, 10)), ('fcc', 'lap3', (21, 21, 21)), ('fcc', 'guc2', (17, 17, 17)),
         ('fcc', 'grad3', (20, 20, 20)),
         ('ortho', 'mehrstellen', (9, 10, 11)), ('ortho', 'mehrstellen', (31, 34, 65)),
         ('ortho', 'grad1', (5, 6, 7)), ('ortho', 'grad3', (15, 17, 19)),
         ('ortho', 'grad4', (33, 16, 129)), ('ortho', 'grad3', (4, 4, 300))]


@pytest.mark.parametrize('dtype', ['float64', 'complex128', 'float32', 'complex64'])
@pytest.mark.parametrize('pbc', [True, (False, True, False)])
@pytest.mark.parametrize('cell, kind, n', CASES)
def test_equal_to_generic_kernel(cell, kind, n, pbc, dtype):
    import torch

    from gpaw_amd import ops
    from gpaw_amd.grid_descriptor import GridDescriptor
    print('case generic stencil', cell, kind, n, pbc, dtype, flush=True)
    if cell == 'fcc':
        pbc = True
    gd = GridDescriptor(n, CELLS[cell](n), pbc)
    cplx = dtype.startswith('complex')
    ph = gd.phase_cd(np.where(gd.pbc_c, (0.15, -0.3, 0.4), 0.0)) if cplx else None
    g = torch.Generator(device='cuda').manual_seed(5)
    for op in _operators(kind, gd, complex if cplx else float):
        for nb in (1, 7):
            a = torch.randn((nb,) + tuple(gd.n_c), dtype=getattr(torch, dtype), device='cuda',
                            generator=g)
            got, want = torch.full_like(a, 3.0), torch.full_like(a, 5.0)
            op.apply(a, got, ph)
            prev = ops.stencil_kernel('generic')
            try:
                op.apply(a, want, ph)
            finally:
                ops.stencil_kernel(prev)
            assert torch.equal(got, want)
            assert bool(torch.isfinite(torch.view_as_real(got) if cplx else got).all())


@pytest.mark.parametrize('kind, cell, n', [('lap3', 'hex', (16, 16, 18)), ('lap2', 'fcc', (14, 14, 14)),
                                           ('mehrstellen', 'ortho', (17, 20, 35))])
def test_modes_equal_to_generic_kernel(kind, cell, n):
    """Residual, Jacobi sweeps and the potential term."""
    import torch

    from gpaw_amd import ops
    from gpaw_amd.grid_descriptor import GridDescriptor
    print('case generic stencil modes', kind, cell, n, flush=True)
    gd = GridDescriptor(n, CELLS[cell](n), True)
    op = _operators(kind, gd, float)[0].operator
    cop = _operators(kind, gd, complex)[0].operator
    g = torch.Generator(device='cuda').manual_seed(6)
    f, s, v = (torch.randn(tuple(gd.n_c), dtype=torch.float64, device='cuda', generator=g)
               for _ in range(3))
    psi = torch.randn((3,) + tuple(gd.n_c), dtype=torch.complex128, device='cuda', generator=g)
    ph = gd.phase_cd((0.2, 0.1, -0.4))

    def run():
        r, x, h = torch.full_like(f, 2.0), f.clone(), torch.full_like(psi, 2.0)
        op.residual(f, s, r)
        op.relax(2, x, s, 3, 0.7)
        cop.apply_potential(psi, h, v, ph)
        return r, x, h
    got = run()
    prev = ops.stencil_kernel('generic')
    try:
        want = run()
    finally:
        ops.stencil_kernel(prev)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_non_finite_values_stay_local():
    """Infinities and NaN reach exactly the points whose terms read them."""
    import torch

    from gpaw_amd import ops
    from gpaw_amd.grid_descriptor import GridDescriptor
    n = (16, 16, 30)
    gd = GridDescriptor(n, CELLS['hex'](n), True)
    op = _operators('lap2', gd, float)[0]
    a = torch.ones((2,) + n, dtype=torch.float64, device='cuda')
    a[0, 3, 4, 5] = float('inf')
    a[1, 0, 15, 29] = float('nan')
    got, want = torch.zeros_like(a), torch.zeros_like(a)
    op.apply(a, got)
    prev = ops.stencil_kernel('generic')
    try:
        op.apply(a, want)
    finally:
        ops.stencil_kernel(prev)
    assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(want))


@pytest.mark.parametrize('dtype', ['float64', 'complex128', 'float32', 'complex64'])
@pytest.mark.parametrize('n, pbc, nn', [
    ((5, 6, 15), True, 3), ((5, 6, 16), True, 3),        # shortest rows of the LDS kernel
    ((6, 5, 17), False, 4), ((40, 13, 16), False, 1),    # 64 rows a block, partial last block
    ((4, 5, 255), False, 2), ((4, 5, 342), True, 3),     # 4 and 2 rows a block
    ((5, 5, 513), True, 4),                              # one row a block
    ((4, 3, 1024), True, 3), ((4, 3, 1025), True, 3),    # a full block; too long for one
])
def test_gradient_along_rows(n, pbc, nn, dtype):
    """Axis 2: whole rows in LDS, where they fit, against the generic kernel."""
    import torch

    from gpaw_amd import ops
    from gpaw_amd.fd_operators import Gradient
    from gpaw_amd.grid_descriptor import GridDescriptor
    print('case gradient rows', n, pbc, nn, dtype, flush=True)
    m = n if pbc else tuple(x + 1 for x in n)
    gd = GridDescriptor(m, CELLS['ortho'](m), pbc)
    cplx = dtype.startswith('complex')
    ph = gd.phase_cd((0.15, -0.3, 0.4)) if cplx and pbc else None
    op = Gradient(gd, 2, n=nn, dtype=complex if cplx else float)
    g = torch.Generator(device='cuda').manual_seed(7)
    for nb in (1, 3):
        a = torch.randn((nb,) + tuple(gd.n_c), dtype=getattr(torch, dtype), device='cuda',
                        generator=g)
        got, want = torch.full_like(a, 3.0), torch.full_like(a, 5.0)
        op.apply(a, got, ph)
        prev = ops.stencil_kernel('generic')
        try:
            op.apply(a, want, ph)
        finally:
            ops.stencil_kernel(prev)
        assert torch.equal(got, want)
