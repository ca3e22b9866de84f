"""The kernel that a large star apply takes: grids on either side of each line of
the rule, among them those where another choice was slower than the tile kernel
(times in us), against the column kernel bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # dtype, bands, stored points, range, potential, kernel
    ('float64', 95, (94, 48, 32), 3, False, 'tile'),       # 52; pair 57
    ('float64', 256, (31, 62, 23), 3, True, 'tile'),       # 58; pair 65
    ('float64', 57, (105, 42, 45), 3, True, 'pair'),       # 74; tile 84
    ('float64', 188, (50, 21, 63), 3, True, 'box'),        # tile 52, box 54; pair 70
    ('float64', 66, (67, 111, 86), 3, True, 'pair'),       # tile 255; box 311, pair 242
    ('float64', 66, (71, 111, 96), 3, True, 'box'),        # filled boxes
    ('float64', 46, (66, 72, 91), 3, True, 'box'),         # in the last-level cache
    ('float64', 44, (101, 64, 87), 3, True, 'box'),        # tile 142; pair 155
    ('float64', 95, (94, 48, 40), 3, False, 'pair'),
    ('float64', 95, (94, 48, 32), 2, False, 'pair'),
    ('complex128', 256, (26, 26, 37), 3, False, 'tile'),   # 95; pair 108
    ('complex128', 256, (26, 26, 48), 3, False, 'tile'),
    ('complex128', 10, (23, 53, 39), 3, False, 'pair'),    # 15.7; tile 16.5
    ('complex128', 6, (23, 43, 70), 3, True, 'pair'),
    ('complex128', 24, (23, 53, 39), 3, False, 'tile'),
    ('complex128', 128, (26, 36, 49), 3, False, 'pair'),
    ('complex128', 128, (26, 36, 49), 3, True, 'pair'),
    ('complex128', 128, (26, 36, 32), 3, False, 'pair'),
    ('complex128', 128, (26, 36, 32), 3, True, 'tile'),
    ('complex128', 22, (63, 29, 73), 1, False, 'tile'),    # 26; pair 31
    ('complex128', 122, (33, 28, 99), 3, False, 'pair'),   # tile 1.13 of 1024 threads, pair 0.86
    ('complex128', 40, (33, 28, 99), 3, False, 'tile'),    # in the last-level cache
    ('complex128', 97, (65, 94, 65), 2, True, 'tile'),     # lanes filled to 0.66
    ('complex128', 64, (64, 64, 64), 3, False, 'tile'),
    ('complex64', 60, (56, 60, 51), 3, False, 'box'),
    ('float32', 128, (64, 64, 64), 3, False, 'pair'),
]


@pytest.mark.parametrize('dtype, nb, n, R, potential, kernel', CASES)
def test_kernel_of_a_large_apply(dtype, nb, n, R, potential, kernel):
    torch = pytest.importorskip('torch')
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    from gpaw_amd import ops
    from gpaw_amd.fd_operators import Laplace
    from gpaw_amd.grid_descriptor import GridDescriptor
    print('case rule', dtype, nb, n, R, potential, flush=True)
    gd = GridDescriptor(n, np.array(n) * 0.3, True)
    t = complex if dtype.startswith('complex') else float
    lap = Laplace(gd, -0.5, R, t)
    psi = torch.randn((nb,) + n, dtype=getattr(torch, dtype), device='cuda',
                      generator=torch.Generator(device='cuda').manual_seed(7))
    v = torch.randn(n, dtype=torch.float64, device='cuda')
    ph = gd.phase_cd((0.15, -0.3, 0.4)) if t is complex else None
    assert lap.operator.kernel(psi, potential)[0] == kernel

    def run(fill):
        out = torch.full_like(psi, fill)
        if potential:
            lap.operator.apply_potential(psi, out, v, ph)
        else:
            lap.apply(psi, out, ph)
        return out

    got = run(3.0)
    prev = ops.stencil_kernel('queue')
    try:
        want = run(5.0)
    finally:
        ops.stencil_kernel(prev)
    assert torch.equal(got, want)
