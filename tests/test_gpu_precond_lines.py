"""The preconditioner on either side of the lines between its fused level-0 pass
and the separate steps: the first and last band against the oracle, each band
against a set of another size."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

CASES = [
    # N, pbc, dtype, bands, range; real rows of up to 32 points from 2^18 points
    ((24, 28, 28), False, float, 7, 3),
    ((24, 28, 28), False, float, 16, 3),
    ((28, 24, 32), True, float, 2, 2),
    ((28, 24, 32), True, float, 13, 2),
    ((24, 28, 36), True, float, 3, 3),
    # complex between walls from 2^21 points
    ((48, 20, 60), False, complex, 12, 3),
    ((48, 44, 40), False, complex, 27, 3),
    ((48, 20, 60), (True, True, False), complex, 12, 3),
]


@pytest.mark.parametrize('N, pbc, dtype, nb, nn0', CASES)
def test_either_side(N, pbc, dtype, nb, nn0):
    torch = pytest.importorskip('torch')
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    from gpaw_amd.fd_operators import Laplace
    from gpaw_amd.grid_descriptor import GridDescriptor
    from gpaw_amd.preconditioner import Preconditioner
    print('case precond line', N, pbc, dtype.__name__, nb, nn0, flush=True)
    cell = np.array(N) * 0.2
    og, gd = O.Grid(N, cell, pbc), GridDescriptor(N, cell, pbc)
    ref = O.Preconditioner(og, O.laplace(og, -0.5, nn0, dtype), dtype)
    pc = Preconditioner(gd, Laplace(gd, -0.5, nn0, dtype), dtype, block=nb)
    pc.allocate()
    rng = np.random.default_rng(sum(N) + nb)
    shape = (nb,) + tuple(og.n_c)
    res = rng.standard_normal(shape)

    class Kpt:
        phase_cd = None
    if dtype == complex:
        res = res + 1j * rng.standard_normal(shape)
        Kpt.phase_cd = og.phase_cd(np.where(gd.pbc_c, (0.15, -0.3, 0.4), 0.0))
    kpt = Kpt if dtype == complex else None
    x = torch.from_numpy(res).cuda()
    got = pc(x, kpt).clone()
    ends = [0, nb - 1]
    assert np.array_equal(got[ends].cpu().numpy(), ref(res[ends], Kpt.phase_cd))
    for n in range(nb):
        assert torch.equal(pc(x[n:n + 1], kpt)[0], got[n])
