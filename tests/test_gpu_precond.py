"""The device preconditioner against the oracle's restatement of
gpaw/preconditioner.py:13-70 on the same inputs: bit-identical (every value
is rounded where the oracle rounds it), for real and Bloch-phase complex
bands, periodic and zero boundaries, orthogonal and non-orthogonal cells."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    return torch


class _Kpt:
    def __init__(self, phase_cd):
        self.phase_cd = phase_cd


CASES = [
    # N, cell, pbc, dtype, k, nbands, nn0
    ((32, 32, 32), None, True, float, None, 3, 3),
    ((32, 24, 16), None, False, float, None, 2, 3),
    ((32, 32, 24), None, True, complex, (0.1, 0.25, -0.3), 5, 3),
    ((24, 16, 16), None, True, complex, (0.5, 0.0, 0.2), 1, 1),
    ((16, 16, 16), ((4.0, 0, 0), (1.0, 4.0, 0), (0, 0, 4.0)), True, complex,
     (0.2, -0.1, 0.3), 2, 2),
]


@pytest.mark.parametrize('N,cell,pbc,dtype,k,nb,nn0', CASES)
def test_preconditioner_matches_oracle(N, cell, pbc, dtype, k, nb, nn0):
    print('case precond', N, pbc, dtype.__name__, k, nb, nn0, flush=True)
    torch = _torch()
    from gpaw_amd.grid_descriptor import GridDescriptor
    from gpaw_amd.fd_operators import Laplace
    from gpaw_amd.preconditioner import Preconditioner
    if cell is None:
        cell = np.array(N) * 0.2
    og = O.Grid(N, cell, pbc)
    gd = GridDescriptor(N, cell, pbc)
    ref = O.Preconditioner(og, O.laplace(og, -0.5, nn0, dtype), dtype)
    pc = Preconditioner(gd, Laplace(gd, -0.5, nn0, dtype), dtype, block=nb)
    pc.allocate()
    assert pc.step == ref.step
    rng = np.random.default_rng(sum(N) + nb)
    shape = (nb,) + tuple(og.n_c)
    res = rng.standard_normal(shape)
    if dtype == complex:
        res = res + 1j * rng.standard_normal(shape)
    ph = og.phase_cd(k) if k is not None else None
    expect = ref(res, ph)
    got = pc(torch.from_numpy(res).cuda(), _Kpt(ph) if ph is not None else None)
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy(), expect)


def test_preconditioner_numpy_and_single_band():
    _torch()
    from gpaw_amd.grid_descriptor import GridDescriptor
    from gpaw_amd.fd_operators import Laplace
    from gpaw_amd.preconditioner import Preconditioner
    N = (16, 16, 24)
    og = O.Grid(N, np.array(N) * 0.25)
    gd = GridDescriptor(N, np.array(N) * 0.25)
    ref = O.Preconditioner(og, O.laplace(og, -0.5, 3), float)
    pc = Preconditioner(gd, Laplace(gd, -0.5, 3), float)
    res = np.random.default_rng(7).standard_normal((1,) + N)
    expect = ref(res)
    assert np.array_equal(pc(res, None), expect)            # numpy in/out
    assert np.array_equal(pc(res[0].copy(), None), expect[0])   # 3-D input
    assert pc(np.zeros((0,) + N), None).shape == (0,) + N


def test_preconditioner_reuses_buffers_across_band_counts():
    torch = _torch()
    from gpaw_amd.grid_descriptor import GridDescriptor
    from gpaw_amd.fd_operators import Laplace
    from gpaw_amd.preconditioner import Preconditioner
    N = (16, 16, 16)
    og = O.Grid(N, np.array(N) * 0.3)
    gd = GridDescriptor(N, np.array(N) * 0.3)
    ref = O.Preconditioner(og, O.laplace(og, -0.5, 3, complex), complex)
    pc = Preconditioner(gd, Laplace(gd, -0.5, 3, complex), complex, block=2)
    rng = np.random.default_rng(11)
    ph = og.phase_cd((0.25, 0.25, 0.0))
    for nb in (4, 1, 3):
        res = rng.standard_normal((nb,) + N) + 1j * rng.standard_normal((nb,) + N)
        got = pc(torch.from_numpy(res).cuda(), _Kpt(ph)).cpu().numpy()
        assert np.array_equal(got, ref(res, ph)), nb


FUSED = [
    # N, pbc, dtype, bands, nn0: tiles of 8 and 16 rows, partial tiles, runs
    # that start on either parity, halos across every kind of boundary
    ((36, 28, 44), True, complex, 8, 3),
    ((28, 36, 52), (True, False, True), complex, 8, 3),
    ((44, 28, 40), (False, True, False), complex, 7, 2),
    ((40, 36, 36), False, complex, 8, 1),
    ((32, 32, 36), True, complex, 60, 3),
    ((36, 36, 68), False, float, 30, 3),
    ((36, 28, 44), True, float, 3, 3),
    ((28, 28, 36), (False, True, True), float, 2, 2),
    ((20, 24, 20), False, float, 1, 1),
    # rows of up to 16 points on level 2: 16 x 16 tiles
    ((48, 56, 64), True, complex, 14, 3),
    ((60, 44, 36), (True, False, True), complex, 40, 2),
    ((64, 40, 60), False, float, 3, 3),
]


@pytest.mark.parametrize('N,pbc,dtype,nb,nn0', FUSED)
def test_fused_passes(N, pbc, dtype, nb, nn0):
    """The passes over scaled and interpolated fields: the first and last band
    against the oracle, and every band against the same band alone (which for
    complex data runs the passes step by step)."""
    print('case precond fused', N, pbc, dtype.__name__, nb, nn0, flush=True)
    torch = _torch()
    from gpaw_amd.grid_descriptor import GridDescriptor
    from gpaw_amd.fd_operators import Laplace
    from gpaw_amd.preconditioner import Preconditioner
    cell = np.array(N) * 0.2
    og, gd = O.Grid(N, cell, pbc), GridDescriptor(N, cell, pbc)
    ref = O.Preconditioner(og, O.laplace(og, -0.5, nn0, dtype), dtype)
    pc = Preconditioner(gd, Laplace(gd, -0.5, nn0, dtype), dtype, block=nb)
    rng = np.random.default_rng(sum(N) + nb)
    shape = (nb,) + tuple(og.n_c)
    res = rng.standard_normal(shape)
    ph = kpt = None
    if dtype == complex:
        res = res + 1j * rng.standard_normal(shape)
        ph = og.phase_cd(np.where(gd.pbc_c, (0.15, -0.3, 0.4), 0.0))
        kpt = _Kpt(ph)
    x = torch.from_numpy(res).cuda()
    got = pc(x, kpt).clone()
    ends = sorted({0, nb - 1})
    assert np.array_equal(got[ends].cpu().numpy(), ref(res[ends], ph))
    for n in range(nb):
        assert torch.equal(pc(x[n:n + 1], kpt)[0], got[n])
