"""Restrictions of band sets whose blocks are split into other numbers of chunks
along axis 0: every band equals the one that goes alone, which equals the
oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

CELL = 0.35


@pytest.mark.parametrize('dtype', [float, complex])
@pytest.mark.parametrize('nn', [2, 3, 4])
@pytest.mark.parametrize('N, pbc', [((14, 14, 18), True), ((27, 10, 22), False)])
def test_band_counts(dtype, nn, N, pbc):
    import torch

    from gpaw_amd.grid_descriptor import GridDescriptor
    from gpaw_amd.transformers import Transformer
    print('case chunk counts', dtype.__name__, nn, N, pbc, flush=True)
    cell = tuple(CELL * n for n in N)
    gd, og = GridDescriptor(N, cell, pbc), O.Grid(N, cell, pbc)
    fd, of = gd.refine(), og.refine()
    rng = np.random.default_rng(19)
    a = rng.standard_normal(tuple(of.n_c)).astype(dtype)
    ph = None
    if dtype is complex:
        a = a + 1j * rng.standard_normal(a.shape)
        ph = of.phase_cd((0.15, -0.3, 0.4))
    want = np.zeros(tuple(og.n_c), dtype)
    O.Transformer(of, og, nn, dtype).apply(a, want, ph)
    tr = Transformer(fd, gd, nn, dtype)
    x = torch.from_numpy(a).to('cuda')
    got = torch.full(tuple(gd.n_c), 7.0, dtype=x.dtype, device='cuda')
    tr.apply(x, got, ph)
    assert np.array_equal(got.cpu().numpy(), want)
    # two blocks a band: 8 .. 520 blocks
    for nb in (4, 20, 43, 64, 86, 128, 150, 200, 232, 252, 255, 256, 260):
        many = torch.full((nb,) + tuple(gd.n_c), 7.0, dtype=x.dtype, device='cuda')
        tr.apply(x.expand(nb, *x.shape).contiguous(), many, ph)
        assert bool((many == got).all()), nb
