"""The plane-sweeping transfer kernels split along axis 0 (few bands), and
the helpers that the density and potential transfers run beside them."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

CELL = 0.35


def _grids(N, pbc):
    from gpaw_amd.grid_descriptor import GridDescriptor
    cell = tuple(CELL * n for n in N)
    gd, og = GridDescriptor(N, cell, pbc), O.Grid(N, cell, pbc)
    return gd, gd.refine(), og, og.refine()


@pytest.mark.parametrize('interpolate', [False, True])
@pytest.mark.parametrize('nn', [2, 3, 4])
@pytest.mark.parametrize('N, pbc', [((18, 10, 18), False), ((17, 10, 34), True),
                                    ((26, 18, 66), (True, False, True))])
@pytest.mark.parametrize('dtype', [float, complex])
def test_chunks_against_oracle(interpolate, nn, N, pbc, dtype):
    """One band goes through many chunks of the axis, 600 bands through one:
    both equal the oracle (the last chunk is a partial one on these sizes)."""
    import torch

    from gpaw_amd.transformers import Transformer
    print('case transfer chunks', interpolate, nn, N, pbc, dtype, flush=True)
    gd, fd, og, of = _grids(N, pbc)
    gi, go, oi, oo = (gd, fd, og, of) if interpolate else (fd, gd, of, og)
    rng = np.random.default_rng(17)
    a = rng.standard_normal(tuple(oi.n_c)).astype(dtype)
    ph = None
    if dtype is complex:
        a = a + 1j * rng.standard_normal(a.shape)
        ph = oi.phase_cd((0.15, -0.3, 0.4))
    want = np.zeros(tuple(oo.n_c), dtype)
    O.Transformer(oi, oo, nn, dtype).apply(a, want, ph)
    tr = Transformer(gi, go, nn, dtype)
    x = torch.from_numpy(a).to('cuda')
    got = torch.full(tuple(go.n_c), 7.0, dtype=x.dtype, device='cuda')
    tr.apply(x, got, ph)
    assert np.array_equal(got.cpu().numpy(), want)
    many = torch.full((600,) + tuple(go.n_c), 7.0, dtype=x.dtype, device='cuda')
    tr.apply(x.expand(600, *x.shape).contiguous(), many, ph)
    assert bool((many == got).all())


@pytest.mark.parametrize('shape', [(3, 4, 5), (1, 7, 5, 9), (2, 63, 31, 33), (7, 20, 21, 22)])
def test_renormalize_equals_its_steps(shape):
    """The integral, the sum over functions and the scaling on the device
    give the bits of integrate(), numpy's sum and scale()."""
    import torch

    from gpaw_amd import ops
    gd, _, _, _ = _grids((4, 4, 4), False)
    y = torch.from_numpy(np.random.default_rng(3).uniform(0, 1, shape)).to('cuda')
    want = y.clone()
    ops.scale(want, 5.25 / np.sum(ops.integrate(gd, want)))
    ops.renormalize(gd, y, 5.25)
    assert torch.equal(y, want)


@pytest.mark.parametrize('nin, n', [(1, 1), (1, 257), (2, 1001), (5, 4096)])
def test_axpby_shared_equals_axpby(nin, n):
    import torch

    from gpaw_amd import ops
    rng = np.random.default_rng(4)
    y = torch.from_numpy(rng.standard_normal((nin, n))).to('cuda')
    x = torch.from_numpy(rng.standard_normal(n)).to('cuda')
    want = y.clone()
    for k in range(nin):
        ops.axpby(want[k], x, 0.7, -1.3)
    ops.axpby_shared(y, x, 0.7, -1.3, nin)
    assert torch.equal(y, want)
    empty = y[:0]
    ops.axpby_shared(empty, x, 1.0, 1.0, 0)


@pytest.mark.parametrize('n,pbc,nn,nin', [
    ((16, 16, 16), False, 3, 1),         # 31^3: partial tiles
    ((16, 20, 24), (True, True, False), 2, 3),
    ((10, 16, 34), (False, True, True), 4, 7),
    ((30, 24, 16), False, 1, 2),         # K = 2: its kernel leaves no sums
    ((8, 150, 530), False, 2, 1),        # 38 x 34 tiles: more than a row of sums
    ((64, 12, 12), False, 3, 2),         # many chunks of few tiles
])
def test_interpolation_sums_its_outputs(n, pbc, nn, nin):
    """apply_renormalize against apply and renormalize.  The sums of positive
    values differ by the rounding of two orders of addition, at most about 300
    terms deep each: 600 * 1.1e-16 relative, bound 1e-13."""
    torch = pytest.importorskip('torch')
    if not torch.cuda.is_available():
        pytest.skip('no GPU')
    print('case interpolation sums', n, pbc, nn, nin, flush=True)
    from gpaw_amd import ops
    from gpaw_amd.grid_descriptor import GridDescriptor
    from gpaw_amd.transformers import Transformer
    gd = GridDescriptor(n, np.array(n) * 0.4, pbc)
    fine = gd.refine()
    tr = Transformer(gd, fine, nn)
    g = torch.Generator(device='cuda').manual_seed(3)
    a = torch.rand((nin,) + tuple(int(x) for x in gd.n_c), dtype=torch.float64, device='cuda',
                   generator=g) + 0.5
    want = torch.empty((nin,) + tuple(int(x) for x in fine.n_c), dtype=torch.float64,
                       device='cuda')
    got = torch.full_like(want, 7.0)
    tr.apply(a, want)
    ops.renormalize(fine, want, -3.5)
    tr.transformer.apply_renormalize(fine, a, got, -3.5)
    assert bool(((got - want).abs() <= 1e-13 * want.abs()).all())
    total = float(np.sum(fine.integrate(got)))
    assert abs(total + 3.5) <= 3.5e-13
    with pytest.raises(Exception):
        tr.transformer.apply_renormalize(fine, a[..., 1:].contiguous(), got, -3.5)
