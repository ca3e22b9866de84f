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
