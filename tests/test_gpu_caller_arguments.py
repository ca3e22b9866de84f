"""What the callers refuse, and that they go through the objects they are
given."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = (8, 10, 12)


@pytest.fixture(scope='module')
def torch():
    t = pytest.importorskip('torch')
    if not t.cuda.is_available():
        pytest.skip('no GPU')
    return t


def grids(pbc):
    from gpaw_amd.grid_descriptor import GridDescriptor
    gd = GridDescriptor(N, np.array(N) * 0.4, pbc)
    return gd, gd.refine()


def rand(torch, shape, seed=1):
    g = torch.Generator(device='cuda').manual_seed(seed)
    return torch.rand(tuple(int(x) for x in shape), dtype=torch.float64, device='cuda',
                      generator=g) + 0.5


# shapes of vHt_g for a fine grid n and two spins that are not n
WRONG = {'transposed': lambda n: n[::-1],
         'larger': lambda n: (n[0] + 1,) + n[1:],
         'spins': lambda n: (2,) + n,
         'one spin': lambda n: (1,) + n,
         'flat': lambda n: (int(np.prod(n)),),
         'smaller': lambda n: n[:2] + (n[2] - 1,)}


@pytest.mark.parametrize('spins', [(), (1,), (2,)])
@pytest.mark.parametrize('wrong', sorted(WRONG))
def test_restrict_potential_wants_the_fine_grid(torch, spins, wrong):
    from gpaw_amd.callers import restrict_potential
    from gpaw_amd.transformers import Transformer
    print('case restrict_potential', spins, wrong, flush=True)
    gd, fine = grids(False)
    n = tuple(int(x) for x in fine.n_c)
    vt = rand(torch, spins + n)
    kept = vt.clone()
    out = rand(torch, spins + tuple(gd.n_c))
    vH = rand(torch, WRONG[wrong](n), 2)
    with pytest.raises(ValueError):
        restrict_potential(Transformer(fine, gd, 3), vt, vH, out)
    assert torch.equal(vt, kept)


def test_restrict_potential_of_no_spins(torch):
    from gpaw_amd.callers import restrict_potential
    from gpaw_amd.transformers import Transformer
    gd, fine = grids(True)
    restrict_potential(Transformer(fine, gd, 3), rand(torch, (0,) + tuple(fine.n_c)),
                       rand(torch, fine.n_c), rand(torch, (0,) + tuple(gd.n_c)))


@pytest.mark.parametrize('x, nin', [((4, 3), 2), ((2, 3, 4), 2), ((3, 5), 2), ((12,), 2),
                                    ((3, 4), 1), ((3, 4), 3)])
def test_axpby_shared_wants_the_shape_of_a_function(torch, x, nin):
    from gpaw_amd import ops
    y = rand(torch, (2, 3, 4))
    kept = y.clone()
    with pytest.raises(ValueError):
        ops.axpby_shared(y, rand(torch, x), 1.0, 1.0, nin)
    assert torch.equal(y, kept)


@pytest.mark.parametrize('which', [0, 1, 2])
def test_potential_that_is_one_of_the_spins(torch, which):
    """vt_g += vHt_g spin by spin: where vHt_g is one spin's vt_g, the later
    spins get what the earlier addition made of it."""
    from gpaw_amd.callers import restrict_potential
    from gpaw_amd.transformers import Transformer
    print('case vHt_g = vt_sg[%d]' % which, flush=True)
    gd, fine = grids(False)
    vt = rand(torch, (3,) + tuple(fine.n_c))
    want = vt.clone()
    for s in range(3):
        want[s] += want[which]
    restrict_potential(Transformer(fine, gd, 3), vt, vt[which],
                       rand(torch, (3,) + tuple(gd.n_c)))
    assert torch.equal(vt, want)


def density(torch, gd, fine, nspins=2):
    return rand(torch, (nspins,) + tuple(gd.n_c)), rand(torch, (nspins,) + tuple(fine.n_c), 2)


@pytest.mark.parametrize('where', ['subclass', 'object', 'class', 'handle'])
def test_interpolate_density_goes_through_apply(torch, where, monkeypatch):
    """The interpolator's own apply runs wherever it was put in place of the
    package's: once, and what it leaves is what is scaled."""
    from gpaw_amd import ops
    from gpaw_amd.callers import interpolate_density
    from gpaw_amd.transformers import Transformer, _Transformer
    print('case interpolate_density, apply of the', where, flush=True)
    gd, fine = grids(False)
    n, out = density(torch, gd, fine)
    calls = []

    def hook(apply, at=1):            # at: where the output is among the arguments
        def hooked(*args):
            calls.append(1)
            apply(*args)
            args[at][..., :3] *= 2.0
        return hooked

    plain = Transformer(gd, fine, 3)
    if where == 'subclass':
        class Mine(_Transformer):
            def apply(self, input, output):
                hook(super().apply)(input, output)
        tr = Mine(gd, fine, 3)
    else:
        tr = Transformer(gd, fine, 3)
        if where == 'object':
            tr.apply = hook(tr.apply)
        elif where == 'class':
            monkeypatch.setattr(_Transformer, 'apply', hook(_Transformer.apply, 2))
        else:
            tr.transformer.apply = hook(tr.transformer.apply)
    interpolate_density(tr, fine, n, out, charge=-8.0)
    monkeypatch.undo()
    assert len(calls) == 1
    want = torch.empty_like(out)
    plain.apply(n, want)
    want[..., :3] *= 2.0
    ops.scale(want, 8.0 / np.sum(fine.integrate(want)))
    assert torch.equal(out, want)


def test_interpolate_density_goes_through_integrate(torch):
    from gpaw_amd import ops
    from gpaw_amd.callers import interpolate_density
    from gpaw_amd.grid_descriptor import GridDescriptor
    from gpaw_amd.transformers import Transformer

    class Half(GridDescriptor):       # one of two equal parts of a larger cell
        def integrate(self, a_xg, b_xg=None, global_integral=True):
            return 2.0 * GridDescriptor.integrate(self, a_xg, b_xg)

    gd, plain = grids(False)
    fine = Half(plain.N_c, plain.cell_cv, plain.pbc_c)
    n, out = density(torch, gd, fine)
    tr = Transformer(gd, fine, 3)
    interpolate_density(tr, fine, n, out, charge=-8.0)
    want = torch.empty_like(out)
    tr.apply(n, want)
    ops.scale(want, 8.0 / np.sum(fine.integrate(want)))
    assert torch.equal(out, want)


@pytest.mark.parametrize('pbc', [False, True])
def test_interpolate_density_of_no_spins(torch, pbc):
    """Nothing to scale to a charge is an error, as integrating it is; without
    a scaling there is nothing to do."""
    from gpaw_amd import _lib
    from gpaw_amd.callers import interpolate_density
    from gpaw_amd.transformers import Transformer
    gd, fine = grids(pbc)
    n, out = density(torch, gd, fine, 0)
    if pbc:
        interpolate_density(Transformer(gd, fine, 3), fine, n, out, charge=-8.0)
        return
    with pytest.raises(_lib.GpawAmdError):
        interpolate_density(Transformer(gd, fine, 3), fine, n, out, charge=-8.0)


@pytest.mark.parametrize('dtype', ['float32', 'complex64', 'complex128'])
def test_apply_renormalize_is_of_float64(torch, dtype):
    """The library is told float64: another type would be read past its end, or
    as something else."""
    from gpaw_amd.transformers import Transformer
    gd, fine = grids(False)
    n, out = density(torch, gd, fine)
    t = getattr(torch, dtype)
    with pytest.raises(TypeError):
        Transformer(gd, fine, 3).transformer.apply_renormalize(fine, n.to(t), out.to(t), 8.0)
