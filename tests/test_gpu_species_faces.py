"""The face-by-face forms of the species face passes: boxes too thin for tiles
(compute_mass_fluxdiv), noise beyond and within the caches, matrices beyond the
last-level cache.  The oracle's operations in the oracle's order: the same bits."""
import numpy as np
import pytest

from lowmachmixtures_amd import stokes as S
from oracle import oracle as O
from tests.helpers import bit_equal
from tests.test_gpu_species import _knobs, _mass_noise, _rho

pytestmark = pytest.mark.gpu


def _chain(n, ns, stages, **kw):
    rng = np.random.default_rng(11 * ns + n[0])
    shape = tuple(reversed(n))
    kn = _knobs(ns, rng, k_B=0.5, fraction_tolerance=1e-8, Dtherm=list(rng.uniform(-0.5, 0.5, 8)), **kw)
    sp, g = O.species(ns, **kn), O.geom(3, n, 0.5)
    rho, T = _rho(ns, shape, rng), rng.uniform(0.9, 1.1, shape)
    W, w = _mass_noise(5, stages, 3, ns, shape), [1.0, 0.5][:stages]
    want = O.compute_mass_fluxdiv(g, sp, rho, T, 0.02, W, w)
    with S.Context(3, n, 0.5, stag_mg_minwidth=min(n), mg_minwidth=min(n)) as ctx:
        S.set_species(ctx, ns, **kn)
        S.init_mass_stochastic(ctx, stages)
        S.fill_mass_stochastic(ctx, 5)
        f_rho, diff, stoch = ctx.field(S.CELL, ns, rho), ctx.field(S.CELL, ns), ctx.field(S.CELL, ns)
        ft = [ctx.field(S.FACE_X + d, ns) for d in range(3)]
        S.compute_mass_fluxdiv(ctx, f_rho, None, diff, stoch, ctx.field(S.CELL, 1, T), ft, 0.02, 0.0, w)
        for got, ref in zip((f_rho, diff, stoch), want[:3]):
            assert bit_equal(got.download(), ref)
        assert bit_equal([f.download() for f in ft], want[3])


# just past 1024 tiles, the last cell short of 12 in x, a partly filled last workgroup
@pytest.mark.parametrize("n", [(4, 8, 1026), (10, 10, 514)])
@pytest.mark.parametrize("ns,ideal", [(2, 1), (3, 0), (4, 0), (5, 1), (6, 0), (7, 1), (8, 0)])
def test_thin_boxes(n, ns, ideal):
    _chain(n, ns, 1, is_ideal_mixture=ideal)


def test_thin_box_noise_past_the_caches():
    _chain((8, 8, 9216), 2, 2)  # 57 MB of noise


def test_stochastic_flux_noise_past_the_caches():
    n, ns, n_rngs = (64, 96, 96), 2, 2  # 57 MB
    rng = np.random.default_rng(53)
    shape = tuple(reversed(n))
    kn = _knobs(ns, rng, k_B=0.3)
    sp, g = O.species(ns, **kn), O.geom(3, n, 0.5)
    rho = _rho(ns, shape, rng, tiny=False)
    rt, x, mt = O.convert_cons_to_prim(g, sp, rho)
    Db, Dt, H = O.compute_mixture_properties(g, sp, shape)
    G = O.compute_Gama(g, sp, x, H)
    chi, _ = O.compute_chi(g, sp, rho, rt, x, Db, Dt, np.ones(shape))
    W = _mass_noise(77, n_rngs, 3, ns, shape)
    want, want_ft = O.stochastic_mass_fluxdiv(g, sp, rho, rt, x, mt, chi, G, [np.zeros((ns,) + shape)] * 3, 0.01, W,
                                              [0.75, -0.5])
    with S.Context(3, n, 0.5, stag_mg_minwidth=64, mg_minwidth=64) as ctx:
        S.set_species(ctx, ns, **kn)
        S.init_mass_stochastic(ctx, n_rngs)
        S.fill_mass_stochastic(ctx, 77)
        ft, div = [ctx.field(S.FACE_X + d, ns) for d in range(3)], ctx.field(S.CELL, ns)
        S.stochastic_mass_fluxdiv(ctx, ctx.field(S.CELL, ns, rho), ctx.field(S.CELL, 1, rt), ctx.field(S.CELL, ns, x),
                                  ctx.field(S.CELL, 1, mt), ctx.field(S.CELL, ns * ns, chi),
                                  ctx.field(S.CELL, ns * ns, G), div, ft, 0.01, [0.75, -0.5])
        assert bit_equal(div.download(), want)
        assert bit_equal([f.download() for f in ft], want_ft)


@pytest.mark.parametrize("ns,copies", [(5, 10), (6, 8)])
def test_matrices_beyond_the_last_level_cache(ns, copies):
    """A box of copies of a smaller one has the smaller one's fluxes, copied: the
    larger one's matrices exceed 256 MB, the smaller one's do not."""
    n = (64, 64, 32)
    rng = np.random.default_rng(ns)

    def run(m):
        N = (n[0], n[1], n[2] * m)
        with S.Context(3, N, 0.5, stag_mg_minwidth=min(N), mg_minwidth=min(N)) as ctx:
            S.set_species(ctx, ns, **kn)
            f = [ctx.field(S.CELL, a.shape[0], np.tile(a, (1, m, 1, 1))) for a in fields]
            ft, div = [ctx.field(S.FACE_X + d, ns) for d in range(3)], ctx.field(S.CELL, ns)
            S.diffusive_mass_fluxdiv(ctx, ns, f[0], f[1], f[2], f[3], f[4], div, f[5], f[6], None, ft)
            return [div.download()] + [q.download() for q in ft]

    kn = _knobs(ns, rng)
    shape = tuple(reversed(n))
    fields = [rng.uniform(0.2, 1.0, (k,) + shape) for k in (ns, 1, ns, ns * ns, ns * ns, 1, ns)]
    small, large = run(1), run(copies)
    assert ns * ns * np.prod(n) * copies * 8 > 256e6 > ns * ns * np.prod(n) * 8
    assert bit_equal(large, [np.tile(a, (1, copies, 1, 1)) for a in small])
