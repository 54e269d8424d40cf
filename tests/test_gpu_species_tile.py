"""The face pass of compute_mass_fluxdiv in 32 x 8 tiles: extents below, at and
past the tile's edges, every species count, with and without Gama, the
temperature and barodiffusion terms, one and two noise stages.  The oracle's
operations in the oracle's order: the same bits."""
import numpy as np
import pytest

from lowmachmixtures_amd import stokes as S
from oracle import oracle as O
from tests.helpers import bit_equal
from tests.test_gpu_species import _knobs, _mass_noise, _rho

pytestmark = pytest.mark.gpu

BOXES = [(2, (4, 2)), (2, (32, 8)), (2, (34, 10)), (2, (66, 18)), (3, (4, 2, 2)), (3, (32, 8, 2)), (3, (34, 6, 4)),
         (3, (30, 10, 6))]


@pytest.mark.parametrize("dim,n", BOXES)
@pytest.mark.parametrize("ns", range(2, 9))
@pytest.mark.parametrize("ideal,baro,stages", [(1, 0, 2), (0, 1, 1)])
def test_tiles(dim, n, ns, ideal, baro, stages):
    rng = np.random.default_rng(7 * ns + n[0])
    shape = tuple(reversed(n))
    kw = dict(is_ideal_mixture=ideal, fraction_tolerance=1e-8, Dtherm=list(rng.uniform(-0.5, 0.5, 8)))
    if baro and dim == 2:
        kw["barodiffusion_type"] = 1
    kn = _knobs(ns, rng, k_B=0.5, **kw)
    sp, g = O.species(ns, **kn), O.geom(dim, n, 0.5)
    rho, T = _rho(ns, shape, rng), rng.uniform(0.9, 1.1, shape)
    gpb = [rng.standard_normal(shape) for _ in range(dim)] if "barodiffusion_type" in kw else None
    W, w = _mass_noise(5, stages, dim, ns, shape), [1.0, 0.5][:stages]
    want = O.compute_mass_fluxdiv(g, sp, rho, T, 0.02, W, w, gradp_baro=gpb)
    # one multigrid level, so that no extent is halved to an odd one
    with S.Context(dim, n, 0.5, stag_mg_minwidth=min(n), mg_minwidth=min(n)) as ctx:
        S.set_species(ctx, ns, **kn)
        S.init_mass_stochastic(ctx, stages)
        S.fill_mass_stochastic(ctx, 5)
        f_rho, diff, stoch = ctx.field(S.CELL, ns, rho), ctx.field(S.CELL, ns), ctx.field(S.CELL, ns)
        ft = [ctx.field(S.FACE_X + d, ns) for d in range(dim)]
        gp = [ctx.field(S.FACE_X + d, 1, gpb[d]) for d in range(dim)] if gpb is not None else None
        S.compute_mass_fluxdiv(ctx, f_rho, gp, diff, stoch, ctx.field(S.CELL, 1, T), ft, 0.02, 0.0, w)
        for got, ref in zip((f_rho, diff, stoch), want[:3]):
            assert bit_equal(got.download(), ref)
        assert bit_equal([f.download() for f in ft], want[3])
