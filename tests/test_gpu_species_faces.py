"""The face-by-face form of compute_mass_fluxdiv's face pass, which boxes too thin
for tiles take.  The oracle's operations in the oracle's order: the same bits."""
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

