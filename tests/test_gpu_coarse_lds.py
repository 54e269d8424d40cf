"""The coarse V-cycle held in LDS, at the edges of its point-to-thread rule.

A thread owns one x-pair of a level per 1024 colour points: boxes whose first
coarse level has 2048 cells (one pair on every thread), just more (a second,
partly filled set), 4096 (two full sets), a handful of cells, extents that are
no powers of two, every viscosity type, 2D and 3D.  FP64 against the oracle
(the same bits: the division by a stored reciprocal rounds as x / d does) and
FP32 against one launch per pass."""
import numpy as np
import pytest

from lowmachmixtures_amd import problems as P
from lowmachmixtures_amd import stokes as S
from oracle import oracle as O
from tests.helpers import bit_equal, oracle_args, relerr

pytestmark = pytest.mark.gpu

# box, coarsest width of both multigrids
BOXES = [((32, 32, 16), 2), ((48, 32, 32), 3), ((32, 32, 32), 2), ((8, 4, 4), 2), ((40, 24, 8), 2),
         ((64, 128), 2), ((96, 96), 6), ((128, 128), 2), ((4, 4), 2), ((4096, 4), 2)]


@pytest.mark.parametrize("n,w", BOXES)
@pytest.mark.parametrize("visc", [-1, 1, 2, 3, -2, -3])
def test_staggered_matches_the_oracle_and_per_pass(n, w, visc, monkeypatch):
    dim = len(n)
    pb = P.small_problem(dim, n, visc_type=visc, seed=31, contrast=300.0)
    kw = dict(visc_type=visc, stag_mg_minwidth=w, mg_minwidth=w)
    rng = np.random.default_rng(6)
    rhs = [rng.standard_normal(pb.shape) for _ in range(dim)]
    guess = [rng.standard_normal(pb.shape) for _ in range(dim)]
    g, p, cf = oracle_args(pb, **kw)
    want = O.stag_mg_solver(g, p, cf, 0.7, rhs, phi=guess)
    with S.Context(dim, pb.n, pb.dx, **kw) as ctx:
        dp = S.DeviceProblem(ctx, pb, rhs=rhs)
        phi = ctx.faces(guess)
        ctx.profiling(True)
        S.stag_mg_solver(ctx, dp.alpha, dp.beta, dp.beta_ed, dp.gamma, 0.7, phi, dp.b_u)
        assert ctx.kernel_stats("stag_coarse")["launches"] > 0
        got = [f.download() for f in phi]
    assert bit_equal(got, want), relerr(got, want)
    sol = []
    for mode in ("0", "1"):
        monkeypatch.setenv("LMM_COARSE", mode)
        with S.Context(dim, pb.n, pb.dx, precision=S.FP32_MG, gmres_max_iter=3, **kw) as ctx:
            dp = S.DeviceProblem(ctx, pb, rhs=rhs)
            dp.solve()
            sol.append(dp.solution())
    assert bit_equal(sol[0][0], sol[1][0]) and bit_equal(sol[0][1], sol[1][1])


@pytest.mark.parametrize("n,w", BOXES)
def test_cell_centred_matches_the_oracle(n, w):
    dim = len(n)
    rng = np.random.default_rng(8)
    shape = tuple(reversed(n))
    ainv = [np.exp(2.0 * rng.standard_normal(shape)) for _ in range(dim)]
    rhs = rng.standard_normal(shape)
    rhs -= rhs.mean()
    kw = dict(mg_minwidth=w, stag_mg_minwidth=w)
    want = O.macproject(O.geom(dim, n, 0.3), O.params(**kw), ainv, rhs)
    with S.Context(dim, n, 0.3, **kw) as ctx:
        phi = ctx.field(S.CELL)
        ctx.profiling(True)
        S.macproject(ctx, phi, None, ctx.faces(ainv), ctx.field(S.CELL, 1, rhs))
        assert ctx.kernel_stats("cc_coarse")["launches"] > 0
        got = phi.download()
    assert bit_equal(got, want), relerr(got, want)
