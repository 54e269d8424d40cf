"""The 2D red-black sweep in 32 x 16 tiles: every viscosity type, boxes that the
tiles divide, hang over and are larger than, odd and even sweep counts, the
zero-guess first sweep; against the oracle in FP64 and against the colour
kernels (LMM_SMOOTHER=colour) in a whole FP32 solve.  Same point code: the same bits."""
import numpy as np
import pytest

from lowmachmixtures_amd import problems as P
from lowmachmixtures_amd import stokes as S
from oracle import oracle as O
from tests.helpers import bit_equal, oracle_args, relerr

pytestmark = pytest.mark.gpu

# box, coarsest width (every level's extents stay even)
BOXES = [((32, 16), 4), ((64, 64), 2), ((96, 80), 10), ((34, 18), 18), ((4, 6), 4), ((66, 34), 34), ((30, 50), 30)]
SWEEPS = [(2, 2, 8), (1, 3, 3)]


def _kw(w, sweeps, visc=-1):
    return dict(visc_type=visc, stag_mg_minwidth=w, mg_minwidth=w, stag_mg_nsmooths_down=sweeps[0],
                stag_mg_nsmooths_up=sweeps[1], stag_mg_nsmooths_bottom=sweeps[2], mg_nsmooths_down=sweeps[0],
                mg_nsmooths_up=sweeps[1], mg_nsmooths_bottom=sweeps[2])


@pytest.mark.parametrize("n,w", BOXES)
@pytest.mark.parametrize("visc", [-1, 1, 2, 3, -2, -3])
@pytest.mark.parametrize("sweeps", SWEEPS)
def test_staggered(n, w, visc, sweeps, monkeypatch):
    pb = P.small_problem(2, n, visc_type=visc, seed=43, contrast=50.0)
    kw = _kw(w, sweeps, visc)
    rng = np.random.default_rng(3)
    rhs, guess = ([rng.standard_normal(pb.shape) for _ in range(2)] for _ in range(2))
    g, p, cf = oracle_args(pb, **kw)
    want = O.stag_mg_solver(g, p, cf, 0.9, rhs, phi=guess)
    monkeypatch.setenv("LMM_COARSE", "0")
    with S.Context(2, pb.n, pb.dx, **kw) as ctx:
        dp = S.DeviceProblem(ctx, pb, rhs=rhs)
        phi = ctx.faces(guess)
        ctx.profiling(True)
        S.stag_mg_solver(ctx, dp.alpha, dp.beta, dp.beta_ed, dp.gamma, 0.9, phi, dp.b_u)
        assert ctx.kernel_stats("stag_rb_fused")["launches"] > 0
        got = [f.download() for f in phi[:2]]
    assert bit_equal(got, want[:2]), relerr(got, want[:2])
    sol = []
    for smoother in ("colour", "fused"):
        monkeypatch.setenv("LMM_SMOOTHER", smoother)
        with S.Context(2, pb.n, pb.dx, precision=S.FP32_MG, gmres_max_iter=3, **kw) as ctx:
            dp = S.DeviceProblem(ctx, pb, rhs=rhs)
            ctx.profiling(True)
            dp.solve()
            assert (ctx.kernel_stats("stag_rb_fused")["launches"] > 0) == (smoother == "fused")
            sol.append(dp.solution())
    assert bit_equal(sol[0][0], sol[1][0]) and bit_equal(sol[0][1], sol[1][1])


@pytest.mark.parametrize("n,w", BOXES)
@pytest.mark.parametrize("sweeps", SWEEPS)
def test_cell_centred(n, w, sweeps, monkeypatch):
    rng = np.random.default_rng(9)
    shape = tuple(reversed(n))
    ainv = [0.5 + rng.random(shape) for _ in range(2)]
    rhs = rng.standard_normal(shape)
    rhs -= rhs.mean()
    kw = _kw(w, sweeps)
    want = O.macproject(O.geom(2, n, 0.4), O.params(**kw), ainv, rhs)
    monkeypatch.setenv("LMM_COARSE", "0")
    with S.Context(2, n, 0.4, **kw) as ctx:
        phi = ctx.field(S.CELL)
        S.macproject(ctx, phi, None, ctx.faces(ainv), ctx.field(S.CELL, 1, rhs))
        got = phi.download()
    assert bit_equal(got, want), relerr(got, want)
