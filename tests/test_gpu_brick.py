"""The brick form of the fused red-black sweep: every viscosity type, boxes
that 32 x 4 x 4 bricks divide and boxes they hang over, extents smaller than a
brick, odd and even sweep counts, the zero-guess first sweep; against the
oracle in FP64 and against the plane-marching / colour kernels
(LMM_SWEEP_BRICK=0) in a whole FP32 solve.  Same point code: the same bits."""
import numpy as np
import pytest

from lowmachmixtures_amd import problems as P
from lowmachmixtures_amd import stokes as S
from oracle import oracle as O
from tests.helpers import bit_equal, oracle_args, relerr

pytestmark = pytest.mark.gpu

# box, coarsest width (every level's extents stay even)
BOXES = [((32, 32, 32), 2), ((48, 40, 24), 6), ((36, 4, 6), 6), ((4, 8, 4), 4), ((64, 12, 20), 6), ((34, 6, 10), 6)]


@pytest.mark.parametrize("n,w", BOXES)
@pytest.mark.parametrize("visc", [-1, 1, 2, 3, -2, -3])
@pytest.mark.parametrize("sweeps", [(2, 2, 8), (1, 3, 3)])
def test_staggered(n, w, visc, sweeps, monkeypatch):
    pb = P.small_problem(3, n, visc_type=visc, seed=41, contrast=50.0)
    kw = dict(visc_type=visc, stag_mg_minwidth=w, mg_minwidth=w, stag_mg_nsmooths_down=sweeps[0],
              stag_mg_nsmooths_up=sweeps[1], stag_mg_nsmooths_bottom=sweeps[2])
    rng = np.random.default_rng(3)
    rhs = [rng.standard_normal(pb.shape) for _ in range(3)]
    guess = [rng.standard_normal(pb.shape) for _ in range(3)]
    g, p, cf = oracle_args(pb, **kw)
    want = O.stag_mg_solver(g, p, cf, 0.9, rhs, phi=guess)
    monkeypatch.setenv("LMM_COARSE", "0")
    with S.Context(3, pb.n, pb.dx, **kw) as ctx:
        dp = S.DeviceProblem(ctx, pb, rhs=rhs)
        phi = ctx.faces(guess)
        ctx.profiling(True)
        S.stag_mg_solver(ctx, dp.alpha, dp.beta, dp.beta_ed, dp.gamma, 0.9, phi, dp.b_u)
        assert ctx.kernel_stats("stag_rb_fused")["launches"] > 0
        got = [f.download() for f in phi]
    assert bit_equal(got, want), relerr(got, want)
    sol = []
    for brick in ("0", "1000000"):
        monkeypatch.setenv("LMM_SWEEP_BRICK", brick)
        with S.Context(3, pb.n, pb.dx, precision=S.FP32_MG, gmres_max_iter=3, **kw) as ctx:
            dp = S.DeviceProblem(ctx, pb, rhs=rhs)
            dp.solve()
            sol.append(dp.solution())
    assert bit_equal(sol[0][0], sol[1][0]) and bit_equal(sol[0][1], sol[1][1])


@pytest.mark.parametrize("n,w", BOXES)
def test_cell_centred(n, w, monkeypatch):
    rng = np.random.default_rng(9)
    shape = tuple(reversed(n))
    ainv = [0.5 + rng.random(shape) for _ in range(3)]
    rhs = rng.standard_normal(shape)
    rhs -= rhs.mean()
    kw = dict(mg_minwidth=w, stag_mg_minwidth=w, mg_nsmooths_down=1, mg_nsmooths_up=2, mg_nsmooths_bottom=3)
    want = O.macproject(O.geom(3, n, 0.4), O.params(**kw), ainv, rhs)
    monkeypatch.setenv("LMM_COARSE", "0")
    with S.Context(3, n, 0.4, **kw) as ctx:
        phi = ctx.field(S.CELL)
        S.macproject(ctx, phi, None, ctx.faces(ainv), ctx.field(S.CELL, 1, rhs))
        got = phi.download()
    assert bit_equal(got, want), relerr(got, want)


# 8 rows are the rule from 768 bricks on; boxes that 8 rows divide, hang over by a
# row, by four, and are larger than
ROW_BOXES = [((32, 16, 8), 8), ((36, 12, 6), 6), ((34, 10, 10), 10), ((4, 4, 8), 4), ((66, 22, 4), 4)]


@pytest.mark.parametrize("n,w", ROW_BOXES)
@pytest.mark.parametrize("rows", ["4", "8"])
@pytest.mark.parametrize("visc", [-1, 1])
def test_brick_rows(n, w, rows, visc, monkeypatch):
    """Both row counts of the three-component and of the cell-centred sweep: FP64
    against the oracle, FP32 against the colour kernels."""
    monkeypatch.setenv("LMM_BRICK_ROWS", rows)
    monkeypatch.setenv("LMM_SWEEP_BRICK", "1000000")
    monkeypatch.setenv("LMM_COARSE", "0")
    pb = P.small_problem(3, n, visc_type=visc, seed=43, contrast=50.0)
    kw = dict(visc_type=visc, stag_mg_minwidth=w, mg_minwidth=w, stag_mg_nsmooths_down=1, stag_mg_nsmooths_bottom=3)
    rng = np.random.default_rng(5)
    rhs = [rng.standard_normal(pb.shape) for _ in range(3)]
    guess = [rng.standard_normal(pb.shape) for _ in range(3)]
    g, p, cf = oracle_args(pb, **kw)
    want = O.stag_mg_solver(g, p, cf, 0.9, rhs, phi=guess)
    ainv = [0.5 + rng.random(pb.shape) for _ in range(3)]
    r0 = rhs[0] - rhs[0].mean()
    want_phi = O.macproject(g, p, ainv, r0)
    with S.Context(3, pb.n, pb.dx, **kw) as ctx:
        dp = S.DeviceProblem(ctx, pb, rhs=rhs)
        phi, cc = ctx.faces(guess), ctx.field(S.CELL)
        ctx.profiling(True)
        S.stag_mg_solver(ctx, dp.alpha, dp.beta, dp.beta_ed, dp.gamma, 0.9, phi, dp.b_u)
        S.macproject(ctx, cc, None, ctx.faces(ainv), ctx.field(S.CELL, 1, r0))
        for multigrid in ("stag", "cc"):
            assert ctx.kernel_stats(f"{multigrid}_sweep_brick{rows}")["launches"] > 0
            assert ctx.kernel_stats(f"{multigrid}_sweep_brick{12 - int(rows)}")["launches"] == 0
        got, got_phi = [f.download() for f in phi], cc.download()
    assert bit_equal(got, want), relerr(got, want)
    assert bit_equal(got_phi, want_phi), relerr(got_phi, want_phi)
    sol = []
    for smoother in ("colour", None):
        if smoother:
            monkeypatch.setenv("LMM_SMOOTHER", smoother)
        else:
            monkeypatch.delenv("LMM_SMOOTHER")
        with S.Context(3, pb.n, pb.dx, precision=S.FP32_MG, gmres_max_iter=3, **kw) as ctx:
            dp = S.DeviceProblem(ctx, pb, rhs=rhs)
            dp.solve()
            sol.append(dp.solution())
    assert bit_equal(sol[0][0], sol[1][0]) and bit_equal(sol[0][1], sol[1][1])
