"""Which form of the fused sweep a level takes by default (kernel_stats counts
each form's launches): bricks where they pay, the colour kernels where bricks
hang far over the box or a single component's are many, at the edges of the
rule; and the same bits whatever the form."""
import pytest

from lowmachmixtures_amd import problems as P
from lowmachmixtures_amd import stokes as S
from tests.helpers import bit_equal

pytestmark = pytest.mark.gpu

FORMS = ["brick4", "brick8", "march", "march_pairs", "march_narrow", "plane", "block", "tile2d"]


def forms(ctx, multigrid):
    return {f for f in FORMS if ctx.kernel_stats(f"{multigrid}_sweep_{f}")["launches"] > 0}


# one-level boxes: box, visc_type, precision, form of the staggered and of the cell-centred sweep (None: colour)
CASES = [
    ((32, 32, 32), -1, "fp64", "brick4", "brick4"),
    ((64, 64, 64), -1, "fp64", "brick8", "brick4"),
    ((64, 64, 64), -1, "fp32", "brick8", "brick4"),
    ((16, 64, 64), 1, "fp64", "brick4", "brick4"),   # thin, but few bricks
    ((8, 128, 128), -1, "fp64", "brick8", None),     # a quarter of each brick lies in the box; 512 of 8 rows
    ((8, 128, 176), -1, "fp64", None, None),         # 704
    ((8, 128, 176), -1, "fp32", "brick8", None),
    ((8, 128, 304), -1, "fp32", None, None),         # 1216
    ((128, 12, 128), -1, "fp32", "brick4", "brick4"),  # 8 rows would hang over by a third
    ((32, 32, 32), -2, "fp64", "brick4", "brick4"),  # launch-bound
    ((32, 32, 32), -3, "fp32", "brick4", "brick4"),
    ((64, 32, 32), 2, "fp64", "brick4", "brick4"),
    ((64, 64, 64), 3, "fp64", "brick4", "brick4"),
    ((64, 64, 64), -2, "fp64", None, "brick4"),      # one component, variable coefficients
    ((64, 64, 64), -3, "fp32", "brick4", "brick4"),
    ((96, 64, 64), -3, "fp32", None, "brick4"),      # more than 640 bricks
    ((48, 48, 48), 2, "fp64", None, "brick4"),       # three quarters full
    ((36, 72, 72), 1, "fp64", "brick8", "brick4"),   # 648 bricks, half full
    ((40, 72, 80), 1, "fp64", "brick8", None),       # 720 bricks; 8 rows: 360 for each of three components
    ((96, 64, 64), 2, "fp32", None, "brick4"),
    ((80, 64, 52), 2, "fp64", None, "brick4"),       # 624 bricks, 83 % full
    ((96, 48, 64), 3, "fp64", "brick4", "brick4"),   # 576, full
]


@pytest.mark.parametrize("n,visc,prec,stag,cc", CASES)
def test_form_by_default(n, visc, prec, stag, cc, monkeypatch):
    pb = P.small_problem(3, n, visc_type=visc, seed=51, contrast=20.0)
    b_u = P.rhs_from_noise_host(pb)
    kw = dict(visc_type=visc, stag_mg_minwidth=min(n), mg_minwidth=min(n), gmres_max_iter=2,
              precision=S.FP32_MG if prec == "fp32" else S.FP64)
    sol = []
    for smoother in (None, "colour"):
        if smoother:
            monkeypatch.setenv("LMM_SMOOTHER", smoother)
        with S.Context(3, pb.n, pb.dx, **kw) as ctx:
            dp = S.DeviceProblem(ctx, pb, rhs=b_u)
            ctx.profiling(True)
            dp.solve()
            want = (set(), set()) if smoother else ({stag} - {None}, {cc} - {None})
            assert (forms(ctx, "stag"), forms(ctx, "cc")) == want
            sol.append(dp.solution())
    assert bit_equal(sol[0][0], sol[1][0]) and bit_equal(sol[0][1], sol[1][1])


@pytest.mark.parametrize("tiles,stag,cc", [(64, True, True), (65, True, False), (128, True, False), (129, False, False)])
def test_min_tiles_counts_a_sweeps_workgroups(tiles, stag, cc, monkeypatch):
    """256 x 128: 64 tiles, 128 workgroups for the two components of a sweep."""
    monkeypatch.setenv("LMM_FUSED_MIN_TILES", str(tiles))
    pb = P.small_problem(2, (256, 128), visc_type=-1, seed=52)
    with S.Context(2, pb.n, pb.dx, stag_mg_minwidth=128, mg_minwidth=128, visc_type=-1, gmres_max_iter=1) as ctx:
        dp = S.DeviceProblem(ctx, pb, rhs=P.rhs_from_noise_host(pb))
        ctx.profiling(True)
        dp.solve()
        assert (forms(ctx, "stag"), forms(ctx, "cc")) == ({"tile2d"} if stag else set(), {"tile2d"} if cc else set())
