"""The level kernels of the V-cycle against one launch per sweep: the same
arithmetic in the same order, so the same bits, cycles and residual. Shapes:
all in the tail, level kernels above it, extents no multiple of the tile,
axes that stop coarsening early, and a finest level stored by colour."""

import numpy as np
import pytest

from fopis_amd import lib as F

pytestmark = pytest.mark.gpu


def _solve(monkeypatch, dims, precision, fused):
    monkeypatch.setenv("FOPIS_MG_FUSED", fused)
    ctx = F.Context(F.make_desc(*dims, [(-1.0, 1.0, 1.0)], 1.0, mg_precision=precision))
    try:
        rho = np.random.default_rng(11).standard_normal(ctx.field_shape(F.RHO))
        ctx.set_field(F.RHO, rho)
        out = [ctx.solve_poisson()]
        ctx.set_field(F.RHO, rho[::-1].copy())  # a warm start
        out.append(ctx.solve_poisson())
        return out, ctx.get_field(F.PHI)
    finally:
        ctx.close()


@pytest.mark.parametrize(
    "dims",
    [
        (9, 17, 11),
        (17, 17, 17),
        (33, 33, 33),
        (41, 21, 57),
        (33, 49, 25),
        (18, 16, 21),
        (65, 5, 35),
        (97, 81, 113),
        (129, 97, 161),
    ],
)
@pytest.mark.parametrize("precision", [F.FP64, F.FP32])
def test_levels_match_single_sweeps(monkeypatch, dims, precision):
    if precision == F.FP64 and dims == (129, 97, 161):
        pytest.skip("the colour-split finest level is FP32")
    got, phi = _solve(monkeypatch, dims, precision, "1")
    want, ref = _solve(monkeypatch, dims, precision, "0")
    assert np.isfinite(phi).all()
    assert got == want
    assert np.array_equal(phi, ref)


@pytest.mark.parametrize("dims", [(17, 17, 17), (33, 49, 25), (65, 65, 65)])
def test_whole_solve_graph_matches_launches(monkeypatch, dims):
    """Enough solves of alternating charges that a whole solve becomes one
    graph, replayed between other work, against the solves launch by launch."""
    rng = np.random.default_rng(4)
    rhos = None
    out = []
    for graph in ("1", "0"):
        monkeypatch.setenv("FOPIS_MG_GRAPH", graph)
        ctx = F.Context(F.make_desc(*dims, [(-1.0, 1.0, 1.0)], 1.0, mg_precision=F.FP32))
        try:
            if rhos is None:
                rhos = [rng.standard_normal(ctx.field_shape(F.RHO)) for _ in range(3)]
            zero = np.zeros(ctx.field_shape(F.PHI))
            got = []
            for k in range(60):
                ctx.set_field(F.RHO, rhos[k % 3])
                ctx.set_field(F.PHI, zero)
                got.append((ctx.solve_poisson(), ctx.get_field(F.PHI)))
                if k % 7 == 0:
                    ctx.update_efield()
            out.append(got)
        finally:
            ctx.close()
    for (a, phi), (b, ref) in zip(*out):
        assert a == b and np.array_equal(phi, ref)
