"""Face conditions after a solve, applied in one launch, against the reference's
order of six faces: all kinds, kinds that meet at an edge, the smallest grid."""

import numpy as np
import pytest

from fopis_amd import lib as F

pytestmark = pytest.mark.gpu


def _in_order(phi, bc):
    for f, kind in enumerate(bc):
        axis, up = f // 2, f % 2
        a = np.moveaxis(phi, axis, 0)[:, 1:-1, 1:-1]
        t, s = (-2, -3) if up else (1, 2)
        a[t] = a[s] if kind == "N" else 0.0


@pytest.mark.parametrize("dims", [(4, 4, 4), (17, 9, 70), (33, 65, 12)])
@pytest.mark.parametrize("bc", ["DDDDDD", "NNNNNN", "DNNDND", "NDDDDN", "NNDDDD", "DDDDNN"])
def test_faces_match_the_order(dims, bc):
    ctx = F.Context(F.make_desc(*dims, [(-1.0, 1.0, 1.0)], 1.0, boundary=bc))
    try:
        rng = np.random.default_rng(5)
        ctx.set_field(F.RHO, rng.standard_normal(ctx.field_shape(F.RHO)))
        ctx.set_field(F.PHI, rng.standard_normal(ctx.field_shape(F.PHI)))
        ctx.solve_poisson()
        phi = ctx.get_field(F.PHI)
    finally:
        ctx.close()
    want = phi.copy()
    for f in range(6):
        np.moveaxis(want, f // 2, 0)[:, 1:-1, 1:-1][-2 if f % 2 else 1] = 7.0
    _in_order(want, bc)
    assert np.array_equal(phi, want)
