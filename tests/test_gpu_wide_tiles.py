"""The binning pass with 1024 threads a tile (launches of at most 256 tiles)
against the one with 256 in place, on both sides of that number: the same
charge, counts and particles after steps with arrivals and staged particles."""

import numpy as np
import pytest

from fopis_amd import lib as F

pytestmark = pytest.mark.gpu

NAMES = ("x", "y", "z", "vx", "vy", "vz")


def _run(monkeypatch, dims, precision, inplace):
    monkeypatch.setenv("FOPIS_TILE_INPLACE", inplace)
    species = [(-1.0, 1.0, 1e-3), (1.0, 100.0, 1e-3)]
    ctx = F.Context(F.make_desc(*dims, species, 1.0, precision=precision, mg_precision=F.FP32))
    rng = np.random.default_rng(8)
    lim = np.array(dims) - 1.0
    try:
        for s, n in enumerate((5003, 257)):
            p = np.concatenate([rng.uniform(0.0, 1.0, (n, 3)) * lim, rng.normal(0.0, 0.6, (n, 3))], axis=1)
            ctx.set_particles(s, {k: p[:, q] for q, k in enumerate(NAMES)})
        for k in range(3):
            for s in range(2):
                ctx.inject_maxwellian(s, [20, 30, 0, 7, 1, 5], 10 * k + s, [0.0, 0.0, 0.0], 0.3, 0.3)
            ctx.main_loop_es()
        out = [ctx.get_field(F.RHO), ctx.get_field(F.DENSITY, 0), ctx.get_field(F.DENSITY, 1)]
        for s in range(2):
            got = ctx.get_particles(s)
            a = np.stack([got[k] for k in NAMES], axis=1)
            out.append(a[np.lexsort(a.T)])
        return out
    finally:
        ctx.close()


@pytest.mark.parametrize("dims", [(9, 9, 9), (33, 33, 33), (33, 33, 65), (33, 33, 73)])
@pytest.mark.parametrize("precision", [F.FP64, F.FP32])
def test_wide_tiles_match(monkeypatch, dims, precision):
    for a, b in zip(_run(monkeypatch, dims, precision, "0"), _run(monkeypatch, dims, precision, "1")):
        assert np.array_equal(a, b)
