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


def _species(monkeypatch, dims, precision, inplace, which, fused):
    """One step of the given species of eight, in one context: what each of them leaves."""
    monkeypatch.setenv("FOPIS_TILE_INPLACE", inplace)
    eight = [((-1.0) ** s, 1.0 + s, 1e-3 * (1 + s)) for s in range(8)]
    ctx = F.Context(F.make_desc(*dims, [eight[s] for s in which], 1.0, precision=precision, mg_precision=F.FP32))
    lim = np.array(dims) - 1.0
    try:
        for q, s in enumerate(which):
            rng = np.random.default_rng(20 + s)
            n = 300 * (8 - s) + 1
            p = np.concatenate([rng.uniform(0.0, 1.0, (n, 3)) * lim, rng.normal(0.0, 0.5, (n, 3))], axis=1)
            ctx.set_particles(q, {k: p[:, c] for c, k in enumerate(NAMES)})
            ctx.inject_maxwellian(q, [5 + s, 0, 3, 1, 9, 2], 40 + s, [0.0, 0.0, 0.0], 0.3, 0.3)
        e = np.random.default_rng(3)
        for w in (F.EXREF, F.EYREF, F.EZREF):
            ctx.set_field(w, 0.1 * e.standard_normal(ctx.field_shape(w)))
        if fused:
            ctx.main_loop_es()
        else:
            ctx.update_particle_velocity_es()
            ctx.update_particle_position_es()
            ctx.update_density()
            ctx.update_rho()
        out = []
        for q in range(len(which)):
            got = ctx.get_particles(q)
            a = np.stack([got[k] for k in NAMES], axis=1)
            out.append([a[np.lexsort(a.T)], ctx.get_field(F.RHO, q + 1), ctx.get_field(F.DENSITY, q), ctx.num_particles(q),
                        ctx.moments(q)["mean_v"]])
        return out
    finally:
        ctx.close()


@pytest.mark.parametrize("count", [4, 5, 8])
@pytest.mark.parametrize("precision", [F.FP64, F.FP32])
@pytest.mark.parametrize("inplace", ["0", "1"])
@pytest.mark.parametrize("fused", [True, False])
def test_species_of_several_launches(monkeypatch, count, precision, inplace, fused):
    """Four species go through a launch; with more, each leaves what it leaves alone."""
    together = _species(monkeypatch, (17, 25, 17), precision, inplace, list(range(count)), fused)
    for s in range(count):
        (alone,) = _species(monkeypatch, (17, 25, 17), precision, inplace, [s], fused)
        for a, b in zip(together[s][:4], alone[:4]):
            assert np.array_equal(a, b)
        np.testing.assert_allclose(together[s][4], alone[4], rtol=1e-12, atol=1e-12)
