"""Staged particles in tile order: host-staged ones first, then the ones drawn
on the device, each tile's in the order they came, those outside the domain
dropped; around the sizes of a wave, a block and the most blocks, and with
tile keys of one, two and three digits."""

import numpy as np
import pytest

from fopis_amd import lib as F

pytestmark = pytest.mark.gpu

NAMES = ("x", "y", "z", "vx", "vy", "vz")


def _tile(p, dims):
    c = [np.minimum(np.floor(p[:, q]).astype(np.int64), dims[q] - 2) // 8 for q in range(3)]
    t = [-(-(n - 1) // 8) for n in dims]
    return (c[0] * t[1] + c[1]) * t[2] + c[2]


@pytest.mark.parametrize(
    "dims, counts",
    [
        ((9, 9, 9), (1, 0)),  # a single tile
        ((33, 25, 17), (63, 65)),
        ((33, 25, 17), (256, 16385)),  # 64 blocks and one particle more
        ((129, 57, 41), (16384, 257)),  # two digits
        ((65, 65, 65), (2**20 + 3, 70000)),  # more than 64 blocks
        ((8 * 65537 + 1, 5, 5), (5000, 3)),  # three digits
    ],
)
def test_staged_order(monkeypatch, dims, counts):
    # (binning in place keeps a tile's order: residents, then staged; the
    # residents give each tile the capacity for its staged ones)
    monkeypatch.setenv("FOPIS_TILE_INPLACE", "1")
    ctx = F.Context(F.make_desc(*dims, [(-1.0, 1.0, 1.0), (1.0, 100.0, 1.0)], 1.0, capacity_slack=4.0))
    rng = np.random.default_rng(3)
    xmax = np.array(dims) - 1.0
    try:
        for s, n in enumerate(counts):
            p = np.empty((n, 6))
            p[:, :3] = rng.uniform(-0.01, 1.01, (n, 3)) * xmax
            p[: n // 3, :3] = rng.uniform(0.0, 1.0, (n // 3, 3)) * np.minimum(xmax, 9.0)  # a crowded corner
            p[:, 3:] = rng.standard_normal((n, 3))
            inside = p[((p[:, :3] >= 0.0) & (p[:, :3] <= xmax)).all(axis=1)][::-1]
            ctx.set_particles(s, {k: inside[:, q] for q, k in enumerate(NAMES)})
            ctx.add_particles(s, {k: p[:, q] for q, k in enumerate(NAMES)})
            ctx.inject_maxwellian(s, [3, 2, 1, 4, 0, 5 if n > 1 else 0], 9 + s, [0.0, 0.0, 0.0], 0.01, 0.01)
        want = []
        for s in range(2):
            got = ctx.get_particles(s)  # residents, host-staged as they came, drawn ones inside
            a = np.stack([got[k] for k in NAMES], axis=1)
            a = a[((a[:, :3] >= 0.0) & (a[:, :3] <= xmax)).all(axis=1)]
            want.append(a[np.argsort(_tile(a, dims), kind="stable")])
        ctx.update_rho()
        for s in range(2):
            got = ctx.get_particles(s)
            assert np.array_equal(np.stack([got[k] for k in NAMES], axis=1), want[s])
    finally:
        ctx.close()
