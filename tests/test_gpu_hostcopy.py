"""Copies between caller arrays and the device through the pinned chunks: sizes
below and at the first chunked one, with a short last chunk, and two threads
that copy at the same time (one of them goes the plain way)."""

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _roundtrip(dims, rounds, seed, out):
    from fopis_amd import lib as F

    ctx = F.Context(F.make_desc(*[n - 2 for n in dims], [(-1.0, 1.0, 1.0)], 1.0))
    try:
        rng = np.random.default_rng(seed)
        for _ in range(rounds):
            a = rng.standard_normal(ctx.field_shape(F.RHO))
            ctx.set_field(F.RHO, a)
            out.append(np.array_equal(ctx.get_field(F.RHO), a))
    finally:
        ctx.close()


@pytest.mark.parametrize(
    "dims",
    [
        (6, 6, 7),  # small: one chunk
        (16, 16, 32),  # 64 KiB: the largest of those
        (16, 16, 33),  # plain
        (64, 64, 63),  # short of 2 MiB: plain both ways
        (64, 64, 64),  # 2 MiB: chunked on the way out
        (64, 64, 257),  # 8 MiB and 32 KiB: a short last chunk
        (128, 128, 192),  # 24 MiB: chunked both ways, whole chunks
        (131, 129, 193),  # odd
        (257, 259, 261),  # more chunks than slots
    ],
)
@pytest.mark.parametrize("threads", [1, 2])
def test_field_roundtrip(dims, threads):
    out = []
    th = [threading.Thread(target=_roundtrip, args=(dims, 3, 7 + t, out)) for t in range(threads)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert out == [True] * (3 * threads)


@pytest.mark.parametrize("n", [1, 1_365, 1_366, 700_001, 1_000_002])
def test_particle_roundtrip(n):
    """Six components in one copy, each at another address modulo 16 when n is odd."""
    from fopis_amd import lib as F

    ctx = F.Context(F.make_desc(17, 17, 17, [(-1.0, 1.0, 1.0)], 1.0))
    try:
        rng = np.random.default_rng(2)
        p = {k: rng.uniform(0.0, 16.0, n) for k in ("x", "y", "z")}
        p.update({k: rng.standard_normal(n) for k in ("vx", "vy", "vz")})
        ctx.set_particles(0, p)
        got = ctx.get_particles(0)
    finally:
        ctx.close()
    tile = lambda d: sum((np.minimum(d[k].astype(np.int64), 15) // 8) * f for k, f in (("x", 4), ("y", 2), ("z", 1)))
    order = np.argsort(tile(p), kind="stable")
    for k in p:
        assert np.array_equal(got[k], p[k][order])


def test_field_roundtrip_through_the_large_block():
    """The sizes of one to eight threads after copies large enough for the
    whole pinned block, and again once the last context gave it back."""
    for _ in range(2):
        out = []
        _roundtrip((257, 259, 261), 1, 1, out)
        from fopis_amd import lib as F

        keep = F.Context(F.make_desc(9, 9, 9, [(-1.0, 1.0, 1.0)], 1.0))
        try:
            for dims in ((257, 259, 261), (64, 64, 65), (67, 65, 131), (113, 117, 119), (129, 131, 133)):
                _roundtrip(dims, 3, 5, out)
        finally:
            keep.close()
        assert out == [True] * 16
