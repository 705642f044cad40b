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
        (128, 64, 127),  # one plane short of 8 MiB: plain
        (128, 64, 128),  # 8 MiB, whole chunks
        (64, 64, 257),  # 8 MiB and 32 KiB: a short last chunk
        (131, 129, 133),  # odd, more chunks than slots of its threads
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
