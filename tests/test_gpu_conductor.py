"""Conductor parity on the GPU: capture of particles by the voxel spacecraft
(surface charge, current), the capacitance matrix built by device unit-charge
solves, the FP64 charge redistribution, and whole steps with injection and a
floating conductor through the C++ host facade against the oracle."""
import ctypes
import json
import os

import numpy as np
import pytest

from oracle import refcpu
from tests.cases import CONFIGS, canon, device_desc, dst_poisson, load_config, oracle_params

pytestmark = pytest.mark.gpu

F = pytest.importorskip("fopis_amd.lib")

CUBE4 = os.path.join(CONFIGS, "objects", "cube4.obj")


def _cfg(nx=17):
    cfg = load_config("c2")
    cfg["Object"]["Spacecraft"]["file_name"] = CUBE4
    return cfg


def _oracle(nx=17, ppc=6, cmatrix=True):
    g = refcpu.Grid(oracle_params(_cfg(nx), nx=nx, ppc=ppc))
    if cmatrix:
        g.call("rc_build_cmatrix")
    g.call("rc_load_initial_particles")
    return g


def _ctx_with_object(g, Cm=None):
    ctx = F.Context(device_desc(g))
    ctx.set_object(0, g.cell_map(0), g.cmat_nodes(0))
    if Cm is not None:
        ctx.set_cmatrix(Cm, 0)
    for s in range(g.S):
        ctx.set_particles(s, g.get_particles(s))
    return ctx


def _union_obj(tmp_path, nx):
    """Two overlapping boxes of unequal widths per axis (cells [lo, hi)), so
    the sine-transform build orders its axes by width (z, y, x here)."""
    from fopis_amd.voxel_obj import voxels_from_boxes, write_obj

    boxes = [((9, 7, 5), (13, 13, 17)), ((10, 11, 8), (15, 16, 16))]
    lo = [min(b[0][q] for b in boxes) for q in range(3)]
    hi = [max(b[1][q] for b in boxes) for q in range(3)]
    path = os.path.join(str(tmp_path), "union.obj")
    write_obj(path, voxels_from_boxes(boxes, lo, hi), [lo[q] - nx // 2 for q in range(3)])
    return path


@pytest.mark.parametrize("shape", ["cube4", "union"])
def test_cmatrix_device_build_is_inverse_of_exact_b(tmp_path, shape):
    if shape == "cube4":
        g = _oracle(cmatrix=False)
    else:
        nx = 25
        cfg = _cfg(nx)
        cfg["Object"]["Spacecraft"]["file_name"] = _union_obj(tmp_path, nx)
        g = refcpu.Grid(oracle_params(cfg, nx=nx, ppc=1))
    ctx = F.Context(device_desc(g))
    nodes = g.cmat_nodes(0)
    ctx.set_object(0, g.cell_map(0), nodes)
    ctx.build_cmatrix(0)
    Cm = ctx.get_cmatrix(0)
    n = len(nodes)
    B = np.zeros((n, n))
    shp = (g.nx - 2,) * 3
    for j in range(n):
        b = np.zeros(shp)
        b[tuple(nodes[j] - 2)] = 1.0 / g.eps0()
        B[j] = dst_poisson(b)[tuple((nodes - 2).T)]
    Cx = np.linalg.inv(B)
    assert np.max(np.abs(Cm - Cx)) <= 1e-8 * np.max(np.abs(Cx))
    np.testing.assert_allclose(Cm, Cm.T, rtol=1e-8, atol=1e-8 * np.abs(Cx).max())


@pytest.mark.parametrize("n,dup", [(1, False), (63, False), (64, False), (65, False), (200, False), (70, True)])
def test_cmatrix_tile_edges(n, dup):
    """Node counts around the inversion's 64-wide tiles, on scattered nodes of
    an uneven grid; a node given twice makes B singular, which the call
    completes on as the pivoted elimination does (its values mean nothing).
    C is the one-column-at-a-time elimination's, element by element."""
    dims = (14, 11, 18)
    ctx = F.Context(F.make_desc(*dims, [(-1.0, 1.0, 1.0)], 2.5, mg_precision=F.FP64))
    rng = np.random.default_rng(n)
    inner = np.stack(np.meshgrid(*[np.arange(2, v) for v in dims], indexing="ij"), -1).reshape(-1, 3)
    nodes = inner[rng.permutation(len(inner))[:n]].astype(np.int32)
    if dup:
        nodes[-1] = nodes[0]
    mask = np.zeros([v + 1 for v in dims], np.uint8)
    mask[5, 5, 5] = 1
    ctx.set_object(0, mask, nodes)
    ctx.build_cmatrix(0)
    Cm = ctx.get_cmatrix(0)
    if dup:
        return
    B = np.zeros((n, n))
    for j in range(n):
        b = np.zeros([v - 2 for v in dims])
        b[tuple(nodes[j] - 2)] = 1.0 / 2.5
        B[j] = dst_poisson(b)[tuple((nodes - 2).T)]
    Cx = np.linalg.inv(B)
    # FP64 elimination of a positive definite B: a few n eps cond(B), cond < 1e3 here
    assert np.max(np.abs(Cm - Cx)) <= 1e-11 * np.max(np.abs(Cx))
    # the inverse of C in the same arithmetic: B's columns peak on the diagonal, C's do as well
    M = Cm.copy()
    I = np.eye(n)
    for c in range(n):
        assert np.argmax(np.abs(M[c:, c])) == 0
        d = M[c, c]
        M[c], I[c] = M[c] / d, I[c] / d
        f = M[:, c].copy()
        f[c] = 0.0
        M -= f[:, None] * M[c]
        I -= f[:, None] * I[c]
    assert np.max(np.abs(I - B)) <= 1e-11 * np.max(np.abs(B))


def _invert(ctx, B, peaked):
    """The library's inversion on a matrix of the device's memory: C, and whether the blocks did it."""
    vp = ctypes.c_void_p
    f = getattr(ctx.L, "_ZN5fopis14objects_invertERNS_3CtxEPdS2_ib")
    f.restype, f.argtypes = ctypes.c_bool, [vp, vp, vp, ctypes.c_int, ctypes.c_bool]
    hip = ctx.L  # (the runtime the library runs on)
    hip.hipMalloc.argtypes, hip.hipFree.argtypes = [vp, ctypes.c_size_t], [vp]
    hip.hipMemcpy.argtypes = [vp, vp, ctypes.c_size_t, ctypes.c_int]
    dev = [vp(), vp()]
    out = np.empty_like(B)
    for d in dev:
        assert hip.hipMalloc(ctypes.byref(d), B.nbytes) == 0
    assert hip.hipMemcpy(dev[0], B.ctypes.data, B.nbytes, 1) == 0
    done = f(ctx.h, dev[0], dev[1], len(B), peaked)
    assert hip.hipMemcpy(out.ctypes.data, dev[1], B.nbytes, 2) == 0
    for d in dev:
        hip.hipFree(d)
    return out, done


def _peaked(rng, n):
    """A positive definite matrix whose columns, and those of every Schur complement, peak on the diagonal."""
    a = rng.uniform(0.0, 1.0 / n, (n, n))
    return np.eye(n) + 0.5 * (a + a.T)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 128, 200])
def test_blocked_inversion_has_the_eliminations_bits(n):
    ctx = F.Context(F.make_desc(9, 9, 9, [(-1.0, 1.0, 1.0)], 1.0))
    B = _peaked(np.random.default_rng(n), n)
    got, done = _invert(ctx, B, True)
    want, other = _invert(ctx, B, False)
    assert done and not other
    np.testing.assert_array_equal(got, want)
    assert np.max(np.abs(got @ B - np.eye(n))) <= 1e-13 * n  # cond(B) < 4: a few n eps


@pytest.mark.parametrize("n,col,row", [
    (64, 5, 40),     # inside the first diagonal tile, no tile beside it
    (64, 62, 63),    # its last rows
    (128, 70, 100),  # inside the second one, which k_bj_update takes through its steps
    (128, 3, 64),    # the first row of the tile below
    (200, 10, 199),  # the last row, in a tile filled up with the identity
    (200, 130, 195),
])
def test_inversion_exchanges_rows_where_the_pivot_is_below(n, col, row):
    """A larger entry below the diagonal, found in the pivot's tile or in a
    panel: the pivoted elimination takes over, with the inverse of B."""
    ctx = F.Context(F.make_desc(9, 9, 9, [(-1.0, 1.0, 1.0)], 1.0))
    B = _peaked(np.random.default_rng(7), n)
    B[row, col], B[col, col], B[col, row] = 2.0, 0.25, 1.0
    got, done = _invert(ctx, B, True)
    want, _ = _invert(ctx, B, False)
    assert not done
    np.testing.assert_array_equal(got, want)
    assert np.linalg.cond(B) < 50
    assert np.max(np.abs(got - np.linalg.inv(B))) <= 1e-11 * np.max(np.abs(want))


@pytest.mark.parametrize("nx", [17, 41])
def test_capture_charge_and_current(nx):
    """At nx = 41 most tiles lie more than a tile away from the cube and skip
    the per-particle conductor lookup; capture must not change."""
    g = _oracle(nx=nx)
    Cm = g.cmatrix(0)
    ctx = _ctx_with_object(g, Cm)
    # a strong random field drives particles into the cube
    rng = np.random.default_rng(11)
    shp = g.field_shape(refcpu.EXREF)
    for q, w in enumerate((refcpu.EXREF, refcpu.EYREF, refcpu.EZREF)):
        E = rng.uniform(-0.4, 0.4, shp)
        g.set_field(w, E)
        ctx.set_field(F.EXREF + q, E)
    for _ in range(2):
        g.call("rc_update_velocity")
        g.call("rc_update_position")
        ctx.update_particle_velocity_es()
        ctx.update_particle_position_es()
    g.call("rc_deposit_only")  # capture, CIC, sumWholeCharge
    ctx.update_rho()
    st = ctx.object_state(0)
    cm_ref = g.object_charge(0)
    assert np.abs(cm_ref).sum() > 0, "no particle reached the conductor"
    np.testing.assert_allclose(st["charge_map"], cm_ref, rtol=0, atol=1e-12 * np.abs(cm_ref).max())
    # current = captured superparticles x q: integer-valued, exact
    np.testing.assert_array_equal(st["current"], g.object_charge(2))
    for s in range(g.S):
        a, b = canon(ctx.get_particles(s)), canon(g.get_particles(s))
        np.testing.assert_array_equal(a, b)
        r_a, r_b = ctx.get_field(F.RHO, s + 1), g.get_field(refcpu.RHO, s + 1)
        assert np.max(np.abs(r_a - r_b)) <= 1e-12 * np.max(np.abs(r_b))


def test_redistribution_on_zero_field():
    """With no plasma charge phi stays 0, so V = Q / sum(C) and rho[0] = V * rowsum(C)."""
    g = _oracle(ppc=1)
    Cm = g.cmatrix(0)
    ctx = _ctx_with_object(g, Cm)
    for s in range(g.S):
        ctx.set_particles(s, {k: np.zeros(0) for k in ("x", "y", "z", "vx", "vy", "vz")})
    rng = np.random.default_rng(5)
    n = Cm.shape[0]
    cmap = rng.normal(size=(g.S, n)) * 1e6
    ctx.set_object_charge_map(0, cmap)
    ctx.update_rho()
    st = ctx.object_state(0)
    Q = cmap.sum()
    V = Q / Cm.sum()
    assert abs(st["potential"] - V) <= 1e-12 * abs(V)
    assert abs(st["total_charge"] - Q) <= 1e-12 * np.abs(cmap).sum()
    rho0 = ctx.get_field(F.RHO, 0)
    nodes = g.cmat_nodes(0)
    got = rho0[tuple(nodes.T)]
    np.testing.assert_allclose(got, Cm @ np.full(n, V), rtol=1e-11, atol=1e-12 * np.abs(Cm @ np.full(n, V)).max())
    assert abs(rho0.sum() - Q) <= 1e-10 * np.abs(cmap).sum()


def test_host_steps_with_conductor_and_injection(tmp_path):
    """Whole mainLoopES steps through the C++ host facade (host mt19937 load and
    injection, device capacitance matrix) against the oracle with the same C."""
    from fopis_amd.host import Host

    cfg = _cfg(17)
    p = tmp_path / "c2s.json"
    p.write_text(json.dumps(cfg))
    g = _oracle(ppc=6)
    h = Host(str(p), nx_override=17, ppc_override=6, build_cmatrix=True, initialize=False)
    ctx = h.ctx
    Cg = ctx.get_cmatrix(0)
    Co = g.cmatrix(0)
    # the oracle's C comes from SOR solves stopped on the reference's pointwise test
    assert np.max(np.abs(Cg - Co)) <= 1e-3 * np.max(np.abs(Co))
    ctx.set_cmatrix(Co, 0)
    ctx.initialize()
    g.call("rc_initialize")
    for step in range(3):
        h.main_loop_es()
        g.call("rc_main_loop")
    for s in range(g.S):
        a, b = canon(ctx.get_particles(s)), canon(g.get_particles(s))
        assert abs(len(a) - len(b)) <= 2
        if len(a) == len(b):
            assert np.max(np.abs(a - b)) < 1e-6
    st = ctx.object_state(0)
    info = g.object_info(0)
    assert abs(st["potential"] - info["potential"]) <= 1e-4 * abs(info["potential"]) + 1e-12
    np.testing.assert_allclose(st["charge_map"].sum(), g.object_charge(0).sum(), rtol=1e-6)
    h.close()


def test_lshape_capture_and_cmatrix(tmp_path):
    """A non-convex conductor (an L of two 6 x 2 x 2 bars, as the C5
    spacecraft at small scale, written by fopis_amd.voxel_obj): the device
    capacitance matrix is the inverse of the exact unit-charge responses, and
    capture in a strong random field gives the oracle's charge map, current
    and surviving particles (Spacecraft.cpp:512-613, particle.cpp:82-204)."""
    from fopis_amd import voxel_obj

    path = str(tmp_path / "lsmall.obj")
    voxel_obj.write_boxes(path, [((-3, -1, -1), (3, 1, 1)), ((-1, -3, -1), (1, 3, 1))])
    cfg = load_config("c2")
    cfg["Object"]["Spacecraft"]["file_name"] = path
    g = refcpu.Grid(oracle_params(cfg, nx=17, ppc=6))
    g.call("rc_build_cmatrix")
    g.call("rc_load_initial_particles")
    nodes = g.cmat_nodes(0)
    assert len(nodes) > 30
    ctx = F.Context(device_desc(g))
    ctx.set_object(0, g.cell_map(0), nodes)
    ctx.build_cmatrix(0)
    Cm = ctx.get_cmatrix(0)
    n = len(nodes)
    B = np.zeros((n, n))
    shp = (g.nx - 2,) * 3
    for j in range(n):
        b = np.zeros(shp)
        b[tuple(nodes[j] - 2)] = 1.0 / g.eps0()
        B[j] = dst_poisson(b)[tuple((nodes - 2).T)]
    Cx = np.linalg.inv(B)
    assert np.max(np.abs(Cm - Cx)) <= 1e-8 * np.max(np.abs(Cx))
    for s in range(g.S):
        ctx.set_particles(s, g.get_particles(s))
    rng = np.random.default_rng(12)
    shp = g.field_shape(refcpu.EXREF)
    for q, w in enumerate((refcpu.EXREF, refcpu.EYREF, refcpu.EZREF)):
        E = rng.uniform(-0.4, 0.4, shp)
        g.set_field(w, E)
        ctx.set_field(F.EXREF + q, E)
    for _ in range(2):
        g.call("rc_update_velocity")
        g.call("rc_update_position")
        ctx.update_particle_velocity_es()
        ctx.update_particle_position_es()
    g.call("rc_deposit_only")
    ctx.update_rho()
    st = ctx.object_state(0)
    cm_ref = g.object_charge(0)
    assert np.abs(cm_ref).sum() > 0, "no particle reached the conductor"
    np.testing.assert_allclose(st["charge_map"], cm_ref, rtol=0, atol=1e-12 * np.abs(cm_ref).max())
    np.testing.assert_array_equal(st["current"], g.object_charge(2))
    for s in range(g.S):
        np.testing.assert_array_equal(canon(ctx.get_particles(s)), canon(g.get_particles(s)))
    ctx.close()


def test_thirty_steps_with_conductor_and_injection_track_the_oracle(tmp_path):
    """Thirty whole steps through the host facade (host mt19937 injection, a
    floating conductor with the oracle's C): the conductor's charge, its
    potential, the particle count and both energies stay with the oracle's.
    Measured: the charge equal to the last digit, potential and energies to
    1e-7 and better; the bars leave a margin of 10 to 100."""
    from fopis_amd.host import Host

    cfg = _cfg(17)
    p = tmp_path / "c2l.json"
    p.write_text(json.dumps(cfg))
    g = _oracle(ppc=6)
    h = Host(str(p), nx_override=17, ppc_override=6, build_cmatrix=True, initialize=False)
    ctx = h.ctx
    ctx.set_cmatrix(g.cmatrix(0), 0)
    ctx.initialize()
    g.call("rc_initialize")
    for _ in range(30):
        h.main_loop_es()
        g.call("rc_main_loop")
    st, info = ctx.object_state(0), g.object_info(0)
    q_dev, q_ref = st["charge_map"].sum(), g.object_charge(0).sum()
    assert abs(q_dev - q_ref) <= 1e-9 * abs(q_ref)
    assert abs(st["potential"] - info["potential"]) <= 1e-5 * abs(info["potential"])
    ke, fe = ctx.energy()
    assert abs(ke - g.L.rc_particle_energy(g.h)) <= 1e-8 * abs(ke)
    assert abs(fe - g.L.rc_efield_energy(g.h)) <= 1e-6 * abs(fe)
    for s in range(g.S):
        a, b = canon(ctx.get_particles(s)), canon(g.get_particles(s))  # the oracle's invalid particles dropped
        assert abs(len(a) - len(b)) <= 1e-3 * len(b)
    h.close()
