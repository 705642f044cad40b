"""Error paths of the library's host code, on the CPU in front of a HIP
runtime without a device (fake_hip/fake_hip.cpp, preloaded into a process of
its own per case): failed allocations and launches, a stream that reports an
error, and what a call leaves behind for the next one."""

import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C
import numpy as np
from fopis_amd import guess as G
from fopis_amd import lib as F

ARG, DEVICE, NOMEM = -1, -3, -4
fake = C.CDLL(None)
fake.fake_log.restype = C.c_char_p


def log(clear=True):
    lines = fake.fake_log().decode().splitlines()
    if clear:
        fake.fake_log_clear()
    return lines


def context(*dims, **kw):
    return F.Context(F.make_desc(*dims, [(-1.0, 1.0, 1.0)], 1.0, **kw))


def refused(f, *a, **kw):
    try:
        f(*a, **kw)
    except F.FopisError as e:
        return e.code
    return 0
"""


@pytest.fixture(scope="session")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake_hip") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-w",
                    os.path.join(HERE, "fake_hip", "fake_hip.cpp"), "-o", so, "-lpthread", "-ldl"], check=True)

    def run(body, env=None):
        before = os.environ.get("LD_PRELOAD")
        e = dict(os.environ, LD_PRELOAD=f"{so} {before}" if before else so, PYTHONPATH=ROOT, **(env or {}))
        r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body)], env=e, cwd=ROOT, capture_output=True,
                           text=True, timeout=240)
        assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout}\n{r.stderr}"

    return run


def test_reported_failure_is_not_reported_again(fake):
    """A call that reported a failed allocation, or a program's own failed
    launch: copies afterwards, small and large, return their bytes. (They
    returned the earlier error as theirs.)"""
    fake("""
    for dims in ((9, 9, 9), (81, 81, 81)):
        ctx = context(*dims)
        rho = np.random.default_rng(1).standard_normal(ctx.field_shape(F.RHO))
        ctx.set_field(F.RHO, rho)
        fake.fake_fail_malloc(0)
        assert refused(ctx.get_field, F.EX) == NOMEM
        assert np.array_equal(ctx.get_field(F.RHO), rho)
        fake.hipMemcpy(None, None, 8, 0)  # an error the program has not asked for yet
        assert np.array_equal(ctx.get_field(F.RHO), rho)
        fake.fake_delay(20)  # longer than the copy asks the stream in between
        assert np.array_equal(ctx.get_field(F.RHO), rho)
        fake.fake_delay(0)
        assert fake.hipGetLastError() in (0, 1)  # the program's, or overwritten by the stream's "not ready"
        ctx.set_field(F.RHO, rho)
        ctx.close()
    """)


def test_failed_gradient_leaves_nothing_queued(fake):
    """An allocation that fails in the middle of a backward pass: the next pass
    reduces its own 15 layers, as on a fresh network. (The layers queued by the
    failed pass stayed, and were written past the end of their list.)"""
    fake("""
    def net():
        ctx = context(17, 17, 17)
        g = G.Guess(ctx)
        g.dataset_alloc(1)
        n = G.net_grid(17, 17, 17)
        g.dataset_set(0, np.zeros(n, np.uint16), np.zeros(n, np.uint8), np.zeros(n, np.uint16))
        return ctx, g

    ctx, g = net()
    log()
    g.grad(0)
    clean = log()
    allocs = sum(s.startswith("malloc") for s in clean)
    own = lambda lines: [s for s in lines if s.startswith("launch") and "k_move" not in s and "k_landed" not in s]
    launches = own(clean)
    reduces = [s for s in launches if "k_wgrad_reduce" in s]
    assert len(reduces) == 1
    failed = 0
    for k in range(allocs - 15, allocs):  # the partial sums of each layer
        ctx, g = net()
        fake.fake_fail_malloc(k)
        assert refused(g.grad, 0) == NOMEM
        failed += 1
        log()
        g.grad(0)
        assert own(log()) == launches
    assert failed == 15
    """)


@pytest.mark.parametrize("out", [True, False])
def test_copy_ends_when_its_stream_fails(fake, out):
    """A stream that fails at any chunk of a copy by several threads: the copy
    returns the error, and the next one works. (The threads still waiting for
    a chunk were not told once the calling one had moved its own.)"""
    fake(f"""
    ctx = context(65, 65, 700)
    rho = np.random.default_rng(1).standard_normal(ctx.field_shape(F.RHO))
    ctx.set_field(F.RHO, rho)
    assert np.array_equal(ctx.get_field(F.RHO), rho)
    for k in range(30):
        for again in range(3):
            log()
            fake.fake_break_stream_after(k)
            code = refused(ctx.get_field, F.RHO) if {out} else refused(ctx.set_field, F.RHO, rho)
            fake.fake_break_stream_after(-1)
            fake.fake_break_stream(0)
            n = sum("k_move" in s or "k_landed" in s for s in log())
            assert code == (DEVICE if k < n else 0), (k, n, code)
            assert np.array_equal(ctx.get_field(F.RHO), rho)
    """)


@pytest.mark.parametrize("out", [True, False])
def test_copy_with_fewer_threads(fake, out):
    """Any of a copy's threads cannot be started for want of memory: the others
    move its chunks. (The process ended.)"""
    fake(f"""
    ctx = context(65, 65, 700)
    rho = np.random.default_rng(1).standard_normal(ctx.field_shape(F.RHO))
    for k in range(8):
        ctx.set_field(F.RHO, 0 * rho)
        if {out}:
            ctx.set_field(F.RHO, rho)
        fake.fake_fail_thread(k)
        if not {out}:
            ctx.set_field(F.RHO, rho)
        assert np.array_equal(ctx.get_field(F.RHO), rho)
        fake.fake_fail_thread(-1)
    """)


def test_failed_launch_leaves_no_copy_in_flight(fake):
    """A small copy of six arrays whose k-th launch fails: it returns the error
    when the ones before have ended, so that nothing writes the pinned block
    after another copy has taken it."""
    fake("""
    ctx = context(9, 9, 9)
    f = C.cast(getattr(ctx.L, "_ZN5fopis9host_copyEPKNS_7HostSegEibP12ihipStream_t"), C.c_void_p)
    dev = np.random.default_rng(2).standard_normal((6, 50))
    host = np.zeros_like(dev)
    seg = np.array([(h.ctypes.data, d.ctypes.data, d.nbytes) for h, d in zip(host, dev)], np.uint64)
    fake.fake_delay(20)
    for k in range(8):
        fake.fake_fail_launch(k)
        failed = fake.fake_copy(f, seg.ctypes.data_as(C.c_void_p), 6, 1)
        fake.fake_fail_launch(-1)
        assert failed == (k < 6) and fake.fake_pending() == 0
    assert np.array_equal(host, dev)
    """)


@pytest.mark.parametrize("bytes_", [8, 4096, 1 << 20, 8 << 20, 32 << 20])
@pytest.mark.parametrize("out", [0, 1])
def test_null_array_is_refused(fake, bytes_, out):
    """An array that is not there, alone or behind another one, is an error of
    the call at every size, as a plain copy's. (Pinned copies wrote to it.)"""
    fake(f"""
    ctx = context(9, 9, 9)
    f = C.cast(getattr(ctx.L, "_ZN5fopis9host_copyEPKNS_7HostSegEibP12ihipStream_t"), C.c_void_p)
    a, b = np.ones({bytes_}, np.uint8), np.zeros({bytes_}, np.uint8)
    for rows in ([(0, a)], [(b.ctypes.data, a), (0, a)]):
        seg = np.array([(h, d.ctypes.data, d.nbytes) for h, d in rows], np.uint64)
        assert fake.fake_copy(f, seg.ctypes.data_as(C.c_void_p), len(rows), {out}) == 1
    seg = np.array([(b.ctypes.data, a.ctypes.data, a.nbytes), (0, 0, 0)], np.uint64)  # an empty one may be null
    assert fake.fake_copy(f, seg.ctypes.data_as(C.c_void_p), 2, {out}) == 0
    """)


def test_pinned_block_follows_use(fake):
    """One read of a field pins little; 48 MB of reads pin the large block,
    once; the last context gives it back. Every way returns the bytes."""
    fake("""
    for dims in ((65, 65, 65), (81, 81, 81), (65, 65, 65)):
        ctx = context(*dims)
        rho = np.random.default_rng(1).standard_normal(ctx.field_shape(F.RHO))
        ctx.set_field(F.RHO, rho)
        log()
        for k in range(30):
            assert np.array_equal(ctx.get_field(F.RHO), rho)
            pins = [int(s.split()[1]) for s in log() if s.startswith("pin")]
            if k == 48 * 2**20 // rho.nbytes:
                assert len(pins) == 1 and pins[0] > 2**25
            else:
                assert sum(pins) <= (2**20 + 64 if k == 0 and rho.nbytes > 2**22 else 0)
        ctx.close()
    ctx = context(129, 129, 193)
    rho = np.zeros(ctx.field_shape(F.RHO))
    log()
    for k in range(3):  # 26 MB in: plain, then through the large block
        ctx.set_field(F.RHO, rho)
        lines = log()
        assert any("k_move" in s for s in lines) == (k > 0)
        assert sum(s.startswith("pin") for s in lines) == (k == 1)
    ctx.close()
    for dims in ((30, 257, 255), (97, 97, 97), (257, 129, 65), (257, 129, 225)):
        ctx = context(*dims)
        rho = np.random.default_rng(1).standard_normal(ctx.field_shape(F.RHO))
        ctx.set_field(F.RHO, rho)
        assert np.array_equal(ctx.get_field(F.RHO), rho)
        ctx.close()
    """)


def test_threads_start_on_an_idle_stream(fake):
    """A copy's threads start when the stream has done what came before."""
    fake("""
    ctx = context(81, 81, 81)
    fake.fake_delay(5)
    for k in range(20):
        log()
        fake.fake_busy()
        ctx.get_field(F.RHO)
        threads = [s for s in log() if s.startswith("thread")][k == 0:]  # the first one is the fake stream's
        assert threads and set(threads) == {"thread idle"}
    """)


def test_pinned_array_is_copied_directly(fake):
    """An array that the caller has pinned goes by one plain copy at every size.
    (It went through the library's own pinned memory, which takes longer.)"""
    fake("""
    ctx = context(9, 9, 9)
    f = C.cast(getattr(ctx.L, "_ZN5fopis9host_copyEPKNS_7HostSegEibP12ihipStream_t"), C.c_void_p)
    p = C.c_void_p()
    fake.hipHostMalloc.argtypes = [C.c_void_p, C.c_size_t, C.c_uint]
    fake.hipHostMalloc(C.byref(p), 64 << 20, 0)
    for n in (8, 4096, 3 << 20, 8 << 20, 60 << 20):
        for out in (0, 1):
            a = np.ones(n, np.uint8)
            seg = np.array([(p.value + 64, a.ctypes.data, n)], np.uint64)
            log()
            assert fake.fake_copy(f, seg.ctypes.data_as(C.c_void_p), 1, out) == 0
            assert log() == [f"memcpy {n}"]
    """)


def test_cmatrix_without_room_for_the_blocked_inversion(fake):
    """Any allocation of the blocked inversion fails: the elimination in place
    inverts, as it did where only it was there. (The call failed.)"""
    fake("""
    def build(k):
        ctx = context(17, 17, 17)
        mask = np.zeros((18, 18, 18), np.uint8)
        mask[8, 8, 8] = 1
        ctx.set_object(0, mask, np.array([(i, j, 8) for i in range(6, 11) for j in range(6, 11)], np.int32))
        log()
        fake.fake_fail_malloc(k)
        code = refused(ctx.build_cmatrix, 0)
        fake.fake_fail_malloc(-1)
        ctx.close()
        return code, log()

    code, clean = build(-1)
    assert code == 0 and not any("k_gj_elim" in s for s in clean)
    n = sum(s.startswith("malloc") for s in clean)
    for k in range(n - 5, n):  # W, F, V, the steps, the flag
        code, lines = build(k)
        assert code == 0 and any("k_gj_elim" in s for s in lines), (k, code)
        assert not any("k_bj" in s for s in lines)
    assert build(0)[0] == NOMEM
    """)


def test_whole_solve_graphs_are_made_for_use(fake):
    """A context's solves capture the graphs of a cycle and a pair once, and the
    whole solve's only for a number of cycles expected 16 times, once each; a
    solve of many launches a cycle (its coarsest level outside the tail) none.
    (The second solve of every context captured one, and each change another.)"""
    fake("""
    def made(ctx, solves):
        n = []
        for k in range(solves):
            log()
            ctx.solve_poisson()
            n.append(sum(s.startswith("instantiate") for s in log()))
        return n

    ctx = context(33, 33, 33)
    assert made(ctx, 18) == [2] + [0] * 17  # the first two expect one cycle
    assert made(ctx, 100) == [1] + [0] * 99
    n = 0
    for k in range(10):  # the expected number changes with every third solve
        for c in (6, 6, 6, 5, 5, 5):
            fake.fake_cycles(c)
            n += sum(made(ctx, 1))
    fake.fake_cycles(6)
    assert n + sum(made(ctx, 100)) == 1
    fake.fake_cycles(5)
    assert sum(made(ctx, 100)) == 0
    ctx.close()
    ctx = context(101, 101, 101)
    assert made(ctx, 100) == [2] + [0] * 99
    """)


def test_lds_grants_hold_per_device_and_context(fake):
    """A kernel's LDS beyond 64 KB is granted on the device it runs on, and a
    context with a smaller coarse tail takes none from an earlier one."""
    fake("""
    x, w = np.zeros((8, 8, 8, 64), np.uint16), np.zeros((27, 64, 64), np.float32)
    for device in (0, 1):
        fake.fake_set_device(device)
        G.conv3d(x, w, np.zeros(64, np.float32))
        G.conv3d_backward(x, w, x)
    ctxs = [context(*n, mg_precision=F.FP64) for n in ((17, 17, 17), (13, 13, 13), (11, 11, 11))]
    for c in ctxs:
        c.solve_poisson()
    """)


def test_initial_weights_of_a_seed(fake):
    """A new network's weights, drawn on the host, are the same for a seed from build to build."""
    fake("""
    import hashlib
    for seed, want in ((1, "841a4fca852919ddf61027e7cccc90e8"), (7, "1ef2ac797bdd072dc3e99739cc079aba"),
                       (12345678901, "bac7c9fefc400aedf4aad85c20e5dc22")):
        p = G.Guess(context(17, 17, 17), seed=seed).get_params()[0]
        assert hashlib.sha256(p.tobytes()).hexdigest()[:32] == want
    """)


def test_copy_threads_follow_the_cpu_quota(fake, tmp_path):
    """A control group's quota bounds a copy's threads, which spin while they
    wait: with fewer CPUs than threads they would be throttled. (Only the
    affinity set did.)"""
    cases = [("max 100000", None, 2**31 - 1), ("200000 100000", None, 2), ("150000 100000", None, 1), ("50000 100000", None, 1),
             ("1600000 100000", None, 16), (None, ("-1", "100000"), 2**31 - 1), (None, ("400000", "100000"), 4),
             (None, None, 2**31 - 1)]
    for k, (v2, v1, _) in enumerate(cases):
        d = tmp_path / str(k)
        (d / "cpu").mkdir(parents=True)
        if v2:
            (d / "cpu.max").write_text(v2 + "\n")
        if v1:
            (d / "cpu" / "cpu.cfs_quota_us").write_text(v1[0] + "\n")
            (d / "cpu" / "cpu.cfs_period_us").write_text(v1[1] + "\n")
    fake(f"""
    f = getattr(F.load(), "_ZN5fopis10quota_cpusEPKc")
    f.argtypes = [C.c_char_p]
    assert [f(b"{tmp_path}/%d" % k) for k in range({len(cases)})] == {[c[2] for c in cases]}
    """)
