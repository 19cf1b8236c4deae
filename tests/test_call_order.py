"""What the host code waits for, allocates and refuses, on the CPU: the libraries run on
a HIP runtime that only keeps a log (fake_hip)."""
import pytest

import fake_hip


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    lib = fake_hip.build(tmp_path_factory.mktemp("hip"))
    return lambda script: fake_hip.run(lib, script)


@pytest.mark.parametrize("table", ["filter", "views"])
def test_tables_wait_for_calls_beside_noalloc(run, table):
    """A table is replaced after the call that reads it on one stream, although a
    cbct_fp_noalloc on another stream came in between (and after that one too)."""
    run(f"""
g = geom(16, 16, 16, 32, 24)
h = context(angles_full(6), filt=32)
for s in (S1, S2, S1):
    assert prefilter(h, g, 6, s) == 0
    assert fp_noalloc(h, g, 6, S3 if s == S1 else S1) == 0
    rc = set_filter(h, 32) if {table!r} == "filter" else views(h, angles_full(6, start=3.0))
    assert rc == 0
o = Order(log())
assert o.launches and all(not u for u in o.unwaited), [u for u in o.unwaited if u]
""")


def test_noalloc_makes_nothing(run):
    """cbct_fp_noalloc makes no event and takes no memory, also right after the context's
    other calls, and records none of its own while its stream is captured."""
    run("""
g = geom(16, 16, 16, 32, 24)
h = context(angles_full(6))
assert fp(h, g, 6, S1) == 0 and fp_noalloc(h, g, 6, S1) == 0 and bp(h, g, 6, S1) == 0
sim.hip_log_clear()
for s in (S1, S2, S1):
    assert fp(h, g, 6, S1) == 0 and fp_noalloc(h, g, 6, s) == 0 and bp(h, g, 6, S1) == 0
    assert fp_noalloc(h, g, 6, s) == 0
assert count("event_create") == count("event_destroy") == count("malloc") == count("host_malloc") == 0, log()
sim.hip_log_clear()
sim.hip_capture(S2, 1)
assert fp_noalloc(h, g, 6, S2) == 0
sim.hip_capture(S2, 0)
assert count("launch") and count("record") == 0
""")


@pytest.mark.parametrize("between", [False, True])
@pytest.mark.parametrize("table", ["filter", "views"])
def test_tables_wait_for_calls_in_the_workspace_before(run, table, between):
    """A table is replaced after the context's calls in the workspace that it had before
    the present one, whether or not another context has used that one since."""
    run(f"""
g = geom(16, 16, 16, 32, 24)
a, b, other = context(angles_full(6), filt=32), context(angles_full(6)), context()
assert L.cbct_ctx_share_workspace(b, a) == 0
sim.hip_log_clear()
assert prefilter(a, g, 6, S1) == 0
read = len(log())
if {between}:
    assert bp(b, g, 6, S2) == 0
assert L.cbct_ctx_share_workspace(a, other) == 0
assert fp(a, g, 6, S3) == 0
rc = set_filter(a, 32) if {table!r} == "filter" else views(a, angles_full(6, start=3.0))
assert rc == 0
o = Order(log())
late = [x for u in o.unwaited for x in u if x in log()[:read]]
assert o.unwaited and not late, late
# and the workspace's own last call is still waited for by its next one
assert fp(b, g, 6, S1) == 0
""")


SLAB = """
# most rays of the slab leave through its top or bottom: 30 views take them from the
# packed copy (four padded volumes), one view does not
g = geom(64, 64, 16, 48, 48)
CELLS = 4 * 67 * 67 * 32 * 4
def clip():
    n = sum("k_fp_clip" in l for l in log())
    sim.hip_log_clear()
    return n
h = context(angles_full(30))
live = lambda: ctypes.c_size_t.in_dll(sim, "hip_live").value
"""


def test_packed_copy_without_memory(run):
    """A packed copy that cannot be had is done without: no error, no further try until a
    trim."""
    run(SLAB + """
assert fp(h, g, 1, S1) == 0 and clip() == 0
limit(live() + CELLS - 1)
assert fp(h, g, 30, S1) == 0 and count("launch") and clip() == 0
assert L.cbct_last_error(h) == b""
assert fp(h, g, 30, S1) == 0 and count("malloc") == 0 and clip() == 0
limit(1 << 40)
assert fp(h, g, 30, S1) == 0 and count("malloc") == 0 and clip() == 0
assert L.cbct_ctx_trim(h) == 0 and fp(h, g, 30, S1) == 0 and clip() > 0
""")


def test_packed_copy_is_given_back(run):
    """Memory that a call needs takes the packed copy's place, once, after the call that
    used it."""
    run(SLAB + """
assert fp(h, g, 30, S1) == 0 and clip() > 0
limit(live() + 4096)
assert bp(h, g, 30, S2) == 0, L.cbct_last_error(h)
assert fp(h, g, 30, S1) == 0 and bp(h, g, 30, S1) == 0 and count("launch")
assert sum(l.startswith("malloc %d" % CELLS) for l in log()) == 0
sim.hip_log_clear()
assert fp(h, g, 30, S1) == 0 and bp(h, g, 30, S1) == 0 and count("malloc") == count("free") == 0
assert L.cbct_last_error(h) == b""
""")


def test_packed_copy_under_capture(run):
    """No memory is taken under capture, and what a captured call uses is not given back."""
    run(SLAB + """
assert fp(h, g, 1, S1) == 0
sim.hip_log_clear()
sim.hip_capture(S1, 1)
assert fp(h, g, 30, S1) == 0 and count("malloc") == 0 and count("launch") and clip() == 0
sim.hip_capture(S1, 0)
assert fp(h, g, 30, S1) == 0 and clip() > 0
sim.hip_capture(S1, 1)
assert fp(h, g, 30, S1) == 0 and count("malloc") == 0 and clip() > 0
sim.hip_capture(S1, 0)
limit(live() + 4096)
assert bp(h, g, 30, S1) == -4 and count("free") == 0
limit(1 << 40)
wide = geom(200, 200, 20, 16, 16)                    # sizes the padded copy alone
assert fp(h, wide, 1, S1) == 0 and clip() == 0
held = L.cbct_workspace_bytes(h)
assert fp(h, geom(80, 80, 20, 48, 48), 30, S1) == 0 and count("free") == 0 and clip() > 0
assert L.cbct_workspace_bytes(h) == held + 4 * 83 * 83 * 32 * 4
assert L.cbct_ctx_trim(h) == 0 and L.cbct_workspace_bytes(h) == 0
""")


SERVED = """
from gtt import serving as S
def request(kind, n, nz, nu, nv, views, offset=0.0, **more):
    g = geom(n, n, nz, nu, nv)
    off = np.tile(np.array([[0.0, offset]], np.float32), (views, 1))
    return S.Request(kind=kind, geom=g, angles=angles_full(views), offsets=off, subsets=5, iterations=1,
                     projections=np.zeros(g.proj_shape(views), np.float32), **more)
def base(r):     # without the packed copy
    g, v = r.geom, len(r.angles)
    nvox, nproj = g.nx * g.ny * g.nz, (g.nu + 3) * (g.nv + 3) * v
    blocks = -(-g.nx // 16) * -(-g.ny // 16) * -(-g.nz // 8)
    if r.kind == S.REQ_FDK:
        return 4 * (nvox * 23 // 10 + 8 * nproj) + 8 * blocks * v + (64 << 20)
    return 4 * (nvox * 83 // 10 + 4 * nproj + 4 * -(-nproj // 5)) + 8 * blocks * -(-v // 5) + (64 << 20)
def cells(r):
    g = r.geom
    return 4 * (g.nx + 3) * (g.ny + 3) * ((g.nz + 18) // 16 * 16) * (2 if r.storage == "bf16" else 4)
def serve(r, budget):
    sim.hip_log_clear()
    with S.Server(lanes=1, hbm_budget_bytes=budget) as srv:
        srv.wait(srv.submit(r))
    return sum("k_fp_clip" in l for l in log())
"""


def test_footprint_counts_the_packed_copy_where_it_is_built(run):
    """A request is charged for the projector's packed copy when a projection of it
    builds one: not for a few clipped rays, not above 4 GB, by storage type."""
    run(SERVED + """
for kind in (S.REQ_FDK, S.REQ_OS_SART):
    for storage in ("f32", "bf16"):
        few = request(kind, 96, 96, 48, 36, 10, 12.0, storage=storage)      # some rays clipped
        many = request(kind, 64, 16, 96, 96, 40, storage=storage)
        assert few.footprint() == base(few), (kind, storage)
        assert many.footprint() == base(many) + cells(many), (kind, storage)
        assert serve(few, 1 << 32) == 0 and serve(many, 1 << 32) > 0
    tall = request(kind, 900, 340, 2, 2000, 40)
    assert cells(tall) >= 1 << 32 and tall.footprint() == base(tall)
""")


def test_admission_does_not_depend_on_the_packed_copy(run):
    """A request that fits the budget without the packed copy is served without it."""
    run(SERVED + """
for kind in (S.REQ_FDK, S.REQ_OS_SART):
    r = request(kind, 64, 16, 96, 96, 40)
    assert serve(r, r.footprint()) > 0
    assert serve(r, r.footprint() - 1) == 0 and count("launch")
    assert serve(r, base(r)) == 0 and count("launch")
    with S.Server(lanes=1, hbm_budget_bytes=base(r) - 1) as srv:
        try:
            srv.submit(r)
            assert False
        except RuntimeError as e:
            assert "budget" in str(e)
    # the next request of the lane has it again
    with S.Server(lanes=1, hbm_budget_bytes=r.footprint() - 1) as srv:
        srv.wait(srv.submit(r))
        sim.hip_log_clear()
        small = request(kind, 48, 8, 96, 96, 20)
        assert small.footprint() < r.footprint() and small.footprint() > base(small)
        srv.wait(srv.submit(small))
        assert sum("k_fp_clip" in l for l in log()) > 0
""")


COPIES = """
import os, threading
from gtt import operators as ops
G = ops.load()
h2d, d2h, stream = G._ZN3gtt8copy_h2dEPvPKvm, G._ZN3gtt8copy_d2hEPvPKvm, G._ZN3gtt18set_current_streamEPv
trim, release = G._ZN3gtt18trim_thread_memoryEv, G._ZN3gtt24release_thread_resourcesEv
for f in (h2d, d2h):
    f.argtypes, f.restype = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t], None
for f in (stream, trim, release):
    f.argtypes, f.restype = [ctypes.c_void_p] if f is stream else [], None
MB = 1 << 20
def copies():      # (stream, thread) of each
    return [(int(l.split()[1], 0) if l.split()[1] != "(nil)" else 0, int(l.split()[4])) for l in log() if l.startswith("copy")]
"""


def test_host_copies_on_the_threads_own_default_stream(run):
    """hipStreamPerThread is another queue in every thread: the calling thread alone
    queues the copies."""
    run(COPIES + """
a, b = np.arange(32 * MB, dtype=np.uint8), np.zeros(32 * MB, np.uint8)
me = threading.get_native_id()
for s, alone in ((S1, False), (2, True)):
    stream(s)
    for f in (h2d, d2h):
        sim.hip_log_clear()
        b[:] = 0
        f(b.ctypes.data, a.ctypes.data, b.size)
        assert np.array_equal(a, b)
        assert {c[0] for c in copies()} == {s}
        assert ({c[1] for c in copies()} == {me}) or not alone
""")


def test_copies_back_wait_once(run):
    """A copy back to the host waits for the stream's earlier work on the calling thread,
    before any helper does: no helper waits for more than its own chunks."""
    run(COPIES + """
a, b = np.arange(32 * MB, dtype=np.uint8), np.zeros(32 * MB, np.uint8)
stream(S1)
sim.hip_log_clear()
d2h(b.ctypes.data, a.ctypes.data, b.size)
assert np.array_equal(a, b)
lines = [l.split() for l in log() if l.split()[0] in ("copy", "sync_stream", "sync_event")]
assert lines[0] == ["sync_stream", hex(S1), str(threading.get_native_id())], lines[0]
""")


def test_pinned_slots_are_kept_for_copies_at_once(run):
    """Slots are pinned for the copies that run at once, up to eight, and kept while the
    threads that copy are there; a thread's trim or end frees no others'."""
    run(COPIES + """
def work(n, gate, ok, done):
    a = np.arange(20 * MB, dtype=np.uint8)
    b = np.zeros_like(a)
    stream(S1)
    for r in range(6):
        gate.wait()
        d2h(b.ctypes.data, a.ctypes.data, b.size)
    ok.append(np.array_equal(a, b))
    gate.wait()      # the log is looked at
    gate.wait()
    release()
    done.wait()
for n in (1, 5, 12):
    sim.hip_log_clear()
    gate, done, ok = threading.Barrier(n + 1), threading.Barrier(n + 1), []
    ts = [threading.Thread(target=work, args=(n, gate, ok, done), daemon=True) for _ in range(n)]
    for t in ts:
        t.start()
    for r in range(6):
        gate.wait()
    gate.wait()
    assert len(ok) == n and all(ok)
    made = count("host_malloc")
    assert made <= min(n, 8) and count("host_free") == 0, (n, made, count("host_free"))
    trim()           # this thread copies nothing
    assert count("host_free") == 0
    gate.wait()
    done.wait()
    assert count("host_free") == made, (made, count("host_free"))
    for t in ts:
        t.join()
""")


def test_tuned_window_follows_the_offsets(run):
    """A tuned forward projector takes the z window that the views of the call need, not
    the one of the views it was tuned with; where no window of its tile holds them it
    takes what an untuned one takes."""
    run("""
import re
nviews, g = 5, geom(12, 12, 500, 14, 70, fov=(24.0, 90.0))
h = context()
def offsets(v):
    views(h, angles_full(nviews), np.stack([np.zeros(nviews), np.linspace(-v, v, nviews)], 1))
def kernel():     # (name, template arguments: rows and z per lane, steps in flight)
    sim.hip_log_clear()
    assert fp(h, g, nviews, S1) == 0
    m, = [m for m in (re.search("k_fp_colc?IfLi(.*?)EEEv", l) for l in log()) if m]
    return m.group(0), [int(x) for x in re.findall("[0-9]+", m.group(0).split("If", 1)[1])]
spans = (0.0, 20.0, 60.0, 150.0, 330.0, 0.0)
plain = []
for v in spans:
    offsets(v)
    plain.append((L.cbct_fp_kernel(h, ctypes.byref(g), 0, nviews, 0, 1.5), kernel()))
zc = [k[1][1][1] for k in plain[:4]]
assert zc == sorted(zc) and zc[0] < zc[-1] and plain[4][0] == b"k_fp_col", plain
for tune in range(4):
    L.cbct_fp_autotune_clear()
    offsets(spans[tune])
    best = ctypes.c_double()
    assert L.cbct_fp_autotune(h, ctypes.byref(g), 0, nviews, 0, 1.5, 0, S1, ctypes.byref(best)) == 0
    for v, p in zip(spans, plain):
        offsets(v)
        assert L.cbct_fp_kernel(h, ctypes.byref(g), 0, nviews, 0, 1.5) == p[0], (tune, v)
        k = kernel()
        assert k[0] == p[1][0] or k[1][0] != p[1][1][0], (tune, v, k, p)
""")


def test_backprojection_of_many_block_views(run):
    """A launch holds less than 2^32 work-items: block-views just below that and the
    padded copy's blocks are more together, but not each alone."""
    run("""
n = 65535
h = context(angles_full(n))
for g in (geom(512, 512, 1008, 1, 1), geom(512, 512, 1024, 1, 1)):
    sim.hip_log_clear()
    assert bp(h, g, n, S1) == 0, L.cbct_last_error(h)
    prep = [l.split() for l in log() if "k_bpp_prep" in l]
    blocks = 32 * 32 * (g.nz // 16)
    assert len(prep) == (1 if g.nz < 1024 else 2)
    assert sum(int(w[2]) for w in prep) == blocks * n // 256 + 16 * 1024 and "k_bpp" in log()[-2]
    assert L.cbct_ctx_trim(h) == 0
""")


def test_filter_waits_for_replays(run):
    """A filter is replaced in place, also where a captured call reads it: no event marks
    a replay's end, so the device is waited for then, and only then."""
    run("""
g = geom(16, 16, 16, 32, 24)
h = context(angles_full(6), filt=32)
assert prefilter(h, g, 6, S1) == 0 and set_filter(h, 32) == 0 and count("sync_device") == 0
assert prefilter(h, g, 6, S1) == 0
sim.hip_capture(S1, 1)
assert prefilter(h, g, 6, S1) == 0
sim.hip_capture(S1, 0)
for _ in range(2):
    sim.hip_log_clear()
    assert set_filter(h, 32) == 0
    first = [l.split()[0] for l in log() if l.split()[0] in ("sync_device", "copy")]
    assert first[0] == "sync_device", first
    # the tables made from it on the next call come after that
    sim.hip_log_clear()
    assert prefilter(h, g, 6, S1) == 0 and count("sync_device") == 0
assert L.cbct_ctx_reset(h) == 0 and set_filter(h, 32) == 0 and count("sync_device") == 0
""")
