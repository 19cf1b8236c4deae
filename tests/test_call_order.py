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
