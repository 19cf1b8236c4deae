"""Calls that share a workspace from several streams and contexts, with the call that
needs no workspace in between, a context that moves to another workspace while its last
call runs, and the view table replaced behind a running call: every result is that of
the call alone, bit for bit."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from gtt import capi  # noqa: E402
from helpers import angles_full, geom  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nviews", [(12, 3), (40, 7), (72, 24)])
def test_shared_workspace_streams(n, nviews):
    g = geom(n, n, n, 2 * n, 2 * n - 3)
    angles = [angles_full(nviews, start=7.0 * i) for i in range(2)]
    print("CASE shared workspace", n, nviews, flush=True)
    rng = np.random.default_rng(n)
    vol = torch.from_numpy(rng.random(g.vol_shape).astype(np.float32)).cuda()
    want = []
    for a in angles:
        c = capi.Context(0)
        c.set_views(a)
        p = torch.zeros(g.proj_shape(nviews), device="cuda")
        x = torch.zeros_like(vol)
        c.fp(g, vol, p)
        c.bp(g, p, x)
        torch.cuda.synchronize()
        want.append((p, x))
        c.close()
    owner, a, b = capi.Context(0), capi.Context(0), capi.Context(0)
    streams = [torch.cuda.Stream() for _ in range(3)]
    a.set_views(angles[0])
    b.set_views(angles[1])
    got = []

    def pair(c, i, stream):
        p = torch.zeros(g.proj_shape(nviews), device="cuda")
        q, x = torch.zeros_like(p), torch.zeros_like(vol)
        torch.cuda.current_stream().synchronize()
        c.fp(g, vol, p, stream=stream)
        c.fp_noalloc(g, vol, q, stream=stream)
        c.bp(g, p, x, stream=stream)
        got.append((i, p, x, q))

    pair(a, 0, streams[0])            # in its own workspace,
    a.share_workspace(owner)          # then in another's
    b.share_workspace(owner)
    for r in range(4):
        pair(a, 0, streams[r % 3])
        pair(b, 1, streams[(r + 1) % 3])
    a.set_views(angles[1])            # waits for the calls that read the old table
    pair(a, 1, streams[1])
    owner.close()
    pair(b, 1, streams[2])
    a.close()
    pair(b, 1, streams[0])
    torch.cuda.synchronize()
    b.close()
    for i, p, x, q in got:
        assert torch.equal(p, want[i][0]) and torch.equal(q, want[i][0]) and torch.equal(x, want[i][1])
