"""TV step at the edges of its tiles (64 x by 2 rows per wave, 4 waves, slices
in chunks) and of its division's range, against the FP64 oracle.  The bound is
the one of the other TV tests (relative L2 of 1e-6)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle as O  # noqa: E402
from gtt import capi  # noqa: E402
from helpers import rel_l2  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


# (nz, ny, nx) or (nvol, nz, ny, nx)
SHAPES = [(1, 1, 1), (2, 1, 64), (1, 2, 65), (3, 3, 63), (5, 8, 130), (4, 9, 1), (33, 7, 66), (2, 3, 17, 129),
          (200, 2, 3), (70, 65, 64)]


@pytest.mark.parametrize("scale", [1.0, 1e12, 1e17, 1e-30])
@pytest.mark.parametrize("shape", SHAPES)
def test_tv_tiles(ctx, shape, scale):
    """scale 1e12: norms far above one; 1e17: their squares near the largest
    float; 1e-30: gradients far below one, passed through."""
    print("CASE tv", shape, scale, flush=True)
    rng = np.random.default_rng(abs(hash(shape)) % 1000)
    x = (rng.random(shape) * scale).astype(np.float32)
    xd = torch.from_numpy(x).cuda()
    out = torch.full_like(xd, 7.0)
    ctx.tv_primal_dual(xd, out, 3.0, 0.0, 1.0, accumulate=False)
    ref = np.zeros(shape)
    O.tv_primal_dual(x.astype(np.float64), ref, 3.0, 0.0, 1.0)
    assert rel_l2(out.cpu().numpy(), ref) <= 1e-6


def test_tv_nonfinite_stays_local(ctx):
    """An infinite voxel reaches only the voxels whose gradients read it."""
    x = np.random.default_rng(4).random((6, 6, 70)).astype(np.float32)
    x[2, 3, 64] = np.inf
    out = torch.zeros((6, 6, 70), device="cuda")
    ctx.tv_primal_dual(torch.from_numpy(x).cuda(), out, 3.0, 0.0, 1.0, accumulate=False)
    got = np.argwhere(~np.isfinite(out.cpu().numpy()))
    assert len(got) and np.abs(got - [2, 3, 64]).max() <= 1


@pytest.mark.parametrize("scale", [1.0, 1e12])
@pytest.mark.parametrize("shape", SHAPES)
def test_tv_update_tiles(ctx, shape, scale):
    """The fused update at the same edges: bit for bit the TV gradient added to zeros and
    then updateG, and within the bound of the FP64 oracle; accumulation likewise."""
    print("CASE tv update", shape, scale, flush=True)
    rng = np.random.default_rng(sum(shape))
    x, s, P, out0 = [(rng.random(shape) * k + o).astype(np.float32) for k, o in ((scale, 0), (1, 0), (1, 0.5), (1, 0))]
    xd, sd, Pd, od = [torch.from_numpy(a).cuda() for a in (x, s, P, out0)]
    g, xf, xu = torch.zeros_like(xd), torch.empty_like(xd), xd.clone()
    ctx.tv_primal_dual(xd, g, 3.0, 0.0, 1.0, accumulate=True)
    ctx.update_g(g, xu, sd, Pd, 0.05, 1e-3)
    ctx.tv_update_g(xd, xf, sd, Pd, 3.0, 0.0, 1.0, 0.05, 1e-3)
    assert torch.equal(xf, xu)
    ctx.tv_primal_dual(xd, od, 3.0, 0.0, 1.0, accumulate=True)
    d = lambda a: a.astype(np.float64)
    gref, oref = np.zeros(shape), d(out0)
    O.tv_primal_dual(d(x), gref, 3.0, 0.0, 1.0)
    O.tv_primal_dual(d(x), oref, 3.0, 0.0, 1.0, accumulate=True)
    assert rel_l2(od.cpu().numpy(), oref) <= 1e-6
    assert rel_l2(xf.cpu().numpy(), O.update_g(gref, d(x), d(s), d(P), 0.05, 1e-3)) <= 1e-6


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_tv_nonfinite_values(ctx, bad):
    """Every voxel beside non-finite ones against the two passes in plain FP32.  Projected
    gradients are at most 1; each may differ by two last bits (2.4e-7), six of them and
    five roundings of their sum (up to 2.4e-7 each) make 2.7e-6."""
    print("CASE tv non-finite", bad, flush=True)
    x = np.random.default_rng(6).random((5, 6, 70)).astype(np.float32)
    for at in ((2, 3, 64), (0, 0, 0), (4, 5, 69), (3, 1, 10), (3, 1, 11)):
        x[at] = bad
    t = torch.from_numpy(x)
    p = [(torch.roll(t, -1, d) - t) * 3.0 for d in (2, 1, 0)]
    den = torch.fmax(torch.ones(()), torch.sqrt(p[0] * p[0] + p[1] * p[1] + p[2] * p[2]))
    want = torch.zeros_like(t)
    for q, d in zip(p, (2, 1, 0)):
        want += torch.roll(q / den, 1, d) - q / den
    out = torch.zeros(t.shape, device="cuda")
    ctx.tv_primal_dual(t.cuda(), out, 3.0, 0.0, 1.0, accumulate=False)
    assert torch.allclose(out.cpu(), want, rtol=0.0, atol=2.7e-6, equal_nan=True)
