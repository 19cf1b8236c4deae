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
