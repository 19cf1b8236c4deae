"""LDS rows of the staged backprojector: scans of 1 to 2.8 detector texels per
voxel cross the lines between narrow rows, wide rows and no staging at all, with
single blocks that do not fit on either side of each.  Bit for bit the quad
engine's volumes, and within the single-pass bound (relative L2 of 1e-5) of the
FP64 oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle as O  # noqa: E402
from gtt import capi  # noqa: E402
from helpers import angles_full, geom, rel_l2, to_oracle  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("nu", [50, 90, 97, 103, 110, 117, 126, 140])
def test_bp_rows(ctx, nu, dtype):
    n, nviews = 50, 9
    g = geom(n, n - 3, n + 5, nu, (3 * nu) // 4 + 1)
    angles = angles_full(nviews, start=3.0)
    offsets = np.tile(np.array([[0.7, -0.4]], np.float32), (nviews, 1))
    print("CASE bp rows", nu, dtype, flush=True)
    p = np.random.default_rng(nu).random(g.proj_shape(nviews)).astype(np.float32)
    pd = torch.from_numpy(p).cuda()
    if dtype == "bf16":
        pd = pd.to(torch.bfloat16)
    ctx.set_views(angles, offsets)
    try:
        for kz in (8, 16):
            ctx.bp_kz(kz)
            for fbp in (False, True):
                outs = []
                for e in (1, 2, 3):
                    ctx.bp_engine(e)
                    outs.append(ctx.bp(g, pd, torch.empty(g.vol_shape, device="cuda"), fbp=fbp))
                assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2]), (kz, fbp)
    finally:
        ctx.bp_engine(2)
        ctx.bp_kz(0)
    ref = O.bp(to_oracle(g), angles, offsets, pd.double().cpu().numpy(), fbp=True)
    assert rel_l2(outs[0].cpu().numpy(), ref) <= 1e-5
