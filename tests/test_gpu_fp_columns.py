"""Column forward projector at the edges of its own splits, against the
per-ray engine (bit for bit) and the FP64 oracle (relative L2 of 1e-5, the
single-pass bound of the other parity tests).

Clipped rays: rays leaving through the top or bottom are taken 8 samples x 8
rays at a time, so sample counts off the multiples of 8, row blocks with a few
clipped rays, blocks of 64 rows that end ragged, and odd z for the BF16 pairs
are where it can go wrong.

Cached z windows: 64 to 384 z in pieces of several widths, chosen by the z
range that a row group's rays cross; volume heights on both sides of every
width, ragged row counts and up to 12 rows per lane."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle as O  # noqa: E402
from gtt import capi  # noqa: E402
from helpers import angles_full, geom, phantom_volume, rel_l2, to_oracle  # noqa: E402

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def project(ctx, g, vol, nviews, engine):
    out = torch.zeros(g.proj_shape(nviews), device="cuda")
    ctx.fp_engine(engine)
    ctx.fp(g, vol, out)
    ctx.fp_engine(1)
    torch.cuda.synchronize()
    return out


# (nx, ny, nz, nu, nv, detector height in mm, v offset in mm)
CLIPPED = [(17, 17, 3, 9, 63, 40.0, 0.0), (17, 13, 8, 11, 65, 25.0, 3.0), (5, 5, 4, 6, 200, 9.0, 0.0),
           (31, 29, 11, 7, 129, 19.0, -2.5), (1, 1, 1, 5, 64, 6.0, 0.4), (40, 40, 21, 9, 70, 33.0, 0.0)]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("case", CLIPPED)
def test_clipped_rays(ctx, case, dtype):
    nx, ny, nz, nu, nv, fv, ov = case
    g = geom(nx, ny, nz, nu, nv, fov=(2.0 * nx, fv))
    angles = angles_full(5)
    offsets = np.tile(np.array([[0.3, ov]], np.float32), (5, 1))
    print("CASE clipped", case, dtype, flush=True)
    vol = phantom_volume(g) + 0.05 * np.random.default_rng(3).random((nz, ny, nx))
    v = torch.from_numpy(vol.astype(np.float32)).cuda()
    if dtype == "bf16":
        v = v.to(torch.bfloat16)
    ctx.set_views(angles, offsets)
    a, b = project(ctx, g, v, 5, 0), project(ctx, g, v, 5, 1)
    assert torch.equal(a, b)
    # without memory of its own the call takes them from the plain copy
    c = torch.zeros_like(a)
    ctx.fp_noalloc(g, v, c)
    assert torch.equal(a, c)
    ctx.fp(g, v, c, accumulate=True)
    assert torch.equal(a + a, c)
    ref = O.fp(to_oracle(g), angles, offsets, v.double().cpu().numpy())
    assert rel_l2(b.cpu().numpy(), ref) <= TOL


# (nz, nv): the window grows with nz; 12 rows per lane at most
WINDOWS = [(1, 1), (50, 64), (57, 65), (60, 130), (118, 129), (122, 300), (180, 257), (186, 383), (245, 320),
           (251, 449), (310, 512), (314, 577), (372, 700), (378, 768), (420, 768)]


# launches of 8192 waves (detector columns x row groups x views) and more leave
# the variant that keeps several steps in flight; the last one is just below
MANY = [(1, 1, 70, 118), (50, 64, 64, 128), (118, 129, 70, 120), (60, 130, 66, 125), (122, 240, 127, 64)]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("case", [w + (6, 7) for w in WINDOWS] + MANY)
def test_z_windows(ctx, case, dtype):
    nz, nv, nu, nviews = case
    # magnification 1.5: the detector sees the whole height and no more, so the
    # rays cross the window's whole width
    g = geom(9, 7, nz, nu, nv, fov=(20.0, 1.48 * nz))
    angles = angles_full(nviews)
    offsets = np.tile(np.array([[0.2, 0.3]], np.float32), (nviews, 1))
    print("CASE window", case, dtype, flush=True)
    vol = np.random.default_rng(nz).random((nz, 7, 9)) + 0.1
    v = torch.from_numpy(vol.astype(np.float32)).cuda()
    if dtype == "bf16":
        v = v.to(torch.bfloat16)
    ctx.set_views(angles, offsets)
    a, b = project(ctx, g, v, nviews, 0), project(ctx, g, v, nviews, 1)
    assert torch.equal(a, b)
    ref = O.fp(to_oracle(g), angles, offsets, v.double().cpu().numpy())
    assert rel_l2(b.cpu().numpy(), ref) <= TOL
