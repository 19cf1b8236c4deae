"""Short-scan weights of the FFT pre-filter, which a thread keeps per view while its
workgroup goes through consecutive row groups: rows per view that fill the groups,
nearly fill them and do not (groups then span views), fewer rows than a group, one
row, a sub-range of the views, and more groups than workgroups.  Within the
single-pass bound (relative L2 of 1e-5) of the FP64 oracle, in place as well."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle as O  # noqa: E402
from gtt import capi  # noqa: E402
from helpers import angles_full, geom, rel_l2, to_oracle  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nu,nv,nviews", [
    (32, 64, 12), (32, 61, 12), (32, 40, 12), (31, 3, 70), (64, 32, 9), (100, 15, 7), (100, 13, 7),
    (300, 1, 1), (500, 8, 5), (500, 7, 5), (1024, 9, 4), (1024, 7, 4), (2000, 16, 150)])
def test_short_scan_filter(nu, nv, nviews):
    g = geom(8, 8, 8, nu, nv, fov=(400.0, 300.0))
    angles = angles_full(nviews + 2, 200.0)
    print("CASE short-scan filter", nu, nv, nviews, flush=True)
    proj = np.random.default_rng(nu + nv).random((nviews, nv, nu)).astype(np.float32)
    F = O.ramlak_filter(nu).astype(np.float32)
    ref = O.fdk_prefilter(to_oracle(g), angles[1:nviews + 1], np.zeros((nviews, 2), np.float32), proj, F,
                          short_scan=True, offset_correct=False)
    ctx = capi.Context(0)
    try:
        ctx.set_views(angles)
        ctx.set_filter(F)
        ctx.filter_engine(2)
        pin = torch.from_numpy(proj).cuda()
        out = torch.full_like(pin, float("nan"))
        ctx.fdk_prefilter(g, pin, out, view0=1, nviews=nviews, short_scan=True)
        ctx.fdk_prefilter(g, pin, pin, view0=1, nviews=nviews, short_scan=True)
        assert rel_l2(out.cpu().numpy(), ref) <= 1e-5
        assert torch.equal(out, pin)
    finally:
        ctx.close()
