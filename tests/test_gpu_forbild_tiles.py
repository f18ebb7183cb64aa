"""The analytic projector where its tiles, shape batches and culls have edges, against
the FP64 oracle: detectors around whole tiles of 16 x 16 pixels (8 x 8 per wave), one
shape, a whole batch of 64 and one more, sub-rays, clip planes, cones, degenerate sizes,
and panels so close that a tile's rays fan out beyond what the cone test takes.

Both sides are FP64, with roots off by about 1e-10 for a source some 100 radii away:
relative L2 <= 1e-7 in an F64 sinogram, 1e-6 in F32, whose rounding is 6e-8.  A shape
that a tile wrongly leaves out would show as 1e-3 and more.
"""

from __future__ import annotations

import numpy as np
import pytest

from aprict_amd import phantoms as ph
from aprict_amd.cb import flatpanel as cbfp
from aprict_amd.volume import FBVolume, forbild
from helpers import random_geometry, rel_l2
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _shapes(rng, count, span=12.0):
    out = []
    for i in range(count):
        q, _ = np.linalg.qr(rng.standard_normal((3, 3)))
        cen, size = rng.uniform(-span, span, 3), rng.uniform(0.4, 6.0, 3)
        clips = []
        for _ in range(int(rng.integers(0, 4))):
            n = rng.standard_normal(3)
            n = (n / np.linalg.norm(n)).astype(np.float32)
            clips.append((n, np.float32(n @ cen + rng.uniform(-0.5, 0.5) * size.mean()), int(rng.integers(1, 3))))
        rho = float(rng.uniform(-0.5, 1.0))
        kind = i % 5
        if kind == 0:
            out.append(forbild.ellipsoid_free(cen, size, q, rho, clips=clips))
        elif kind == 1:
            out.append(forbild.ellipt_cyl(cen, size[0], size[1], 2 * size[2], q[0], q[1], q[2], rho, clips=clips))
        elif kind == 2:
            out.append(forbild.box(cen, *(2 * size), rho, clips=clips))
        elif kind == 3:
            out.append(forbild.cone(cen, size[0], 0.3 * size[1], 2 * size[2], q[2], rho, clips=clips))
        else:
            out.append(forbild.cylinder(cen, 0.2 * size[0], 4 * size[1], q[0], rho, clips=clips))
    return forbild.stack(out)


# views, nu, nv, shapes, sub-rays, geometry
CASES = {
    "one_pixel": (2, 1, 1, 3, 1, "circular"),
    "below_a_tile": (3, 15, 7, 1, 1, "circular"),
    "whole_tiles": (4, 32, 16, 20, 1, "tilted"),
    "one_more_pixel": (3, 17, 33, 20, 1, "tilted"),
    "whole_batch": (2, 40, 41, 64, 1, "tilted"),
    "two_batches": (2, 40, 41, 65, 1, "circular"),
    "three_batches_sub_rays": (2, 19, 23, 130, 2, "tilted"),
    "sub_rays": (3, 21, 24, 30, 3, "circular"),
    "close_panel": (4, 24, 24, 30, 1, "close"),
    "many_tiles_per_workgroup": (24, 150, 140, 12, 1, "circular"),
}


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("name", list(CASES))
def test_tiles_match_oracle(device, name, dtype):
    import torch

    views, nu, nv, count, ss, geom = CASES[name]
    rng = np.random.default_rng(len(name) + count)
    shapes = _shapes(rng, count)
    if geom == "circular":
        pg = ph.circular_geometry(views, nu, nv, 80.0 / max(nu, nv), R=60.0, L=120.0)
    elif geom == "tilted":
        pg = random_geometry(rng, views, nu, nv, pitch=80.0 / max(nu, nv), tilt_deg=20.0)
    else:   # a source 16 from the centre, pixels of 4 at a distance of 20
        pg = random_geometry(rng, views, nu, nv, R=16.0, L=20.0, pitch=4.0, tilt_deg=20.0, offset=1.0)
    cfg = cbfp.ConfigProject(ssu=ss, ssv=ss)
    start = rng.uniform(0.0, 1.0, (views, nu, nv)).astype(np.float32)
    ps = cbfp.ProjectionSet(pg, data=torch.from_numpy(start).cuda().to(getattr(torch, dtype)))
    cbfp.project(cfg, FBVolume(shapes), ps, block=True)
    got = ps.data.cpu().numpy().astype(np.float64) - start
    want = orc.project_forbild(cfg.contents_fb, pg.to_proj_spec_array(), shapes, np.zeros((views, nu, nv)))
    assert np.count_nonzero(want) or name == "one_pixel"
    bound = 1e-6 if dtype == "float32" else 1e-7
    scale = max(float(np.abs(want).max()), 1.0)
    assert rel_l2(got + start, want + start) <= bound
    np.testing.assert_allclose(got, want, rtol=0, atol=20 * bound * scale)


@pytest.mark.parametrize("count", [8, 9, 63, 64, 65, 80])
def test_rays_through_many_separate_pieces(device, count):
    # slabs one behind the other: rays along x are covered in `count` separate pieces (8
    # are kept in registers, 64 in memory; more are recomputed)
    x = np.linspace(-10.0, 10.0, count)
    gap = 20.0 / count
    shapes = forbild.stack([forbild.box((x[(7 * i) % count if count % 7 else i], 0.0, 0.0), 0.6 * gap, 14.0, 14.0,
                                        0.1 + 0.01 * i) for i in range(count)])
    pg = ph.circular_geometry(4, 22, 18, 1.5, R=60.0, L=120.0)
    cfg = cbfp.ConfigProject()
    ps = cbfp.ProjectionSet(pg)
    cbfp.project(cfg, FBVolume(shapes), ps, block=True)
    got = ps.data.cpu().numpy()
    want = orc.project_forbild(cfg.contents_fb, pg.to_proj_spec_array(), shapes, np.zeros((4, 22, 18)))
    assert np.count_nonzero(want) > 0.2 * want.size
    assert rel_l2(got, want) <= 1e-6
    np.testing.assert_allclose(got, want, rtol=0, atol=2e-5 * float(want.max()))
