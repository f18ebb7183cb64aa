"""The analytic projector where a workgroup takes several tiles: the number per workgroup
grows with the tiles of the call (a 4096th of them, 32 at most), so a call of many views is
compared, bit for bit, with its views projected one at a time, a tile per workgroup, and
some of those with the FP64 oracle.  The object covers the middle of the detector, so that
tiles without shapes lie between others.
"""

from __future__ import annotations

import numpy as np
import pytest

from aprict_amd import phantoms as ph
from aprict_amd.cb import flatpanel as cbfp
from aprict_amd.volume import FBVolume, forbild
from helpers import rel_l2
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _shapes(rng, count):
    out = []
    for i in range(count):
        q, _ = np.linalg.qr(rng.standard_normal((3, 3)))
        cen, size = rng.uniform(-9, 9, 3), rng.uniform(0.5, 5.0, 3)
        rho = float(rng.uniform(-0.5, 1.0))
        if i % 3 == 0:
            out.append(forbild.ellipsoid_free(cen, size, q, rho))
        elif i % 3 == 1:
            out.append(forbild.ellipt_cyl(cen, size[0], size[1], 2 * size[2], q[0], q[1], q[2], rho))
        else:
            out.append(forbild.box(cen, *(2 * size), rho))
    return forbild.stack(out)


def _project(pg, shapes, cfg, start, views=None):
    import torch

    if views is not None:
        pg = cbfp.ProjGeom(source_pos=pg.source_pos[views], det_pos=pg.det_pos[views], det_uvec=pg.det_uvec[views],
                           det_vvec=np.broadcast_to(pg.det_vvec, pg.det_uvec.shape)[views].copy(), nu=pg.nu, nv=pg.nv)
        start = start[views]
    ps = cbfp.ProjectionSet(pg, data=torch.from_numpy(start).cuda())
    cbfp.project(cfg, FBVolume(shapes), ps, block=True)
    return pg, ps.data.cpu().numpy()


# views, nu, nv (tiles of 16 x 16 pixels, tiles per workgroup, tiles of the last one), shapes, sub-rays
CASES = {
    "three_tiles": (90, 200, 200, 12, 1),       # 169, 3, 1
    "four_tiles": (110, 190, 200, 64, 1),       # 156, 4, 4
    "shape_batches": (70, 200, 195, 70, 1),     # 169, 2, 1
    "shape_batches_sub_rays": (64, 180, 190, 130, 2),   # 144, 2, 2
    "most_tiles": (320, 335, 330, 7, 1),        # 441, 32, 25
}


@pytest.mark.parametrize("name", list(CASES))
def test_several_tiles_per_workgroup(device, name):
    views, nu, nv, count, ss = CASES[name]
    tiles = -(-nu // 16) * -(-nv // 16)
    assert tiles * views // 4096 >= 2
    rng = np.random.default_rng(count)
    shapes = _shapes(rng, count)
    pg = ph.circular_geometry(views, nu, nv, 90.0 / nu, R=60.0, L=120.0)
    cfg = cbfp.ConfigProject(ssu=ss, ssv=ss)
    start = rng.uniform(0.0, 1.0, (views, nu, nv)).astype(np.float32)
    _, got = _project(pg, shapes, cfg, start)
    for p in (0, views // 3, views - 1):
        one, alone = _project(pg, shapes, cfg, start, [p])
        np.testing.assert_array_equal(got[p:p + 1], alone)
        if nu <= 200:
            want = orc.project_forbild(cfg.contents_fb, one.to_proj_spec_array(), shapes, np.zeros((1, nu, nv)))
            touched = np.count_nonzero(want)
            assert 0 < touched < 0.9 * want.size
            assert rel_l2(alone, want + start[p:p + 1]) <= 1e-6
