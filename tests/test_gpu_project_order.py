"""The forward projectors where their block orders have remainders: views beyond whole
groups of 8, a last row block of one row or of all but one, single columns and views;
for tilted panels also 32 rows of two columns per wave.  A sample's sum does not depend
on the block it is computed in: every launch shape, and each view projected alone, gives
the same bits.  Tilted panels are also compared with the FP64 oracle, relative L2 <= 1e-5
as in the other forward tests.
"""

from __future__ import annotations

import numpy as np
import pytest

from aprict_amd import _abi, autotune
from aprict_amd import phantoms as ph
from aprict_amd.cb import flatpanel as cbfp
from aprict_amd.volume import Volume
from helpers import chunk_for, random_geometry, rel_l2
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _project(pg, vol):
    ps = cbfp.ProjectionSet(pg)
    cbfp.project(cbfp.ConfigProject(), vol, ps, block=True)
    return ps.data.cpu().numpy()


@pytest.mark.parametrize(("views", "nu", "nv"), [(1, 1, 1), (9, 3, 129), (7, 5, 127), (8, 1, 257), (17, 6, 64)])
def test_every_block_of_the_order(device, views, nu, nv):
    rng = np.random.default_rng(views + nu + nv)
    vol = Volume(rng.uniform(0.5, 1.0, (15, 14, 60)).astype(np.float32), voxwid=0.5)
    pg = ph.circular_geometry(views, nu, nv, min(0.6, 48.0 / nv), R=60.0, L=120.0)
    op = _abi.TUNE_PROJECT_COLUMN
    try:
        got = []
        for var in range(autotune.variant_count(op)):
            autotune.set_variant(op, var)
            got.append(_project(pg, vol))
    finally:
        autotune.set_variant(op, 0)
    assert np.count_nonzero(got[0]) > 0.5 * got[0].size
    for g in got[1:]:
        np.testing.assert_array_equal(g, got[0])
    v = np.broadcast_to(pg.det_vvec, (views, 3))
    for p in range(views):
        one = cbfp.ProjGeom(source_pos=pg.source_pos[p:p + 1], det_pos=pg.det_pos[p:p + 1],
                            det_uvec=pg.det_uvec[p:p + 1], det_vvec=v[p:p + 1].copy(), nu=nu, nv=nv)
        np.testing.assert_array_equal(_project(one, vol)[0], got[0][p])


@pytest.mark.parametrize("ss", [1, 2])
@pytest.mark.parametrize(("views", "nu", "nv"), [(1, 1, 1), (9, 5, 96), (3, 17, 129), (2, 7, 160), (2, 9, 65), (5, 8, 64)])
def test_every_tile_of_tilted_panels(device, views, nu, nv, ss):
    rng = np.random.default_rng(views + nu + nv)
    shape, w = (15, 14, 40), 0.6
    x = rng.uniform(0.5, 1.0, shape).astype(np.float32)
    vol = Volume(x, voxwid=w)
    pg = random_geometry(rng, views, nu, nv, pitch=min(0.6, 40.0 / nv))
    cfg = cbfp.ConfigProject(ssu=ss, ssv=ss)
    op = _abi.TUNE_PROJECT_RAY
    got = []
    try:
        for var in range(autotune.variant_count(op)):
            autotune.set_variant(op, var)
            ps = cbfp.ProjectionSet(pg)
            cbfp.project(cfg, vol, ps, block=True)
            got.append(ps.data.cpu().numpy())
    finally:
        autotune.set_variant(op, 0)
    for g in got[1:]:
        np.testing.assert_array_equal(g, got[0])
    want = orc.project_voxel(cfg.contents, pg.to_proj_spec_array(), chunk_for(shape, w), x, np.zeros((views, nu, nv)))
    assert np.count_nonzero(want)
    assert rel_l2(got[0], want) <= 1e-5
