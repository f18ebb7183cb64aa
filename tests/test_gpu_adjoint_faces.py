"""The upright-view matched adjoint (face sums) at the sizes where its tiling,
its rows and its view slices change, against the FP64 oracle's transpose.

Tiles are 8 x 8 cells and 64 to 256 planes; views are split between workgroups
when there are few tiles and at least 16 views; a detector column's rows are kept
apart at the source height, where an odd row count puts a horizontal or nearly
horizontal ray.  (Column counts are even: the middle column of an odd count runs
within a grid plane in some views, where rounding alone says on which side.)  The weights are the forward's FP32 crossing parameters: relative
L2 <= 1e-5, the bound of the other matched-adjoint tests.  Sums are FP64 in a fixed
order: a repeated call gives the same bits.
"""

from __future__ import annotations

import numpy as np
import pytest

from aprict_amd import phantoms as ph
from aprict_amd.cb import flatpanel as cbfp
from aprict_amd.volume import Volume
from helpers import chunk_for, rel_l2
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# shape, voxel width, views, nu, nv, source heights (first, last), sub-samples
CASES = {
    "one_plane": ((8, 8, 1), 0.5, 5, 18, 9, (0.0, 0.0), 1),
    "horizontal_ray_in_a_plane": ((9, 8, 64), 0.5, 6, 20, 41, (0.0, 0.0), 1),
    "horizontal_ray_off_planes": ((9, 8, 63), 0.5, 6, 20, 41, (0.0, 0.0), 1),
    "helical_odd_rows": ((17, 16, 65), 0.37, 20, 30, 37, (-9.1, 8.3), 1),
    "two_waves": ((16, 17, 128), 0.23, 18, 28, 33, (-3.0, 3.0), 1),
    "three_waves": ((7, 25, 129), 0.21, 17, 34, 45, (-14.0, 14.0), 1),
    "four_waves": ((8, 9, 193), 0.17, 16, 26, 49, (-2.0, 20.0), 1),
    "two_layers": ((10, 9, 257), 0.13, 9, 22, 43, (-20.0, 4.0), 1),
    "source_above": ((12, 11, 40), 0.4, 16, 24, 31, (10.0, 10.0), 1),
    "fine_subsampled": ((11, 10, 30), 0.5, 16, 90, 70, (-1.0, 1.0), 3),
    "many_views_few_tiles": ((8, 8, 20), 0.6, 150, 16, 17, (0.0, 0.0), 1),
}


@pytest.mark.parametrize("sino_dtype", ["float32", "float16"])
@pytest.mark.parametrize("name", list(CASES))
def test_upright_adjoint_matches_oracle(device, name, sino_dtype):
    import torch

    shape, w, views, nu, nv, lift, ss = CASES[name]
    rng = np.random.default_rng(len(name))
    pitch = 0.35 if ss > 1 else 1.0
    pg = ph.circular_geometry(views, nu, nv, pitch, R=40.0, L=80.0)
    dz = np.linspace(lift[0], lift[1], views)[:, None] * [0, 0, 1]
    pg = cbfp.ProjGeom(source_pos=pg.source_pos + dz, det_pos=pg.det_pos + dz, det_uvec=pg.det_uvec,
                       det_vvec=np.broadcast_to(pg.det_vvec, pg.det_uvec.shape).copy(), nu=nu, nv=nv)
    y = torch.from_numpy(rng.uniform(-1, 2, (views, nu, nv)).astype(np.float32)).cuda()
    if sino_dtype == "float16":
        y = y.to(torch.float16)
    cfg = cbfp.ConfigProject(ssu=ss, ssv=ss)
    outs = []
    for _ in range(2):
        v = Volume(np.zeros(shape, np.float32), voxwid=w)
        cbfp.backproject_matched(cfg, v, cbfp.ProjectionSet(pg, data=y), block=True)
        outs.append(v.data.clone())
    assert torch.equal(outs[0], outs[1])
    want = orc.backproject_matched(cfg.contents, pg.to_proj_spec_array(), chunk_for(shape, w), np.zeros(shape),
                                   y.float().cpu().numpy())
    err = rel_l2(outs[0].cpu().numpy(), want)
    print(f"upright adjoint [{name}, {sino_dtype}]: rel L2 {err:.3e}")
    assert np.abs(want).max() > 0 and err <= 1e-5
