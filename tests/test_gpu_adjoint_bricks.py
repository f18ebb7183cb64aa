"""The matched adjoint of tilted views where its bricks and batches of views have edges,
against the FP64 oracle's transpose: bricks of 8 (few of them) and of 16 with remainders,
64 views and one more, footprints cut by the detector, brick corners behind the source,
sub-rays.  The weights are the forward's FP32 crossing parameters: relative L2 <= 1e-5,
the bound of the other matched-adjoint tests.  Sums are integers: a repeated call gives
the same bits.
"""

from __future__ import annotations

import numpy as np
import pytest

from aprict_amd.cb import flatpanel as cbfp
from aprict_amd.volume import Volume
from helpers import chunk_for, random_geometry, rel_l2
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# shape, voxel width, views, nu, nv, pitch, sub-rays, source radius
CASES = {
    "one_small_brick": ((8, 8, 8), 1.0, 3, 20, 18, 1.0, 1, 60.0),
    "small_bricks_remainders": ((17, 9, 23), 0.7, 64, 24, 20, 1.6, 1, 60.0),
    "one_more_view": ((12, 20, 15), 0.8, 65, 22, 19, 1.7, 1, 60.0),
    "sub_rays": ((16, 15, 14), 0.8, 7, 15, 14, 2.4, 2, 60.0),
    "source_inside_the_box": ((24, 24, 24), 1.0, 6, 18, 18, 3.0, 1, 11.0),
    "large_bricks": ((81, 82, 90), 0.25, 5, 40, 44, 1.4, 1, 60.0),
    "large_bricks_two_batches": ((96, 81, 85), 0.25, 66, 14, 12, 3.5, 1, 60.0),
    "large_bricks_cut_footprints": ((85, 96, 81), 0.4, 4, 33, 29, 0.7, 1, 60.0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_tilted_adjoint_matches_oracle(device, name):
    import torch

    shape, w, views, nu, nv, pitch, ss, radius = CASES[name]
    rng = np.random.default_rng(len(name) + views)
    pg = random_geometry(rng, views, nu, nv, R=radius, L=2 * radius, pitch=pitch, tilt_deg=8.0, offset=1.0)
    y = torch.from_numpy(rng.uniform(-1, 2, (views, nu, nv)).astype(np.float32)).cuda()
    cfg = cbfp.ConfigProject(ssu=ss, ssv=ss)
    outs = []
    for _ in range(2):
        v = Volume(np.zeros(shape, np.float32), voxwid=w)
        cbfp.backproject_matched(cfg, v, cbfp.ProjectionSet(pg, data=y))
        outs.append(v.data.cpu().numpy())
    np.testing.assert_array_equal(outs[0], outs[1])
    want = orc.backproject_matched(cfg.contents, pg.to_proj_spec_array(), chunk_for(shape, w), np.zeros(shape),
                                   y.cpu().numpy())
    assert np.count_nonzero(want) > 0
    assert rel_l2(outs[0], want) <= 1e-5
