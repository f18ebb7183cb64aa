"""The upright-view matched adjoint where the sums of its gather can go wrong, against
the FP64 oracle's transpose: dim detector rows beside bright ones seen from 1000 voxels
away, and views split between workgroups on tiles of every height, with a short last
slice and on a part of the volume.
"""

from __future__ import annotations

import numpy as np
import pytest

from aprict_amd import _abi
from aprict_amd import phantoms as ph
from aprict_amd.cb import flatpanel as cbfp
from aprict_amd.volume import Volume
from helpers import chunk_for, rel_l2
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _adjoint(pg, shape, w, y):
    import torch

    cfg = cbfp.ConfigProject()
    v = Volume(np.zeros(shape, np.float32), voxwid=w)
    cbfp.backproject_matched(cfg, v, cbfp.ProjectionSet(pg, data=torch.from_numpy(y).cuda()), block=True)
    return v.as_numpy().astype(np.float64)


def _oracle(pg, shape, w, y):
    return orc.backproject_matched(cbfp.ConfigProject().contents, pg.to_proj_spec_array(), chunk_for(shape, w),
                                   np.zeros(shape), y)


@pytest.mark.parametrize("signed", [False, True])
@pytest.mark.parametrize("bright", ["low", "high"])
def test_dim_voxels_far_from_the_source(device, bright, signed):
    # Voxels of 0.04 at a distance of 1000 of them, half of the detector's rows at 1 and
    # half at 1e-8: an error is measured against the voxel's own terms, A^T |y|, where
    # only dim rows reach.  FP64 sums of prefix sums in units of a cell's chord: 90 views
    # of 1.5 columns of up to 24 rows, 3240 at the end, each addition rounded by 2^-53 / 3
    # of half of that, sqrt(135) of them at random: 7e-13 of a term of 1, 135 terms of
    # 1e-8 to a voxel: 5e-7.  FP32 weights add 1e-7.  Sums in units of the distance from
    # the source would lose 1000 times as much.
    rng = np.random.default_rng(5)
    n, w, nd, views = 32, 0.04, 48, 90
    pg = ph.circular_geometry(views, nd, nd, 0.08, R=40.0, L=80.0)
    up = np.arange(nd) >= nd // 2 if (bright == "high") == (pg.det_vvec[0, 2] > 0) else np.arange(nd) < nd // 2
    y = rng.uniform(0.5, 1.0, (views, nd, nd)) * np.where(up, 1.0, 1e-8)
    if signed:
        y *= rng.choice([-1.0, 1.0], y.shape)
    y = y.astype(np.float32)
    got, want = _adjoint(pg, (n, n, n), w, y), _oracle(pg, (n, n, n), w, y)
    size = _oracle(pg, (n, n, n), w, np.abs(y))
    dim = size < 1e-7 * size.max()
    err = np.abs(got - want)[dim] / size[dim]
    rms = float(np.sqrt((err ** 2).mean()))
    print(f"dim voxels ({bright} rows bright): {dim.sum()}, rms {rms:.2e}, largest {err.max():.2e}")
    assert dim.sum() > n ** 3 // 3
    assert rms <= 3e-6
    assert err.max() <= 3e-5


# shape, views, rows; the part of the volume that is backprojected (offsets, shape)
SPLIT = {
    "tiles_of_64": ((24, 24, 40), 100, 31, None),
    "tiles_of_128": ((24, 24, 100), 100, 33, None),
    "tiles_of_192": ((24, 21, 129), 100, 40, None),
    "two_layers": ((24, 23, 193), 100, 40, None),
    "three_layers": ((24, 24, 257), 100, 41, None),
    "many_rows": ((17, 24, 70), 100, 530, None),
    "more_rows_shorter_tiles": ((16, 17, 200), 40, 1000, None),
    "more_rows_one_workgroup_per_cu": ((16, 17, 60), 40, 900, None),
    "part_of_the_volume": ((30, 29, 150), 100, 40, ((3, 5, 11), (25, 17, 131))),
}


@pytest.mark.parametrize("name", list(SPLIT))
def test_views_split_between_workgroups(device, name):
    import torch

    shape, views, nv, part = SPLIT[name]
    nu, w = 28, 25.0 / max(shape)
    pg = ph.circular_geometry(views, nu, nv, 1.6 if nv < 100 else 64.0 / nv, R=40.0, L=80.0)
    rng = np.random.default_rng(len(name))
    y = rng.uniform(-1.0, 2.0, (views, nu, nv)).astype(np.float32)
    cfg = cbfp.ConfigProject().contents
    off, cshape = part or ((0, 0, 0), shape)
    ch = chunk_for(shape, w, offsets=off, cshape=cshape)
    yt = torch.from_numpy(y).cuda()
    specs = cbfp.ProjectionSet(pg, device="cuda").specs_device()
    lib = _abi.lib()
    size = int(lib.ap_backproject_matched_workspace_size(_abi.struct_ptr(cfg), views, _abi.array3(yt)))
    outs = []
    # the whole workspace; one that leaves no room for partial sums; one for a few views
    # at a time
    for nbytes in (size, size // 3 + 4096, size // 8):
        ws = torch.full((nbytes,), 255, dtype=torch.uint8, device="cuda")   # NaN where it is not written
        v = torch.zeros(shape, dtype=torch.float32, device="cuda")
        rc = lib.ap_backproject_matched(_abi.struct_ptr(cfg), _abi.ptr(specs), views, _abi.struct_ptr(ch),
                                        _abi.array3(v), _abi.ptr(v), None, None, _abi.array3(yt), _abi.ptr(yt), 1.0,
                                        _abi.ptr(ws), nbytes, _abi.stream_handle(yt.device))
        assert rc == 0, lib.ap_last_error()
        outs.append(v.double().cpu().numpy())
    want = orc.backproject_matched(cfg, pg.to_proj_spec_array(), ch, np.zeros(shape), y)
    for got in outs:
        assert np.abs(want).max() > 0 and rel_l2(got, want) <= 1e-5
