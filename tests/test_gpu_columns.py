"""Column backprojection (ap_backproject on upright panels) at the sizes where
its parts meet, against the FP64 oracle: heights around one, two, three and
four voxels per thread (64 planes apart) and around a second part of the
column, panels that hold every tap (no edge handling), panels that cut the
column, and voxel columns in the softening band; v-contiguous data, a slice of
wider data (odd strides, odd start) and fp16.  Relative L2 <= 2e-5 as for the
other interpolating backprojections (FP32 coordinates: 2^-24 of some 50 pixels
against pixel differences of order 1 is 3e-6 per sample).

Nearest-pixel reads flip where a coordinate lies within FP32 rounding of a
pixel edge, so those cases use data that is constant along v in blocks and
linear along u: a flip changes a value by 1 / 40 at most.
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

HEIGHTS = [1, 63, 64, 65, 128, 129, 193, 256, 257]
KINDS = {
    "fdk": dict(approx_mode_bilinear_interpolate=True, Z_on_L_factor_power=-2),
    "soft": dict(approx_mode_bilinear_interpolate=True, soften_det_edges_proportion=0.2),
    "nearest": dict(cyl_mask_rad=1.6, soften_det_edges_proportion=0.1),
}


def panels(views: int, nu: int, nv: int, lift: float) -> cbfp.ProjGeom:
    g = ph.circular_geometry(views, nu, nv, 1.0, R=40.0, L=80.0)
    up = np.linspace(-lift, lift, views)[:, None] * np.array([0.0, 0.0, 1.0])
    return cbfp.ProjGeom(source_pos=g.source_pos + up, det_pos=g.det_pos + up, det_uvec=g.det_uvec,
                         det_vvec=np.broadcast_to(g.det_vvec, g.det_uvec.shape).copy(), nu=nu, nv=nv)


def smooth(rng, views: int, nu: int, nv: int) -> np.ndarray:
    # slope at most 1 / 40 per pixel, sign and slope from view to view
    u, v = np.arange(nu) / 40.0, np.arange(nv) / 40.0
    s = rng.uniform(-1, 1, (views, 2))
    return (1.0 + s[:, :1, None] * u[None, :, None] + s[:, 1:, None] * v[None, None, :]).astype(np.float32)


def layout(y: np.ndarray, name: str):
    import torch

    t = torch.from_numpy(y).cuda()
    if name == "f16":
        t = t.to(torch.float16)
        return t, t.float().cpu().numpy()
    if name == "slice":
        V, nu, nv = y.shape  # noqa: N806
        wide = torch.full((V, nu + 2, nv + 3), float("nan"), device="cuda")
        wide[:, 1 : nu + 1, 1 : nv + 1] = t
        return wide[:, 1 : nu + 1, 1 : nv + 1], y
    return t, y


@pytest.mark.parametrize("name", ["f32", "slice", "f16"])
@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("nz", HEIGHTS)
def test_columns_match_oracle(device, nz, kind, name):
    rng = np.random.default_rng(nz)
    views = 66 if nz in (1, 257) else 5          # more than one batch of views, and a short one
    shape, w = (5, 6, nz), 3.2 / 6
    tall = nz * w                                # magnification 2 about the axis
    nv = max(9, int(2.3 * tall) | 1) if nz != 193 else 41   # 193: the panel cuts the column
    pg = panels(views, 21, nv, 0.2)
    y, yy = layout(smooth(rng, views, 21, nv), name)
    cfg = cbfp.ConfigBackproject(fast_approx=True, **KINDS[kind])
    v = Volume(np.zeros(shape, np.float32), voxwid=w)
    cbfp.backproject(cfg, v, cbfp.ProjectionSet(pg, data=y), block=True)
    want = orc.backproject(cfg.contents, pg.to_proj_spec_array(), chunk_for(shape, w), np.zeros(shape), yy)
    err = rel_l2(v.as_numpy(), want)
    print(f"columns nz={nz} {kind} {name}: rel L2 {err:.3e}")
    assert np.abs(want).max() > 0
    # a flipped pixel moves a value by 1/40 of its neighbours' size; at most a few in 10^4 samples do
    assert err <= (5e-4 if kind == "nearest" else 2e-5)
