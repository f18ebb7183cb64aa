"""Column backprojection (ap_backproject on upright panels) at the sizes where
its parts meet, against the FP64 oracle: heights around one, two, three and
four voxels per thread (64 planes apart) and around a second part of the
column, panels that hold every tap (no edge handling), panels that cut the
column, and voxel columns in the softening band; v-contiguous data, a slice of
wider data (odd strides, odd start) and fp16.  Relative L2 <= 2e-5 as for the
other interpolating backprojections (FP32 coordinates: 2^-24 of some 50 pixels
against pixel differences of order 1 is 3e-6 per sample), 1e-5 for GBC.

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


@pytest.mark.parametrize("name", ["f32", "slice", "f16"])
@pytest.mark.parametrize("nz", HEIGHTS)
@pytest.mark.parametrize("mixed", [False, True], ids=["upright", "mixed"])
def test_gbc_columns_match_oracle(device, mixed, nz, name):
    # the second batch of views tilted in "mixed": both routes add to one sum
    rng = np.random.default_rng(500 + nz)
    views, nu = (70 if mixed else 6), 31
    shape, w = (5, 6, nz), 3.2 / 6
    nv = max(9, int(2.3 * nz * w) | 1) if nz != 193 else 41
    pg = panels(views, nu, nv, 0.3 * nz * w)
    if mixed:
        c, s = np.cos(0.05), np.sin(0.05)
        du, dv = pg.det_uvec.copy(), pg.det_vvec.copy()
        du[64:], dv[64:] = (c * pg.det_uvec + s * pg.det_vvec)[64:], (c * pg.det_vvec - s * pg.det_uvec)[64:]
        pg = cbfp.ProjGeom(source_pos=pg.source_pos, det_pos=pg.det_pos, det_uvec=du, det_vvec=dv, nu=nu, nv=nv)
    y, yy = layout(rng.uniform(-1, 2, (views, nu, nv)).astype(np.float32), name)
    cfg = cbfp.ConfigBackproject(fast_approx=True, backproj_weighting_preset=7, Z_on_val_factor_val=40.0,
                                 approx_mode_bilinear_interpolate=True, soft_vartheta_v=0.4,
                                 soft_vartheta_v_softspan=0.2, soft_vartheta_h=0.06, soft_vartheta_h_softspan=0.04)
    v = Volume(np.zeros(shape, np.float32), voxwid=w)
    sec = Volume(np.zeros(shape, np.float32), voxwid=w)
    cbfp.backproject(cfg, v, cbfp.ProjectionSet(pg, data=y), secondary_volume=sec, block=True)
    wv, ws = orc.backproject_gbc(cfg.contents, pg.to_proj_spec_array(), chunk_for(shape, w), np.zeros(shape),
                                 np.zeros(shape), yy)
    e1, e2 = rel_l2(v.as_numpy(), wv), rel_l2(sec.as_numpy(), ws)
    print(f"GBC columns nz={nz} {name} mixed={mixed}: values {e1:.3e}, weights {e2:.3e}")
    assert np.abs(ws).max() > 0
    assert e1 <= 2e-5 and e2 <= 1e-5
