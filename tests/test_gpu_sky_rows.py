"""The row-by-row sky-view march and the multiple-scattering step tables where they can go wrong: one
and several pieces of a row (64, 128 and 192 columns), ragged rows, more steps than a table holds at
a time (32) or at all (64, direction by direction), one step, fractional counts, the sun up, crossing
and below the horizon, low and high cameras and one above the atmosphere, small and large planets, and
LUTs up to and past the columns a wave's entries hold (288).  Against the FP64 oracle with the bar of
the other LUT tests (1e-3 of the value, floored at 1e-6 of the LUT's largest; these differ by 1e-5 to
6e-5 at most, from FP32 rays near the horizon)."""
import numpy as np
import pytest

import oracle
from skyrendering_amd import Atmosphere, AtmosphereRenderer, AtmosphereRenderInitParameters, presets
from skyrendering_amd.atmosphere import AtmosphereRenderParameters
from skyrendering_amd import surrogate as sg
from skyrendering_amd.batch import LutBatch

pytestmark = pytest.mark.gpu
TOL = 1e-3


def _rel(x, ref):
    x, ref = x[..., :3].astype(np.float64), ref[..., :3].astype(np.float64)
    return float(np.max(np.abs(x - ref) / np.maximum(np.abs(ref), 1e-6 * np.abs(ref).max())))


def _render(theta, altitude, steps):
    cam = presets.bench_camera(altitude_km=altitude)
    return AtmosphereRenderParameters(sun_direction_theta=theta, sun_direction_phi=180.0, sky_view_lut_steps=steps,
                                      camera_position=cam.position, view_projection=cam.view_projection())


@pytest.mark.parametrize("size,t_size,ms_size,steps,theta,altitude,radius", [
    ((64, 16), (256, 64), (32, 32), 30.0, 20.0, 1.0, 6360.0),
    ((65, 9), (64, 16), (16, 16), 32.0, 89.0, 0.1, 6360.0),
    ((193, 21), (128, 32), (33, 17), 33.0, 93.0, 2.0, 6360.0),
    ((384, 20), (256, 64), (32, 32), 70.4, 96.0, 10.0, 6360.0),
    ((100, 30), (255, 40), (33, 20), 30.0, 60.0, 60.0, 3000.0),
    ((96, 22), (256, 64), (33, 32), 30.0, 88.0, 1.0, 6360.0),  # 289 columns: texel by texel
    ((130, 17), (288, 16), (40, 8), 12.7, 85.0, 5.0, 6360.0),
    ((20, 24), (2, 2), (2, 2), 1.0, 45.0, 3.0, 6360.0),
    ((90, 33), (256, 64), (32, 32), 40.0, 50.0, 250.0, 6360.0),  # above the atmosphere
])
def test_sky_view_rows_match_oracle(ctx, size, t_size, ms_size, steps, theta, altitude, radius):
    p = presets.earth_100km()
    p.bottom_radius = radius
    atm = Atmosphere(ctx, transmittance_size=t_size, multiscattering_size=ms_size)
    atm.update_luts(p)
    rend = AtmosphereRenderer(ctx, AtmosphereRenderInitParameters(sky_view_lut_size=size))
    rp = _render(theta, altitude, steps)
    rend.render(atm, p, rp, aerial_perspective=False)
    L, Tr = rend.sky_view()
    refL, refT = oracle.sky_view_lut(atm.buffer, rend.buffer, atm.transmittance(), atm.multiscattering(), *size)
    # The middle row of an odd height looks exactly at the horizon, where rounding decides whether a ray
    # of a thousand kilometres hits the ground at half its length.
    rows = np.arange(size[1]) * 2 != size[1] - 1
    assert _rel(Tr[rows], refT[rows]) < TOL and _rel(L[rows], refL[rows]) < TOL
    # The batch's pieces of a row give the same bits.
    batch = LutBatch(ctx, [(atm.buffer, t_size, ms_size)], [(0, rp.buffer_data(radius), size)])
    batch.launch()
    ctx.synchronize()
    bl, bt = batch.view_outputs(0)
    assert np.array_equal(bl, L) and np.array_equal(bt, Tr)


@pytest.mark.parametrize("size,steps,radius", [((32, 32), 30.0, 6360.0), ((5, 3), 1.0, 6360.0), ((33, 9), 33.5, 3000.0),
                                               ((6, 7), 64.0, 6360.0), ((9, 4), 65.0, 6360.0)])
def test_multiscattering_tables_match_oracle(ctx, size, steps, radius):
    p = presets.earth_100km()
    p.bottom_radius, p.multiscattering_steps = radius, steps
    atm = Atmosphere(ctx, transmittance_size=(64, 16), multiscattering_size=size)
    atm.update_luts(p)
    ms = atm.multiscattering()
    assert _rel(ms, oracle.multiscattering_lut(atm.buffer, atm.transmittance(), *size)) < TOL
    batch = LutBatch(ctx, [(atm.buffer, (64, 16), size)], [])
    batch.launch()
    ctx.synchronize()
    assert np.array_equal(batch.set_outputs(0)[1], ms)
    batch.set_tuning(multiscattering_waves=1)
    batch.launch()
    ctx.synchronize()
    assert np.array_equal(batch.set_outputs(0)[1], ms)


@pytest.mark.parametrize("w,h,steps,t_size,ms_size", [(16, 16, 30.0, (256, 64), (32, 32)), (1, 1, 32.0, (64, 16), (8, 8)),
                                                      (37, 50, 33.0, (64, 16), (16, 16)),
                                                      (50, 17, 0.5, (64, 16), (16, 16)),
                                                      (275, 33, 70.5, (288, 16), (33, 8))])
def test_panorama_tiles_and_probes_match_oracle(ctx, w, h, steps, t_size, ms_size):
    """The plain pass's tiles (ragged edges, more steps than a table, a count of 0) and the residual check's
    probes, by rows and, for LUTs past a wave's entries, one by one, against the FP64 oracle."""
    scales, views = sg.evaluation_views(2, seed=5)
    atm = sg.SkyAtmospheres(ctx, scales, t_size=t_size, ms_size=ms_size, steps=steps)
    pano = sg.SkyPanoramas(ctx, atm, views, w, h)
    blocks, T, MS = atm.host_luts()
    ys, xs = (v.ravel() for v in np.meshgrid(np.arange(h), np.arange(w), indexing="ij"))
    refs = [oracle.sky_radiance(blocks, T, MS, steps, pano.pixel_queries(v, xs, ys)).reshape(h, w, 3) for v in range(2)]
    # Rays within 1e-3 rad of the horizon pass it on one side or the other by rounding.
    mu = np.cos(np.pi * (np.arange(h) + 0.5) / h)
    sure = [np.abs(np.arccos(mu) - np.pi / 2 - np.arccos(6360.0 / (6360.0 + v["altitude"]))) > 1e-3 for v in views]
    pano.render_plain()
    image = pano.image()[..., :3]
    for v in range(2):
        assert _rel(image[v][sure[v]], refs[v][sure[v]]) < TOL if steps > 0.5 else not image[v].any()
    pano.render_surrogate(sg.SkySurrogate(ctx, seed=3), tolerance=1e30)
    image = pano.image()[..., :3]
    py = sorted({min(t + o, h - 1) for t in range(0, h, 16) for o in (4, 12)})
    px = sorted({min(t + o, w - 1) for t in range(0, w, 16) for o in (4, 12)})
    for v in range(2):
        rows = [y for y in py if sure[v][y]]
        got, ref = image[v][np.ix_(rows, px)], refs[v][np.ix_(rows, px)]
        assert _rel(got, ref) < TOL if steps > 0.5 else not got.any()
