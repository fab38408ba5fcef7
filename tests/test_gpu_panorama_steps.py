"""Panoramas of few steps: on both sides of the line between a march per pixel (and per probe) and marches
shared by rows (12 steps), against the FP64 oracle with the bar of the other panorama tests."""

import numpy as np
import pytest

import oracle
from skyrendering_amd import surrogate as sg
from tests.test_gpu_sky_rows import TOL, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [1.0, 4.7, 11.5, 11.6, 13.0])
@pytest.mark.parametrize("t_size", [(64, 16), (300, 8)])
def test_short_marches_match_oracle(ctx, steps, t_size):
    w, h = 37, 50
    scales, views = sg.evaluation_views(2, seed=5)
    atm = sg.SkyAtmospheres(ctx, scales, t_size=t_size, ms_size=(16, 16), steps=steps)
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
        assert _rel(image[v][sure[v]], refs[v][sure[v]]) < TOL
    model = sg.SkySurrogate(ctx, seed=3)
    pano.render_surrogate(model, tolerance=1e30)
    assert pano.fallback_tiles() == 0
    image = pano.image()[..., :3]
    py = sorted({min(t + o, h - 1) for t in range(0, h, 16) for o in (4, 12)})
    px = sorted({min(t + o, w - 1) for t in range(0, w, 16) for o in (4, 12)})
    for v in range(2):
        rows = [y for y in py if sure[v][y]]
        assert _rel(image[v][np.ix_(rows, px)], refs[v][np.ix_(rows, px)]) < TOL
    pano.render_surrogate(model, tolerance=1e-30)
    assert pano.fallback_tiles() == 2 * pano.tiles
    image = pano.image()[..., :3]
    for v in range(2):
        assert _rel(image[v][sure[v]], refs[v][sure[v]]) < TOL
