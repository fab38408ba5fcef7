"""LutSet.build follows the parameters it is given: an object changed in place between two builds, and lists
for its vectors changed in place, give the LUTs of the new values."""

import numpy as np
import pytest

from skyrendering_amd import presets
from skyrendering_amd.lutset import LutSet
from tests.test_gpu_sky_rows import _render

pytestmark = pytest.mark.gpu
SIZES = {"transmittance": (32, 8), "multiscattering": (4, 4), "sky_view": (8, 8), "aerial_perspective": (2, 2, 2)}


@pytest.mark.parametrize("change", ["scale", "list"])
def test_changed_parameters_are_seen(ctx, change):
    p, render = presets.earth_100km(), _render(40.0, 1.0, 8.0)
    p.mie_absorption = list(p.mie_absorption)
    luts = LutSet(ctx, SIZES)
    luts.build(p, render)
    before = luts.download()
    if change == "scale":
        p.mie_scattering_scale *= 3.0
    else:
        p.mie_absorption[1] *= 5.0
    luts.build(p, render)
    after = luts.download()
    fresh = LutSet(ctx, SIZES)
    fresh.build(p, render)
    ref = fresh.download()
    assert not np.array_equal(after["T"], before["T"])
    assert all(np.array_equal(after[k], ref[k]) for k in ref)
