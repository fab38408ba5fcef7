"""The LUT set's multiple scattering at step counts around its tables' 64 steps: none, one, parts of a wave,
whole and partial chunks, fractional counts, against the FP64 oracle with the bar of the other LUT tests."""

import pytest

import oracle
from skyrendering_amd import presets
from skyrendering_amd.lutset import LutSet
from tests.test_gpu_sky_rows import TOL, _rel, _render

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [0.4, 1.0, 33.0, 64.0, 64.6, 96.0, 128.0, 129.0, 300.5])
@pytest.mark.parametrize("size", [(2, 2), (9, 5)])
def test_set_multiscattering_chunks_match_oracle(ctx, steps, size):
    p = presets.earth_100km()
    p.multiscattering_steps = steps
    luts = LutSet(ctx, {"transmittance": (64, 16), "multiscattering": size, "sky_view": (8, 8),
                        "aerial_perspective": (2, 2, 2)})
    luts.build(p, _render(40.0, 1.0, 8.0))
    out = luts.download()
    ref = oracle.multiscattering_lut(p.buffer_data(), out["T"], *size)
    assert _rel(out["MS"], ref) < TOL
