"""Prefiltered levels made by samples (a wave to a texel) and by tiles, on both sides of the line between them:
cubes of up to 32 wide, whose every level goes by samples, and wider ones, whose levels of at most 8 do;
against the FP64 oracle with the bars of the sample tables' test."""

import numpy as np
import pytest

import oracle
from skyrendering_amd import _abi
from skyrendering_amd.ibl import cube_texels
from tests.test_gpu_ibl import _ulp_or_rel
from tests.test_gpu_ibl_tables import _smooth_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ew,pw,count", [(64, 32, 6), (1, 16, 5), (256, 4, 3), (128, 2, 2), (32, 64, 7), (64, 128, 6)])
def test_prefilter_by_samples_matches_oracle(ctx, ew, pw, count):
    cube = _smooth_cube(ew)
    env = ctx.upload(cube)
    n = cube_texels(pw, count)
    out, sh = ctx.alloc((n + 64) * 8), ctx.alloc(9 * 16)
    out.upload(np.full((n + 64, 4), 0x5555, np.uint16))
    _abi.check(_abi.lib().skyhip_ibl_precompute(ctx.handle, env.ptr, ew, sh.ptr, out.ptr, pw, count))
    got = out.download(np.uint16, (n + 64, 4))
    assert (got[n:] == 0x5555).all() and (got[:n, 3] == 0).all()
    ref = oracle.prefiltered_radiance(cube, ew, pw, count)
    ok, rel = _ulp_or_rel(got[:n, :3], ref[:, :3])
    value = cube[:, :3].view(np.float16).astype(np.float64)
    # Samples on a face edge within FP32 rounding may take the other face's texel: their share of a sum
    # is at most 1 / 16.5, and the cubes here have few enough texels for one to count.
    assert ok.mean() >= 0.99 and rel.max() <= (value.max() - value.min()) / 16.5 / value.min()
