"""Mip chains whose rows or slices number more than a grid's second and third dimension hold (65,535
workgroups) where each has a row of them, and the lines between level-by-level and tiled launches: one
level, thin and long textures, volumes; byte for byte against the oracle's box."""

import numpy as np
import pytest

import oracle
from skyrendering_amd import _abi
from skyrendering_amd import cloud as cl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,size,channels,levels", [
    (2, (1, 3_000_000, 1), 1, 0), (2, (2, 2_200_001, 1), 2, 0), (3, (1, 1_100_000, 1), 1, 0),
    (3, (1, 1, 1_200_003), 4, 0),
    (2, (37, 21, 1), 3, 2), (3, (18, 7, 33), 1, 2), (2, (600_001, 1, 1), 4, 4), (2, (15, 40_000, 1), 1, 0),
    (2, (40_000, 33, 1), 2, 5), (3, (300, 3, 1000), 1, 0), (3, (260, 260, 260), 1, 0), (3, (130, 258, 261), 1, 3),
])
def test_mip_chains_of_any_shape_match_the_box(ctx, dims, size, channels, levels):
    levels = levels or cl.mip_levels(*size)
    n = cl.mip_chain_bytes(*size, channels, levels)
    base = np.random.default_rng(n).integers(0, 256, size[0] * size[1] * size[2] * channels, np.uint8)
    chain = np.full(n + 64, 0xA5, np.uint8)
    chain[: base.size] = base
    buf = ctx.upload(chain)
    _abi.check(_abi.lib().skyhip_generate_mipmaps(ctx.handle, buf.ptr, dims, channels, *size, levels))
    got = buf.download(np.uint8, (n + 64,))
    ref = oracle.generate_mipmaps(chain[:n].copy(), dims, channels, *size, levels)
    assert np.array_equal(got[:n], ref) and (got[n:] == 0xA5).all()
