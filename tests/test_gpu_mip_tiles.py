"""Mip chains built several levels to a launch, byte for byte against the oracle's level-by-level box: sizes
below, at and across the tiles, odd and unequal edges (an edge reaches one texel before the others),
1 to 4 channels, chains cut short; nothing past the chain is written."""

import numpy as np
import pytest

import oracle
from skyrendering_amd import _abi
from skyrendering_amd import cloud as cl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,size,channels,cut", [
    (2, (1, 1, 1), 4, 0), (2, (2, 1, 1), 1, 0), (2, (64, 64, 1), 4, 0), (2, (67, 5, 1), 3, 0), (2, (257, 130, 1), 2, 1),
    (2, (1, 300, 1), 1, 0), (2, (512, 512, 1), 2, 2), (3, (2, 2, 2), 1, 0), (3, (16, 16, 16), 1, 0),
    (3, (33, 17, 9), 2, 0), (3, (1, 40, 70), 4, 0), (3, (64, 64, 64), 1, 1), (3, (50, 3, 128), 3, 0),
])
def test_mip_tiles_match_the_box_level_by_level(ctx, dims, size, channels, cut):
    levels = cl.mip_levels(*size) - cut
    n = cl.mip_chain_bytes(*size, channels, levels)
    base = np.random.default_rng(n).integers(0, 256, size[0] * size[1] * size[2] * channels, np.uint8)
    chain = np.full(n + 64, 0xA5, np.uint8)
    chain[: base.size] = base
    buf = ctx.upload(chain)
    _abi.check(_abi.lib().skyhip_generate_mipmaps(ctx.handle, buf.ptr, dims, channels, *size, levels))
    got = buf.download(np.uint8, (n + 64,))
    ref = oracle.generate_mipmaps(chain[:n].copy(), dims, channels, *size, levels)
    assert np.array_equal(got[:n], ref) and (got[n:] == 0xA5).all()
