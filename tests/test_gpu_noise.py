"""Noise generators where their tiles can go wrong: sizes around the tile edges (16 x 16 images, 8 x 8 x 4
volumes), lattice periods below 4, octaves whose cells fit the tile's tables, only their (y, z) columns
do, and neither does (a period far above the size), against the oracle's FP32 texels.

The oracle's FP32 path makes the same float operations except that the compilers contract
multiply-adds differently, which moves a value by a few FP32 ulps: at most one UNORM8 step, and only
within ~1e-6 of a rounding boundary, so in fewer than 1 % of the texels here."""
import numpy as np
import pytest

import oracle
from skyrendering_amd.cloud import CloudTextures, NoiseCreateInfo, VolumetricCloudDefaultMaterial1Worley

pytestmark = pytest.mark.gpu


def _close(got, ref, what):
    diff = np.abs(got.astype(np.int32) - ref.astype(np.int32))
    assert diff.max() <= 1 and np.mean(diff > 0) <= 0.01, (what, diff.max(), float(np.mean(diff > 0)))


@pytest.mark.parametrize("size,base", [(2, 1), (8, 2), (16, 3), (32, 5), (64, 23), (8, 700)])
def test_noise_tiles_match_oracle(ctx, size, base):
    info = lambda seed: NoiseCreateInfo(seed, base, 0.1, 0.9)  # noqa: E731
    m = VolumetricCloudDefaultMaterial1Worley(
        cloud_map_density=info(3), cloud_map_height=info(4), detail_perlin=info(5), detail_worley=info(6),
        displacement_perlin=info(7), worley=info(8))
    tex = CloudTextures(ctx, size, size, size, worley_size=size).generate(m)
    cm, det, disp = tex.download()
    px, vx = np.arange(size * size), np.arange(size ** 3)
    if len(vx) > 40000:
        vx = np.random.default_rng(1).choice(vx, 40000, replace=False)
    _close(cm[:2 * size * size].reshape(-1, 2),
           oracle.cloud_map_texels(info(3).to_c(), info(4).to_c(), size, px, "f32"), "cloud map")
    _close(det[vx], oracle.detail_texels(info(5).to_c(), info(6).to_c(), size, vx, "f32"), "detail")
    _close(disp[:4 * size * size].reshape(-1, 4), oracle.displacement_texels(info(7).to_c(), size, px, "f32"),
           "displacement")
    _close(tex.download_worley()[vx], oracle.worley_texels(info(8).to_c(), size, vx, "f32"), "Worley volume")


@pytest.mark.parametrize("size", [1, 3, 7, 17, 33])
def test_noise_ragged_tiles_match_oracle(ctx, size):
    """Sizes no tile divides (the cell copies need powers of two, so without them)."""
    m = VolumetricCloudDefaultMaterial1Worley()
    tex = CloudTextures(ctx, size, size, size, worley_size=size, cells=False).generate(m)
    cm, det, disp = tex.download()
    px, vx = np.arange(size * size), np.arange(size ** 3)
    _close(cm[:2 * size * size].reshape(-1, 2),
           oracle.cloud_map_texels(m.cloud_map_density.to_c(), m.cloud_map_height.to_c(), size, px, "f32"), "cloud map")
    _close(det[vx], oracle.detail_texels(m.detail_perlin.to_c(), m.detail_worley.to_c(), size, vx, "f32"), "detail")
    _close(disp[:4 * size * size].reshape(-1, 4),
           oracle.displacement_texels(m.displacement_perlin.to_c(), size, px, "f32"), "displacement")
    _close(tex.download_worley()[vx], oracle.worley_texels(m.worley.to_c(), size, vx, "f32"), "Worley volume")
