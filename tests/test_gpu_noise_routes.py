"""Noise by tiles and by texels, on both sides of the line between them (few and many texels, coarse and fine
lattices, periods of 1 to 3 cells, edges no tile divides): textures against the oracle's FP32 texels within
one UNORM8 step, as the generators' other tests, and voxel grids against its FP16 grid."""

import numpy as np
import pytest

import oracle
from skyrendering_amd import _abi
from skyrendering_amd.cloud import CloudTextures, NoiseCreateInfo, VolumetricCloudDefaultMaterial1Worley
from skyrendering_amd.pathtrace import VoxelGrid, VoxelGridCreateInfo
from tests.test_gpu_noise import _close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size,base", [(8, 8), (16, 8), (32, 3), (41, 7), (64, 100), (128, 1), (129, 2), (160, 3),
                                       (250, 90), (270, 8), (260, 500)])
def test_noise_routes_match_oracle(ctx, size, base):
    info = lambda seed: NoiseCreateInfo(seed, base, 0.1, 0.9)  # noqa: E731
    m = VolumetricCloudDefaultMaterial1Worley(
        cloud_map_density=info(3), cloud_map_height=info(4), detail_perlin=info(5), detail_worley=info(6),
        displacement_perlin=info(7), worley=info(8))
    volume = min(size, 64)
    tex = CloudTextures(ctx, size, volume, size, worley_size=volume, cells=False).generate(m)
    cm, det, disp = tex.download()
    px, vx = np.arange(size * size), np.arange(volume ** 3)
    if len(vx) > 20000:
        vx = np.random.default_rng(1).choice(vx, 20000, replace=False)
    _close(cm[:2 * size * size].reshape(-1, 2),
           oracle.cloud_map_texels(info(3).to_c(), info(4).to_c(), size, px, "f32"), "cloud map")
    _close(disp[:4 * size * size].reshape(-1, 4), oracle.displacement_texels(info(7).to_c(), size, px, "f32"),
           "displacement")
    _close(det[vx], oracle.detail_texels(info(5).to_c(), info(6).to_c(), volume, vx, "f32"), "detail")
    _close(tex.download_worley()[vx], oracle.worley_texels(info(8).to_c(), volume, vx, "f32"), "Worley volume")


@pytest.mark.parametrize("dims,base,octaves", [((8, 8, 8), 1, 5), ((40, 41, 39), 2, 3), ((48, 44, 40), 2, 4),
                                               ((48, 44, 40), 100, 4), ((9, 130, 64), 1, 12), ((64, 64, 64), 65536, 2)])
def test_voxel_grid_routes_match_oracle(ctx, dims, base, octaves):
    ci = VoxelGridCreateInfo(base_frequency=base, octaves=octaves, threshold=0.5)
    grid = VoxelGrid(ctx, dims, cells=False).generate(ci)
    got = grid.download().view(np.float16).astype(np.float64)
    ref = oracle.voxel_grid_f16(ci.to_c(), dims).view(np.float16).astype(np.float64)
    # The FP32 forms round differently by a few ulps: at most one FP16 unit (2^-10 of the value), or the
    # rounding of the density before the threshold where little is left of it.
    assert np.abs(got - ref).max() <= 2.0 ** -10 * np.abs(ref).max()
    assert np.mean(got != ref) < 0.01 and got.any()
