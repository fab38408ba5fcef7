"""The limit on a track's tentative collisions (2^20): the cooperative kernel stops at the same draw as the
kernel with one lane per path.  A majorant of 1e6 per kilometre in a medium of 0.7 makes the shadow rays'
tracks reach it (about a kilometre into the layer), each of the limit's lookups a factor of 1 - 7e-7 of
the transmittance: the images agree bit for bit only if the numbers of lookups do."""

import numpy as np
import pytest

from skyrendering_amd import _abi, presets
from skyrendering_amd import cloud as cl
from skyrendering_amd.pathtrace import PathTracingInitParam
from skyrendering_amd.scenes import CloudScene
from tests.test_gpu_pathtrace_coop import _both, _inputs

pytestmark = pytest.mark.gpu


def test_cooperative_tracking_stops_at_the_limit(ctx):
    w, h, n = 128, 96, 2
    scene = CloudScene(ctx, w, h, workload=presets.cloud_workload())
    levels = cl.mip_levels(n, n, n)
    voxels = ctx.upload(np.full(cl.mip_chain_bytes(n, n, n, 1, levels), 255, np.uint8))
    vm = cl.VolumetricCloudVoxelMaterial(density=0.7, base=(0.0, 0.0), width=(1e4, 1e4))
    material = cl.voxel_material(vm, voxels, (n, n, n), levels, (w, h), scene.camera)
    init = PathTracingInitParam(max_bounces=1, region_box_half_width=14.0)
    args = (scene.atmosphere.buffer, scene.renderer.buffer, scene.common, material, _inputs(scene))
    _both(ctx, args, init.to_c(1e6, scene.model), w, h, (0, 0, w, h), 1)
