"""One majorant, either side of the line between a lane per path and the cooperative kernel (a constant
medium; paths of one bounce over full waves, 3,072 of 64 on 256 CUs): bit for bit the kernel with one lane
per path and counters, one and several frames."""

import pytest

from skyrendering_amd import presets
from skyrendering_amd import cloud as cl
from skyrendering_amd.pathtrace import PathTraceScene, PathTracingInitParam
from skyrendering_amd.scenes import CloudScene
from tests.test_gpu_pathtrace_coop import _both, _inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,bounces,frames", [(511, 385, 1, 2), (509, 380, 1, 1), (511, 385, 2, 1), (61, 40, 1, 1)])
@pytest.mark.parametrize("material", ["default1", "worley", "minimal"])
def test_routes_of_procedural_materials_agree(ctx, material, w, h, bounces, frames):
    wl = presets.cloud_workload_config2() if material == "worley" else presets.cloud_workload()
    if material == "minimal":
        wl["material"] = cl.VolumetricCloudMinimalMaterial(density=0.7)
    scene = CloudScene(ctx, w, h, workload=wl)
    sigma = 1.1 if material == "minimal" else scene.material.density
    init = PathTracingInitParam(max_bounces=bounces, region_box_half_width=14.0)
    args = (scene.atmosphere.buffer, scene.renderer.buffer, scene.common, scene.mat_block, _inputs(scene))
    _both(ctx, args, init.to_c(sigma, scene.model), w, h, (0, 0, w, h), frames)


@pytest.mark.parametrize("w,h,bounces", [(640, 360, 1), (640, 360, 3), (100, 90, 1)])
def test_routes_of_a_voxel_grid_agree(ctx, w, h, bounces):
    wl = presets.path_trace_workload()
    wl["grid_dims"], wl["density"] = (32, 32, 32), 2.0
    init = PathTracingInitParam(max_bounces=bounces, region_box_half_width=14.0)
    scene = PathTraceScene(ctx, w, h, workload=wl, init=init, bricks=False)
    args = (scene.atmosphere.buffer, scene.renderer.buffer, scene.common, scene.material, scene.inputs)
    _both(ctx, args, scene.tracer.params, w, h, (0, 0, w, h), 1)
