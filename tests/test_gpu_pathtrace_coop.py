"""Single-majorant tracking by the whole wave against the kernel with one lane per path (the counting
variant), bit for bit: every material, ragged regions smaller and larger than a wave's tile, several
frames, both random sequences and environment modes, at the sizes where a wave takes 64 paths and
fewer."""

import numpy as np
import pytest

from skyrendering_amd import _abi, presets
from skyrendering_amd import cloud as cl
from skyrendering_amd.pathtrace import PathTraceScene, PathTracingInitParam, path_trace
from skyrendering_amd.scenes import CloudScene

pytestmark = pytest.mark.gpu


def _both(ctx, scene_inputs, params, w, h, region, frames):
    atm, render, common, material, inputs = scene_inputs
    out = []
    for counters in (None, ctx.alloc(40)):
        if counters is not None:
            counters.zero()
        acc, mask = ctx.alloc(w * h * 16), ctx.alloc(w * h)
        acc.zero(), mask.zero()
        path_trace(ctx, atm, render, common, material, params, inputs, region, 3, frames, acc, mask, w, h, counters)
        out.append((acc.download(np.uint32, (h, w, 4)), mask.download(np.uint8, (h, w))))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert out[0][0].any()


def _inputs(scene):
    a, r = scene.atmosphere, scene.renderer
    i = _abi.PathTracingInputsC()
    i.transmittance = a.transmittance_texture.ptr
    i.transmittance_width, i.transmittance_height = a.transmittance_size
    i.sky_view_luminance = r.sky_view_luminance_texture.ptr
    i.sky_view_transmittance = r.sky_view_transmittance_texture.ptr
    i.sky_view_width, i.sky_view_height = r.init.sky_view_lut_size
    i.ap_luminance = r.aerial_perspective_luminance_texture.ptr
    i.ap_transmittance = r.aerial_perspective_transmittance_texture.ptr
    i.ap_width, i.ap_height = r.init.aerial_perspective_lut_size
    i.ap_depth = r.init.aerial_perspective_lut_depth
    return i


@pytest.mark.parametrize("material", ["default0", "default1", "worley", "minimal", "voxel"])
@pytest.mark.parametrize("w,h,region,frames,env,prng", [
    (67, 45, (0, 0, 67, 45), 2, "GROUND_MULTI_BOUNCE", "PCGHash"),
    (40, 40, (5, 3, 8, 4), 1, "GROUND_SINGLE_BOUNCE", "WangHash"),
])
def test_cooperative_tracking_matches_per_lane_tracking(ctx, material, w, h, region, frames, env, prng):
    wl = presets.cloud_workload_config2() if material == "worley" else presets.cloud_workload()
    if material == "default0":
        m = cl.VolumetricCloudDefaultMaterial0(
            **{f: getattr(wl["material"], f) for f in cl.DefaultMaterialCommon.__dataclass_fields__})
        m.detail_param = (0.8, 0.1)
        wl["material"] = m
    elif material == "minimal":
        wl["material"] = cl.VolumetricCloudMinimalMaterial(density=0.7)
    scene = CloudScene(ctx, w, h, workload=wl)
    mat, sigma = scene.mat_block, getattr(scene.material, "density", 0.7)
    keep = None
    if material == "minimal":
        sigma = 1.1  # null collisions
    elif material == "voxel":
        n = 16
        levels = cl.mip_levels(n, n, n)
        keep = ctx.alloc(cl.mip_chain_bytes(n, n, n, 1, levels))
        keep.upload(np.random.default_rng(2).integers(0, 256, (n, n, n), np.uint8))
        _abi.check(_abi.lib().skyhip_generate_mipmaps(ctx.handle, keep.ptr, 3, 1, n, n, n, levels))
        vm = cl.VolumetricCloudVoxelMaterial(density=3.0, base=(2.0, 2.0), width=(9.0, 9.0))
        mat, sigma = cl.voxel_material(vm, keep, (n, n, n), levels, (w, h), scene.camera), 3.0
    init = PathTracingInitParam(max_bounces=9, region_box_half_width=14.0, environment_lighting=env, prng=prng,
                                importance_sampling=prng == "PCGHash", albedo=0.98)
    args = (scene.atmosphere.buffer, scene.renderer.buffer, scene.common, mat, _inputs(scene))
    _both(ctx, args, init.to_c(sigma, scene.model), w, h, region, frames)


@pytest.mark.parametrize("w,h", [(33, 21), (250, 300), (700, 500)])
def test_cooperative_tracking_of_a_voxel_grid_matches(ctx, w, h):
    wl = presets.path_trace_workload()
    wl["grid_dims"], wl["density"] = (32, 32, 32), 2.0
    scene = PathTraceScene(ctx, w, h, workload=wl, bricks=False)
    args = (scene.atmosphere.buffer, scene.renderer.buffer, scene.common, scene.material, scene.inputs)
    _both(ctx, args, scene.tracer.params, w, h, (0, 0, w, h), 1)
