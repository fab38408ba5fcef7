"""The workloads this library's users run, as measurable cases.

A case is a dict of plain values; its "kind" names the call a program makes each frame, step or
edit:

  lut_set          LutSet.build: one frame's four atmosphere LUTs
  sky_frame        Atmosphere.update_luts, AtmosphereRenderer.render, EnvironmentLuminance.update and
                   IBL.precompute: the atmosphere's share of one frame, pass by pass
  lut_batch        LutBatch.launch: many atmosphere sets and sun angles in one launch
  cloud_shadow     CloudShadow.render: shadow map (blended with the last frame's), blur, froxel
  raymarch         CloudScene.run: the cloud raymarch, one ray per pixel
  cloud_frame      CloudReconstruction.render: checkerboard, quarter-resolution raymarch, temporal
                   reconstruction and upscale composite
  path_trace       PathTracing.render over an FP16 voxel grid with brick majorants, and display
  path_trace_mat   PathTracing.render over a procedural material with its single majorant
  panorama_plain   SkyPanoramas.render_plain: the integrator at every pixel
  panorama_net     SkyPanoramas.render_surrogate with a tolerance nothing exceeds: the network pass
                   with its probes
  train_step       SkySurrogate.gradient and SkySurrogate.adam on one batch
  textures         CloudTextures.generate: noise textures, mip chains and cell copies after an edit

`exact` restates the atmosphere integrator and the surrogate in 64-bit torch.  The passes that
branch on what they computed (clouds, path tracing), the IBL products and the byte textures have
no such restatement here; they are compared with the tolerances below.

Every state shares one Context, as a program does, so passes run in order on one stream.
"""
import math

import numpy as np
import torch

from skyrendering_amd import (Atmosphere, AtmosphereRenderer, AtmosphereRenderInitParameters, Context, _abi, presets)
from skyrendering_amd import cloud as cl
from skyrendering_amd import surrogate as sg
from skyrendering_amd.atmosphere import AtmosphereRenderParameters
from skyrendering_amd.batch import LutBatch
from skyrendering_amd.ibl import IBL, EnvironmentLuminance, cube_texels
from skyrendering_amd.lutset import LutSet
from skyrendering_amd.pathtrace import PathTraceScene, PathTracing, PathTracingInitParam
from skyrendering_amd.scenes import CloudScene

AP_STEPS = 50.867000579833984  # bin/config.json
AP_DISTANCE = 203.0


def listed():
    return [
        # One frame's LUTs at the Earth preset's sizes: about 50 us, launches and latency count.
        {"name": "lut_set_earth", "kind": "lut_set", "tw": 256, "th": 64, "mw": 32, "mh": 32, "sw": 192, "sh": 108,
         "aw": 32, "ah": 32, "ad": 32},
        # The reference's frame order with its compile-time LUT sizes, environment cube and IBL.
        {"name": "sky_frame_reference", "kind": "sky_frame", "sw": 128, "sh": 128, "aw": 32, "ah": 32, "ad": 32,
         "env": 128},
        # Precomputing skies for many planets and times of day.
        {"name": "lut_batch_256x8", "kind": "lut_batch", "sets": 256, "suns": 8},
        # Cloud shadows of a 1080p frame, the reference's 512^2 map.
        {"name": "cloud_shadow_1080p", "kind": "cloud_shadow", "w": 1920, "h": 1080, "map": 512, "material": "worley"},
        # Full-resolution clouds at 1080p: the headline workload.
        {"name": "raymarch_1080p", "kind": "raymarch", "w": 1920, "h": 1080, "material": "worley"},
        # The reference's real-time cloud frame at 1080p.
        {"name": "cloud_frame_1080p", "kind": "cloud_frame", "w": 1920, "h": 1080, "material": "default1"},
        # Offline rendering of a voxel cloud: one sample a pixel a pass.
        {"name": "path_trace_1024", "kind": "path_trace", "w": 1024, "h": 1024, "grid": 512, "brick": 16},
        # Path-traced preview of the procedural cloud the raymarch shows, at an odd size.
        {"name": "path_trace_procedural", "kind": "path_trace_mat", "w": 321, "h": 181, "material": "default1"},
        # Sky panoramas by the integrator, and by the network that replaces it.
        {"name": "panorama_plain", "kind": "panorama_plain", "views": 8, "w": 1920, "h": 1080},
        {"name": "panorama_network", "kind": "panorama_net", "views": 16, "w": 1920, "h": 1080,
         "network": "f16_gate"},
        # One optimizer step at the batch size training uses.
        {"name": "train_step_8192", "kind": "train_step", "batch": 8192, "network": "bf16_silu"},
        # Regenerating the material's textures after a parameter edit, default sizes.
        {"name": "textures_default", "kind": "textures", "cloud_map": 512, "detail": 128, "displacement": 128,
         "worley": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["lut_set", "sky_frame", "lut_batch", "cloud_shadow", "raymarch", "cloud_frame", "path_trace",
                       "path_trace_mat", "panorama_plain", "panorama_net", "train_step", "textures"])
    c = {"kind": kind}
    if kind == "lut_set":
        c.update(tw=_log_int(rng, 64, 256), th=_log_int(rng, 16, 64), mw=rng.randint(16, 32), mh=rng.randint(16, 32),
                 sw=_log_int(rng, 48, 256), sh=_log_int(rng, 32, 128), aw=rng.randint(8, 32), ah=rng.randint(8, 32),
                 ad=rng.randint(8, 32))
    elif kind == "sky_frame":
        c.update(sw=_log_int(rng, 64, 200), sh=_log_int(rng, 64, 128), aw=rng.randint(16, 32),
                 ah=rng.randint(16, 32), ad=rng.randint(16, 32), env=rng.choice([32, 64, 128]))
    elif kind == "lut_batch":
        c.update(sets=_log_int(rng, 3, 200), suns=rng.randint(1, 8))
    elif kind == "cloud_shadow":
        c.update(w=_log_int(rng, 640, 2560), h=_log_int(rng, 360, 1440), map=_log_int(rng, 200, 640),
                 material=rng.choice(["worley", "default1", "default0"]))
    elif kind == "raymarch":
        c.update(w=_log_int(rng, 320, 1920), h=_log_int(rng, 180, 1080),
                 material=rng.choice(["worley", "default1", "default0"]))
    elif kind == "cloud_frame":
        c.update(w=4 * _log_int(rng, 160, 640), h=4 * _log_int(rng, 90, 360),
                 material=rng.choice(["worley", "default1"]))
    elif kind == "path_trace":
        c.update(w=_log_int(rng, 160, 900), h=_log_int(rng, 120, 900), grid=rng.randint(100, 400),
                 brick=rng.choice([4, 8, 16, 32]))
    elif kind == "path_trace_mat":
        c.update(w=_log_int(rng, 96, 321), h=_log_int(rng, 64, 181), material=rng.choice(["worley", "default1"]))
    elif kind == "panorama_plain":
        c.update(views=rng.randint(1, 8), w=_log_int(rng, 300, 1920), h=_log_int(rng, 150, 1080))
    elif kind == "panorama_net":
        c.update(views=rng.randint(1, 16), w=_log_int(rng, 300, 1920), h=_log_int(rng, 150, 1080),
                 network=rng.choice(["f16_gate", "bf16_silu"]))
    elif kind == "train_step":
        c.update(batch=_log_int(rng, 500, 32768), network=rng.choice(["f16_gate", "bf16_silu"]))
    else:
        c.update(cloud_map=rng.choice([256, 512]), detail=rng.choice([64, 128]), displacement=rng.choice([128, 256]),
                 worley=rng.choice([16, 32, 64]))
    return c


# ---------------------------------------------------------------------------
# What a program has in hand before the call
# ---------------------------------------------------------------------------
_shared = {}


def _context():
    if "ctx" not in _shared:
        _shared["ctx"] = Context(0)
    return _shared["ctx"]


class _Memory:
    """Device memory the library allocated, for torch to view; `owner` keeps it alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (int(ptr), False),
                                         "version": 2}


def _view(owner, ptr, shape, typestr):
    return torch.as_tensor(_Memory(owner, ptr, shape, typestr), device="cuda")


def _buffer(buf, shape, typestr):
    return _view(buf, buf.ptr, shape, typestr)


def _earth(rng):
    """The 100 km Earth with the haze and ozone of some day."""
    p = presets.earth_100km()
    mie = rng.uniform(0.5, 2.0)
    p.mie_scattering_scale *= mie
    p.mie_absorption_scale *= mie
    p.ozone_absorption_scale *= rng.uniform(0.8, 1.2)
    return p


def _render_parameters(rng, theta_max=95.0):
    cam = presets.bench_camera(altitude_km=float(rng.uniform(0.2, 3.0)))
    return AtmosphereRenderParameters(
        sun_direction_theta=float(rng.uniform(0.0, theta_max)), sun_direction_phi=180.0, sky_view_lut_steps=30.0,
        aerial_perspective_lut_steps=AP_STEPS, aerial_perspective_lut_max_distance=AP_DISTANCE,
        camera_position=cam.position, view_projection=cam.view_projection())


def _cloud_workload(material, rng):
    w = presets.cloud_workload_config2() if material == "worley" else presets.cloud_workload()
    if material == "default0":
        m = cl.VolumetricCloudDefaultMaterial0(
            **{f: getattr(w["material"], f) for f in cl.DefaultMaterialCommon.__dataclass_fields__})
        m.detail_param = (0.8, 0.1)
        w["material"] = m
    w["weather_seeds"] = (int(rng.integers(1 << 30)), int(rng.integers(1 << 30)))
    w["blue_noise_seed"] = int(rng.integers(1 << 30))
    w["sun_theta"] = float(rng.uniform(60.0, 75.0))
    return w


def _cloud_scene(case, rng):
    ctx = _context()
    scene = CloudScene(ctx, case["w"], case["h"], workload=_cloud_workload(case["material"], rng))
    sun = np.array(scene.renderer.buffer.sun_direction[:], np.float32)
    cl.cloud_shadow_matrices(scene.cloud, scene.camera, scene.earth.bottom_radius, sun, scene.common)
    cl.cloud_reproject_matrix(scene.camera, scene.earth.bottom_radius, scene.common)
    return scene


def _batch_views(case, rng):
    """The batched workload's sets and views with this seed's coefficients."""
    cam = presets.bench_camera()
    vp = cam.view_projection()
    sets, views = [], []
    for s in range(case["sets"]):
        p = presets.earth_100km()
        ray, mie = rng.uniform(0.25, 4.0, 2)
        p.rayleigh_scattering_scale *= ray
        p.mie_scattering_scale *= mie
        p.mie_absorption_scale *= mie
        p.rayleigh_exponential_distribution *= rng.uniform(0.5, 2.0)
        p.mie_exponential_distribution *= rng.uniform(0.5, 2.0)
        p.bottom_radius = rng.uniform(3000.0, 7000.0)
        # The sizes go round in order, so that every seed's batch is the same amount of work.
        sv = presets.BATCH_SKY_VIEW_SIZES[s % 3]
        sets.append((p.buffer_data(), presets.BATCH_TRANSMITTANCE_SIZES[(s // 3) % 2], (32, 32)))
        for k in range(case["suns"]):
            rp = AtmosphereRenderParameters(
                sun_direction_theta=float(95.0 * (k + rng.random()) / case["suns"]), sun_direction_phi=180.0,
                sky_view_lut_steps=30.0, aerial_perspective_lut_steps=AP_STEPS,
                aerial_perspective_lut_max_distance=AP_DISTANCE, camera_position=cam.position, view_projection=vp)
            views.append((s, rp.buffer_data(p.bottom_radius), sv))
    return sets, views


def _panoramas(case, seed):
    ctx = _context()
    scales, views = sg.evaluation_views(case["views"], seed=seed % (1 << 31), max_altitude=10.0,
                                        max_sun_zenith_deg=90.0)
    atm = sg.SkyAtmospheres(ctx, scales)
    return atm, sg.SkyPanoramas(ctx, atm, views, case["w"], case["h"])


def _network(network, seed):
    """Weights of the size and spread a trained network has: twice Glorot's, so that the hidden layers
    use the activation's curved range, around the sky's mean log radiance."""
    p = 2.0 * sg.init_params(seed % (1 << 31))
    p[13184:13187] = [-4.2, -3.6, -3.0]
    return sg.SkySurrogate(_context(), p, network=network)


def prepare(case, seed):
    kind, ctx, rng = case["kind"], _context(), np.random.default_rng(seed)
    s = {"kind": kind}
    if kind == "lut_set":
        sizes = {"transmittance": (case["tw"], case["th"]), "multiscattering": (case["mw"], case["mh"]),
                 "sky_view": (case["sw"], case["sh"]), "aerial_perspective": (case["aw"], case["ah"], case["ad"])}
        luts = LutSet(ctx, sizes)
        s.update(luts=luts, earth=_earth(rng), render=_render_parameters(rng))
        sv, ap = (case["sh"], case["sw"], 4), (case["ad"], case["ah"], case["aw"], 4)
        s["out"] = [_buffer(luts.T, (case["th"], case["tw"], 4), "<f4"),
                    _buffer(luts.MS, (case["mh"], case["mw"], 4), "<f4"), _buffer(luts.SV_L, sv, "<f4"),
                    _buffer(luts.SV_T, sv, "<f4"), _buffer(luts.AP_L, ap, "<f4"), _buffer(luts.AP_T, ap, "<f4")]
    elif kind == "sky_frame":
        atm = Atmosphere(ctx)
        rend = AtmosphereRenderer(ctx, AtmosphereRenderInitParameters(
            sky_view_lut_size=(case["sw"], case["sh"]), aerial_perspective_lut_size=(case["aw"], case["ah"]),
            aerial_perspective_lut_depth=case["ad"]))
        env, ibl = EnvironmentLuminance(ctx, case["env"]), IBL(ctx, case["env"])
        s.update(atm=atm, rend=rend, env=env, ibl=ibl, earth=_earth(rng), render=_render_parameters(rng, 85.0))
        sv, ap = (case["sh"], case["sw"], 4), (case["ad"], case["ah"], case["aw"], 4)
        s["out"] = [_buffer(atm.transmittance_texture, (64, 256, 4), "<f4"),
                    _buffer(atm.multiscattering_texture, (32, 32, 4), "<f4"),
                    _buffer(rend.sky_view_luminance_texture, sv, "<f4"),
                    _buffer(rend.sky_view_transmittance_texture, sv, "<f4"),
                    _buffer(rend.aerial_perspective_luminance_texture, ap, "<f4"),
                    _buffer(rend.aerial_perspective_transmittance_texture, ap, "<f4"),
                    _buffer(env.texture, (cube_texels(env.width, env.levels), 4), "<f2"),
                    _buffer(ibl.env_radiance_sh_buffer, (9, 4), "<f4"),
                    _buffer(ibl.prefiltered_radiance_texture, (cube_texels(ibl.resolution, ibl.roughness_count), 4),
                            "<f2")]
    elif kind == "lut_batch":
        sets, views = _batch_views(case, rng)
        batch = LutBatch(ctx, sets, views)
        s.update(batch=batch, sets=sets, views=views)

        def pool(ptrs, sizes):  # one tensor over the items of a pool, which lie back to back
            n = sum(w * h for w, h in sizes)
            assert ptrs[-1] + sizes[-1][0] * sizes[-1][1] * 16 == ptrs[0] + 16 * n
            return _view(batch, ptrs[0], (n, 4), "<f4")

        ends = lambda n: [0, n - 1] if n > 1 else [0]  # noqa: E731
        sp = [batch.set_output_ptrs(i) for i in ends(len(sets))]
        vp = [batch.view_output_ptrs(i) for i in ends(len(views))]
        s["out"] = [pool([p[0] for p in sp], [z[1] for z in sets]), pool([p[1] for p in sp], [z[2] for z in sets]),
                    pool([p[0] for p in vp], [z[2] for z in views]), pool([p[1] for p in vp], [z[2] for z in views])]
    elif kind == "cloud_shadow":
        scene = _cloud_scene(case, rng)
        shadow = cl.CloudShadow(ctx, (case["w"], case["h"]), map_size=(case["map"], case["map"]))
        s.update(scene=scene, shadow=shadow)
        n, (fw, fh, fd) = case["map"], shadow.froxel_size
        s["raw"] = {b.ptr: _buffer(b, (n, n, 2), "<f4") for b in shadow.raw}
        s["out"] = [_buffer(shadow.blurred, (n, n, 2), "<f4"), _buffer(shadow.froxel, (fd, fh, fw), "<i2")]
    elif kind == "raymarch":
        scene = _cloud_scene(case, rng)
        s.update(scene=scene)
        s["out"] = [_buffer(scene.out_rgba, (case["h"], case["w"], 4), "<f2"),
                    _buffer(scene.out_dist, (case["h"], case["w"]), "<f4")]
    elif kind == "cloud_frame":
        scene = _cloud_scene(case, rng)
        w, h = case["w"], case["h"]
        rec = cl.CloudReconstruction(ctx, (w, h))
        depth = presets.synthetic_depth_buffer(scene.common.uLinearDepthParam, w, h, seed % (1 << 31))
        hdr = np.concatenate([np.full((h, w, 3), 2.0, np.float16), np.ones((h, w, 1), np.float16)], -1)
        s.update(scene=scene, rec=rec, depth=ctx.upload(depth), hdr=ctx.upload(hdr))
        s["history"] = {b.ptr: _buffer(b, (h // 2, w // 2, 4), "<f2") for b in rec.reconstruct}
        s["out"] = [_buffer(s["hdr"], (h, w, 4), "<f2")]
    elif kind == "path_trace":
        w = presets.path_trace_workload()
        w["grid_dims"], w["brick"] = (case["grid"],) * 3, case["brick"]
        w["grid"].seed = seed % (1 << 31)
        scene = PathTraceScene(ctx, case["w"], case["h"], workload=w)
        s.update(scene=scene, tracer=scene.tracer)
        _tracer_outputs(s, case, seed)
    elif kind == "path_trace_mat":
        scene = _cloud_scene(case, rng)
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
        init = PathTracingInitParam(max_bounces=32, region_box_half_width=14.0)
        s["tracer"] = PathTracing(ctx, (case["w"], case["h"]), init, a.buffer, r.buffer, scene.common,
                                  scene.mat_block, i, scene.material.density, scene.model)
        s.update(scene=scene)
        _tracer_outputs(s, case, seed)
    elif kind == "panorama_plain":
        s["atm"], s["pano"] = _panoramas(case, seed)
        s["out"] = [_buffer(s["pano"].out, (case["views"], case["h"], case["w"], 4), "<f4")]
    elif kind == "panorama_net":
        s["atm"], s["pano"] = _panoramas(case, seed)
        s["model"] = _network(case["network"], seed + 1)
        s["out"] = [_buffer(s["pano"].out, (case["views"], case["h"], case["w"], 4), "<f4"),
                    _buffer(s["pano"].flags, (s["pano"].tiles * case["views"],), "<i4")]
    elif kind == "train_step":
        atm = sg.SkyAtmospheres(ctx, sg.draw_scales(16, seed % (1 << 31)))
        data = sg.SkyTrainingSet(ctx, atm, 4 * case["batch"], seed=seed % (1 << 31), altitude_range=(0.0, 10.0),
                                 mu_sun_range=(0.0, 1.0))
        model = _network(case["network"], seed + 1)
        s.update(data=data, model=model, batch=case["batch"])
        p = (sg.PARAMS,)
        s["out"] = [_buffer(model.params, p, "<f4"), _buffer(model.grad, p, "<f4"), _buffer(model.loss, (1,), "<f4"),
                    _buffer(model.m, p, "<f4"), _buffer(model.v, p, "<f4")]
    elif kind == "textures":
        m = presets.cloud_workload_config2()["material"]
        for info in (m.cloud_map_density, m.cloud_map_height, m.detail_perlin, m.detail_worley, m.displacement_perlin,
                     m.worley):
            info.seed = int(rng.integers(1 << 30))
        tex = cl.CloudTextures(ctx, case["cloud_map"], case["detail"], case["displacement"], case["worley"])
        s.update(material=m, textures=tex)
        s["out"] = [_buffer(b, (b.nbytes,), "|u1") for b in (tex.cloud_map, tex.detail, tex.displacement, tex.worley,
                                                             tex.cloud_map_cells, tex.detail_cells, tex.worley_cells)]
    return s


def _tracer_outputs(s, case, seed):
    ctx, (w, h) = _context(), (case["w"], case["h"])
    # The HDR image the display pass composites over: a sky gradient.
    sky = np.linspace(0.2, 1.0, h, dtype=np.float16)[:, None, None] * np.ones((1, w, 4), np.float16)
    s["display"] = ctx.upload(sky)
    s["out"] = [_buffer(s["tracer"].accumulation, (h, w, 4), "<f4"), _buffer(s["tracer"].rendered_mask, (h, w), "|u1"),
                _buffer(s["display"], (h, w, 4), "<f2")]


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s):
    kind = s["kind"]
    if kind == "lut_set":
        s["luts"].build(s["earth"], s["render"])
    elif kind == "sky_frame":
        s["atm"].update_luts(s["earth"])
        s["rend"].render(s["atm"], s["earth"], s["render"])
        s["env"].update(s["atm"], s["rend"])
        s["ibl"].precompute(s["env"])
    elif kind == "lut_batch":
        s["batch"].launch()
    elif kind == "cloud_shadow":
        c = s["scene"]
        s["shadow"].render(c.common, c.mat_block, c.blue_noise, c.blue_noise_host.shape[0])
        return [s["raw"][s["shadow"].raw[0].ptr]] + s["out"]
    elif kind == "raymarch":
        s["scene"].run()
    elif kind == "cloud_frame":
        c, a, r = s["scene"], s["scene"].atmosphere, s["scene"].renderer
        cl.bind_cloud_phase(c.ctx, c.phase)
        s["rec"].render(a.buffer, c.common, c.cloud_block, c.mat_block, a.transmittance_texture, a.transmittance_size,
                        r.aerial_perspective_luminance_texture, r.aerial_perspective_transmittance_texture,
                        r.init.aerial_perspective_lut_size + (r.init.aerial_perspective_lut_depth,), c.blue_noise,
                        c.blue_noise_host.shape[0], s["depth"], s["hdr"])
        return s["out"] + [s["history"][s["rec"].reconstruct[1].ptr]]
    elif kind in ("path_trace", "path_trace_mat"):
        s["tracer"].render(s["display"])
    elif kind == "panorama_plain":
        s["pano"].render_plain()
    elif kind == "panorama_net":
        s["pano"].render_surrogate(s["model"], tolerance=1e30)
    elif kind == "train_step":
        d, m, n = s["data"], s["model"], s["batch"]
        k = m.step % (d.n // n)
        m.gradient(d.features.ptr + k * n * 32, d.targets.ptr + k * n * 12, n, 1.0 / (3.0 * n),
                   d.weights.ptr + k * n * 4)
        m.adam(2e-3)
    else:
        s["textures"].generate(s["material"])
    return s["out"]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
# FP32 operations per integrator step, per raymarched pixel and per path-traced pixel, from
# profiles/ (measured operations over the work counted there); per noise texel from the
# generators' definition (8 octaves of 8 gradients or 27 feature points).
STEP_FLOP = 211.0
RAYMARCH_STEPS = 17.0
SHADOW_TEXEL_FLOP = 1500.0


def work(case):
    k = case["kind"]
    if k in ("lut_set", "sky_frame"):
        t = case["tw"] * case["th"] if k == "lut_set" else 256 * 64
        m = case["mw"] * case["mh"] if k == "lut_set" else 32 * 32
        sv, ap = case["sw"] * case["sh"], case["aw"] * case["ah"] * case["ad"]
        b, f = 16 * (t + m + 2 * sv + 2 * ap), STEP_FLOP * (40 * t + 64 * 30 * m + 30 * sv + 51 * ap)
        if k == "sky_frame":
            cube = 6 * case["env"] ** 2
            b, f = b + 2 * 8 * cube * 4 / 3, f + cube * (150.0 + 16 * 400.0)
        return {"bytes": b, "flops": f}
    if k == "lut_batch":
        sv = sum(w * h for w, h in (presets.BATCH_SKY_VIEW_SIZES[i % 3] for i in range(case["sets"]))) * case["suns"]
        t = sum(w * h for w, h in (presets.BATCH_TRANSMITTANCE_SIZES[(i // 3) % 2] for i in range(case["sets"])))
        m = 1024 * case["sets"]
        return {"bytes": 16 * (t + m + 2 * sv), "flops": STEP_FLOP * (40 * t + 64 * 30 * m + 30 * sv)}
    if k == "cloud_shadow":
        n, f = case["map"] ** 2, (case["w"] // 12) * (case["h"] // 12) * 128
        return {"bytes": 24 * n + 2 * f, "flops": SHADOW_TEXEL_FLOP * n + 40.0 * f}
    if k in ("raymarch", "cloud_frame"):
        px = case["w"] * case["h"]
        if k == "raymarch":
            return {"bytes": 12 * px, "flops": 210.0 * RAYMARCH_STEPS * px}
        return {"bytes": 35.75 * px, "flops": 210.0 * RAYMARCH_STEPS * px / 16 + 300.0 * px / 4}
    if k == "path_trace":  # 114 lookups, 118 brick crossings and 4 vertices a pixel on the 512^3 grid
        px = case["w"] * case["h"]
        return {"bytes": px * (32 + 16 + 114 * 16 + 118 * 4), "flops": px * (114 * 60.0 + 118 * 20.0 + 4 * 600.0)}
    if k == "path_trace_mat":
        px = case["w"] * case["h"]
        return {"bytes": px * 48, "flops": px * 600 * 250.0}
    if k == "panorama_plain":
        px = case["views"] * case["w"] * case["h"]
        return {"bytes": 16 * px, "flops": STEP_FLOP * 30 * px}
    if k == "panorama_net":
        px = case["views"] * case["w"] * case["h"]
        return {"bytes": 16 * px, "flops": 25856.0 * px + STEP_FLOP * 30 * px / 64}
    if k == "train_step":
        return {"bytes": case["batch"] * 48 + sg.PARAMS * 28, "flops": 3 * 25856.0 * case["batch"]}
    cm, d, di, w = case["cloud_map"] ** 2, case["detail"] ** 3, case["displacement"] ** 2, case["worley"] ** 3
    return {"bytes": cm * (8 / 3 + 8) + (d + w) * (8 / 7 + 8) + di * 16 / 3,
            "flops": 8 * 100.0 * (cm + d + 4 * di) + 8 * 27 * 10.0 * (cm + d + w)}


def tolerance(case):
    """About four times what two builds that round differently (contracted and uncontracted
    multiply-adds, reciprocals for divisions) differ by; at most 0.02."""
    k = case["kind"]
    if k in ("lut_set", "lut_batch", "panorama_plain"):
        # 2e-7 to 5e-7 as a rule; 3e-5 where a row of texels lies on the horizon.
        return {"rel": 1e-4, "max": 2e-3}
    if k == "sky_frame":  # the FP16 cubes: an FP16 unit where a texel lies between two
        return {"rel": 1e-4, "max": 0.03}
    if k == "cloud_shadow":  # the FP32 maps; the 16-bit froxel within the share of ties
        return {"rel": 1e-3, "max": 0.08, "differ": 0.01}
    if k in ("raymarch", "cloud_frame", "path_trace", "path_trace_mat"):
        # Rays and paths that end, light or turn at a threshold: one rounding moves a whole step,
        # or makes another sample of the pixel.
        return {"rel": 2e-2, "max": 0.99}
    if k == "panorama_net":  # 16-bit operands of four layers
        return {"rel": 2e-3, "max": 0.1, "differ": 0.0}
    if k == "train_step":  # 16-bit operands; Adam's first step is the gradient's sign
        return {"rel": 2e-3, "max": 0.1}
    return "exact"


# ---------------------------------------------------------------------------
# The atmosphere integrator and the surrogate in 64 bits
# ---------------------------------------------------------------------------
def _vec(v):
    return torch.tensor([float(x) for x in v][:3], dtype=torch.float64, device="cuda")


class _Atm:
    def __init__(self, b):
        self.solar, self.albedo = _vec(b.solar_illuminance), _vec(b.ground_albedo)
        self.ray, self.mie = _vec(b.rayleigh_scattering), _vec(b.mie_scattering)
        self.mie_ext, self.ozone = self.mie + _vec(b.mie_absorption), _vec(b.ozone_absorption)
        self.ihr = float(b.inv_rayleigh_exponential_distribution)
        self.ihm = float(b.inv_mie_exponential_distribution)
        self.oc, self.iow = float(b.ozone_center_altitude), float(b.inv_ozone_width)
        self.rb, self.rt, self.g = float(b.bottom_radius), float(b.top_radius), float(b.mie_phase_g)
        self.sun = float(b.sun_angular_radius)
        self.t_steps, self.ms_steps = float(b.transmittance_steps), float(b.multiscattering_steps)
        self.mask = float(b.multiscattering_mask)
        self.H = math.sqrt(self.rt * self.rt - self.rb * self.rb)

    def densities(self, alt):
        return (torch.exp(-alt * self.ihr).clamp(max=1.0), torch.exp(-alt * self.ihm).clamp(max=1.0),
                (1.0 - (alt - self.oc).abs() * self.iow).clamp(min=0.0))


def _lin(n):
    return torch.arange(n, dtype=torch.float64, device="cuda") / (n - 1)


def _bilinear(lut, fx, fy):
    h, w = lut.shape[:2]
    fx, fy = fx.clamp(0, w - 1), fy.clamp(0, h - 1)
    x0, y0 = fx.floor().long(), fy.floor().long()
    x1, y1 = (x0 + 1).clamp(max=w - 1), (y0 + 1).clamp(max=h - 1)
    ax, ay = (fx - x0)[..., None], (fy - y0)[..., None]
    return (1 - ay) * ((1 - ax) * lut[y0, x0] + ax * lut[y0, x1]) + ay * ((1 - ax) * lut[y1, x0] + ax * lut[y1, x1])


def _counter(steps, start=0.5):
    i, out = start, []
    while i < steps:
        out.append(i)
        i += 1.0
    return out


def _transmittance(A, w, h):
    x_mu, rho = _lin(w)[None, :], (A.H * _lin(h))[:, None]
    r = (rho * rho + A.rb * A.rb).sqrt()
    d_min, d_max = A.rt - r, rho + A.H
    d = d_min + x_mu * (d_max - d_min)
    mu = torch.where(d == 0, torch.ones_like(d), (A.H * A.H - rho * rho - d * d) / (2 * r * d)).clamp(-1, 1)
    dist = (-r * mu + (r * r * (mu * mu - 1) + A.rt * A.rt).clamp(min=0).sqrt()).clamp(min=0)
    dx, od = dist / A.t_steps, 0.0
    for i in _counter(A.t_steps):
        di = i * dx
        dr, dm, do = A.densities((di * di + 2 * r * mu * di + r * r).sqrt() - A.rb)
        od = od + A.ray * dr[..., None] + A.mie_ext * dm[..., None] + A.ozone * do[..., None]
    return torch.exp(-od * dx[..., None])


def _sun_visibility(A, T, r, mu_s):
    h, w = T.shape[:2]
    rho = (r * r - A.rb * A.rb).clamp(min=0).sqrt()
    d = (-r * mu_s + (r * r * (mu_s * mu_s - 1) + A.rt * A.rt).clamp(min=0).sqrt()).clamp(min=0)
    d_min, d_max = A.rt - r, rho + A.H
    t = _bilinear(T, (d - d_min) / (d_max - d_min) * (w - 1), rho / A.H * (h - 1))
    e = A.rb / r * A.sun
    s = ((mu_s + rho / r + e) / (2 * e)).clamp(0, 1)
    return t * (s * s * (3 - 2 * s))[..., None]


def _ground(A, r, mu):
    """(hits the ground, distance to it or to the top)."""
    disc = r * r * (mu * mu - 1) + A.rb * A.rb
    hit = (mu < 0) & (disc >= 0)
    bottom = (-r * mu - disc.clamp(min=0).sqrt()).clamp(min=0)
    top = (-r * mu + (r * r * (mu * mu - 1) + A.rt * A.rt).clamp(min=0).sqrt()).clamp(min=0)
    return hit, torch.where(hit, bottom, top), top


def _scatter(A, T, MS, r, mu, mu_s0, nu, dist, steps):
    """(luminance, transmittance, multiple-scattering transfer); MS None: the isotropic variant."""
    dx = dist / steps
    if MS is None:
        rp = mp = torch.full_like(nu, 1 / (4 * math.pi))
    else:
        rp = 3 / (16 * math.pi) * (1 + nu * nu)
        g = A.g
        mp = 3 / (8 * math.pi) * (1 - g * g) / (2 + g * g) * (1 + nu * nu) / (1 + g * g - 2 * g * nu) ** 1.5
    L, F = 0.0, 0.0
    Tr = torch.ones(dist.shape + (3,), dtype=torch.float64, device="cuda")
    for i in _counter(steps):
        d = i * dx
        rd = (d * d + 2 * r * mu * d + r * r).clamp(min=0).sqrt()
        alt, mu_s = rd - A.rb, (r * mu_s0 + d * nu) / rd
        dr, dm, do = (x[..., None] for x in A.densities(alt))
        sr, sm = A.ray * dr, A.mie * dm
        ext = sr + A.mie_ext * dm + A.ozone * do
        Li = (sr * rp[..., None] + sm * mp[..., None]) * _sun_visibility(A, T, rd, mu_s)
        if MS is not None:
            mh, mw = MS.shape[:2]
            Li = (Li + A.mask * _bilinear(MS, (mu_s * 0.5 + 0.5) * (mw - 1), alt / (A.rt - A.rb) * (mh - 1)) *
                  (sr + sm)) * A.solar
        k = Tr * -torch.expm1(-ext * dx[..., None]) / ext
        L, F, Tr = L + k * Li, F + k * (sr + sm), Tr * torch.exp(-ext * dx[..., None])
    return L, Tr, F


def _multiscattering(A, T, w, h):
    alt = (_lin(h) * (A.rt - A.rb))[:, None, None]
    mu_s = (_lin(w) * 2 - 1)[None, :, None]
    k = torch.arange(64, device="cuda")
    mu = (1 - 2 * (0.5 + (k // 8).double()) / 8)[None, None, :]
    phi = 2 * math.pi * (0.5 + (k % 8).double()) / 8
    nu = mu * mu_s + phi.sin() * (1 - mu * mu).sqrt() * (1 - mu_s * mu_s).clamp(min=0).sqrt()
    r = alt + A.rb
    r, mu, mu_s, nu = torch.broadcast_tensors(r, mu, mu_s, nu)
    # A ray along the ground at altitude 0 has its sign of mu alone to tell whether it hits.
    hit, dist, _ = _ground(A, r, mu)
    L, Tr, F = _scatter(A, T, None, r, mu, mu_s, nu, dist, A.ms_steps)
    mu_g = (r * mu_s + dist * nu) / A.rb
    ground = Tr * (mu_g.clamp(0, 1) / math.pi)[..., None] * A.albedo * _sun_visibility(A, T, torch.full_like(r, A.rb),
                                                                                       mu_g)
    L = torch.where(hit[..., None], L + ground, L)
    return L.mean(2) / (1 - F.mean(2))


def _rgba(x, a):
    return torch.cat([x, torch.full(x.shape[:-1] + (1,), a, dtype=x.dtype, device=x.device)], -1)


def _frame(R):
    return {k: _vec(getattr(R, k + "_direction")) for k in ("sun", "up", "right", "front")}


def _sky_view(A, R, T, MS, w, h):
    f, r = _frame(R), float(R.camera_earth_center_distance)
    down = math.acos(math.sqrt(r * r - A.rb * A.rb) / r)
    up = math.pi - down
    xl, x = _lin(h)[:, None], _lin(w)[None, :]
    lat = torch.where(xl < 0.5, up * (1 - (1 - 2 * xl) ** 2), up + down * (2 * xl - 1) ** 2)
    cos_lat, sin_lat = lat.cos(), lat.sin().clamp(0, 1)
    cos_lon, sin_lon = 1 - 2 * x * x, (2 * x * (1 - x * x).clamp(min=0).sqrt()).clamp(0, 1)
    cos_lat, sin_lat, cos_lon, sin_lon = torch.broadcast_tensors(cos_lat, sin_lat, cos_lon, sin_lon)
    view = (f["up"] * cos_lat[..., None] + f["front"] * (sin_lat * cos_lon)[..., None] +
            f["right"] * (sin_lat * sin_lon)[..., None])
    rr = torch.full_like(cos_lat, r)
    _, dist, _ = _ground(A, rr, cos_lat)
    L, Tr, _ = _scatter(A, T, MS, rr, cos_lat, torch.full_like(rr, float(f["sun"] @ f["up"])), view @ f["sun"], dist,
                        float(R.sky_view_lut_steps))
    return _rgba(L, 0.0), _rgba(Tr, 0.0)


def _aerial(A, R, T, MS, w, h, d):
    f, r = _frame(R), float(R.camera_earth_center_distance)
    z, y, x = torch.meshgrid(_lin(d), _lin(h), _lin(w), indexing="ij")
    m = torch.tensor([float(v) for v in R.inv_view_projection], dtype=torch.float64, device="cuda").reshape(4, 4)
    p = torch.stack([2 * x - 1, 2 * y - 1, torch.zeros_like(x), torch.ones_like(x)], -1) @ m
    view = p[..., :3] / p[..., 3:] - _vec(R.camera_position)
    view = view / view.norm(dim=-1, keepdim=True)
    mu, rr = view @ f["up"], torch.full_like(x, r)
    march = z * z * float(R.aerial_perspective_lut_max_distance)
    hit, _, top = _ground(A, rr, mu)
    dist = torch.where(hit, march, torch.minimum(march, top))
    L, Tr, _ = _scatter(A, T, MS, rr, mu, torch.full_like(x, float(f["sun"] @ f["up"])), view @ f["sun"], dist,
                        float(R.aerial_perspective_lut_steps))
    return _rgba(L, 0.0), _rgba(Tr, 0.0)


def _mlp(p, x, network):
    """Log radiance [n, 3] of features x [n, 7]."""
    at = 0
    for k, n in sg.LAYERS:
        w, b = p[at:at + n * k].reshape(n, k), p[at + n * k:at + n * k + n]
        at += n * k + n
        x = x @ w.T + b
        if n == 64:
            t = (x / 6 + 0.5).clamp(0, 1)
            x = x * torch.sigmoid(x) if network == "bf16_silu" else x * t * t * (3 - 2 * t)
    return x


def _sphere(s, view):
    """Zenith cosines [h, 1] and azimuths from the sun [1, w] of a panorama's pixels."""
    p = s["pano"]
    mu = torch.cos(math.pi * (torch.arange(p.height, dtype=torch.float64, device="cuda") + 0.5) / p.height)[:, None]
    dphi = (2 * math.pi * (torch.arange(p.width, dtype=torch.float64, device="cuda") + 0.5) / p.width - math.pi).abs()
    return torch.broadcast_tensors(mu, dphi[None, :])


def _plain_view(s, view):
    v, atm = s["pano"].views_host[view], s["atm"]
    A = _Atm(atm.blocks[int(v["atmosphere"])])
    T = _transmittance(A, 256, 64)
    MS = _multiscattering(A, T, 32, 32)
    mu, dphi = _sphere(s, view)
    r, mu_s = torch.full_like(mu, A.rb + float(v["altitude"])), torch.full_like(mu, float(v["mu_sun"]))
    nu = mu * mu_s + ((1 - mu * mu) * (1 - mu_s * mu_s)).clamp(min=0).sqrt() * dphi.cos()
    _, dist, _ = _ground(A, r, mu)
    return _scatter(A, T, MS, r, mu, mu_s, nu, dist, float(atm.luts.steps))[0]


def _network_view(s, view, network):
    v, atm = s["pano"].views_host[view], s["atm"]
    mu, dphi = _sphere(s, view)
    alt, mu_s = float(v["altitude"]), float(v["mu_sun"])
    r = 6360.0 + alt
    down = math.acos(math.sqrt(alt * (r + 6360.0)) / r)
    up, lat = math.pi - down, torch.acos(mu)
    x_lat = torch.where(lat < up, 0.5 - 0.5 * (1 - lat / up).clamp(min=0).sqrt(),
                        0.5 + 0.5 * ((lat - up) / down).clamp(min=0).sqrt())
    nu = mu * mu_s + (1 - mu * mu).clamp(min=0).sqrt() * math.sqrt(max(0.0, 1 - mu_s * mu_s)) * dphi.cos()
    scales = np.log(atm.scales[int(v["atmosphere"])]) / math.log(4.0)
    const = [2 * math.sqrt(alt / atm.thickness) - 1, math.copysign(math.sqrt(abs(mu_s)), mu_s)]
    full = lambda c: torch.full_like(mu, float(c))  # noqa: E731
    x = torch.stack([full(const[0]), 2 * x_lat - 1, full(const[1]), nu] + [full(c) for c in scales], -1)
    p = torch.from_numpy(s["model"].host_params()).double().cuda()
    out = torch.exp(_mlp(p, x.reshape(-1, 7), network)).reshape(mu.shape + (3,))
    # The probes of each 16 x 16 tile keep the integrator's value.
    plain, (h, w) = _plain_view(s, view), mu.shape
    ys = torch.tensor(sorted({min(t + o, h - 1) for t in range(0, h, 16) for o in (4, 12)}), device="cuda")
    xs = torch.tensor(sorted({min(t + o, w - 1) for t in range(0, w, 16) for o in (4, 12)}), device="cuda")
    out[ys[:, None], xs[None, :]] = plain[ys[:, None], xs[None, :]]
    return out


def exact(case, seed):
    k = case["kind"]
    if k not in ("lut_set", "sky_frame", "lut_batch", "panorama_plain", "panorama_net", "train_step"):
        return None
    if k == "lut_batch" and case["sets"] * case["suns"] > 200:
        return None
    s = prepare(case, seed)
    if k in ("lut_set", "sky_frame"):
        A, R = _Atm(s["earth"].buffer_data()), s["render"].buffer_data(s["earth"].bottom_radius)
        T = _transmittance(A, *((case["tw"], case["th"]) if k == "lut_set" else (256, 64)))
        MS = _multiscattering(A, T, *((case["mw"], case["mh"]) if k == "lut_set" else (32, 32)))
        out = [_rgba(T, 1.0), _rgba(MS, 1.0)]
        out += _sky_view(A, R, T, MS, case["sw"], case["sh"])
        out += _aerial(A, R, T, MS, case["aw"], case["ah"], case["ad"])
        return out + ([None] * 3 if k == "sky_frame" else [])
    if k == "lut_batch":
        luts = []
        for b, (tw, th), (mw, mh) in s["sets"]:
            A = _Atm(b)
            T = _transmittance(A, tw, th)
            luts.append((A, T, _multiscattering(A, T, mw, mh)))
        sky = [_sky_view(luts[i][0], R, luts[i][1], luts[i][2], *size) for i, R, size in s["views"]]
        flat = lambda xs: torch.cat([x.reshape(-1, 4) for x in xs])  # noqa: E731
        return [flat([_rgba(t, 1.0) for _, t, _ in luts]), flat([_rgba(m, 1.0) for _, _, m in luts]),
                flat([x[0] for x in sky]), flat([x[1] for x in sky])]
    if k == "panorama_plain":
        return [torch.stack([_rgba(_plain_view(s, v), 0.0) for v in range(case["views"])])]
    if k == "panorama_net":
        return [torch.stack([_rgba(_network_view(s, v, case["network"]), 0.0) for v in range(case["views"])]), None]
    m, d, n = s["model"], s["data"], case["batch"]
    p = torch.from_numpy(m.host_params()).double().cuda().requires_grad_(True)
    x = _buffer(d.features, (d.n, 8), "<f4")[:n, :7].double()
    t, w = (torch.from_numpy(a[:n]).double().cuda() for a in (d.targets_host, d.weights_host))
    loss = (w[:, None] * (_mlp(p, x, case["network"]) - t) ** 2).sum() / (3.0 * n)
    g, = torch.autograd.grad(loss, p)
    step = 2e-3 * g / (g.abs() + 1e-8)
    return [p.detach() - step, g, loss.detach()[None], 0.1 * g, 0.001 * g * g]
