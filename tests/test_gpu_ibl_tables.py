"""The prefilter's per-level sample tables and the environment pass's tiled mip chain at the sizes
where they can go wrong: faces smaller than a tile, of one texel and wider than the tail kernel's LDS,
every number of roughness levels, cubes smaller and larger than the prefiltered one.

The oracle sums in FP64; an FP16 result may lie on the other side of a rounding (one unit).  A sample
whose direction lies on a face edge within FP32 rounding (the texels of a face's diagonal have some that
do exactly) may take the other face's texel, the filter staying on a face: at coarse levels any other
value of the cube, with the sample's share of the sum, at most 1 / 16.5 (the cosines of roughness 1's 64
samples sum to 16.5, those of other levels to more).
"""

import numpy as np
import pytest

import oracle
from skyrendering_amd import _abi
from skyrendering_amd.ibl import cube_texels
from tests.test_gpu_ibl import _scene, _ulp_or_rel

pytestmark = pytest.mark.gpu


def _smooth_cube(w):
    c = (np.arange(w) + 0.5) / w * 2.0 - 1.0
    u, v = np.meshgrid(c, -c)
    one = np.ones_like(u)
    faces = [(one, v, -u), (-one, v, u), (u, one, -v), (u, -one, v), (u, v, one), (-u, v, -one)]
    d = np.stack([np.stack(f, -1) / np.linalg.norm(np.stack(f, -1), axis=-1, keepdims=True) for f in faces])
    k = np.array([[0.7, -0.2, 0.3], [0.1, 0.6, -0.5], [-0.4, 0.3, 0.6]])
    cube = np.zeros((cube_texels(w, int(np.log2(w)) + 1), 4), np.float16)
    cube[: 6 * w * w, :3] = (1.5 + np.sin(d @ k.T)).reshape(-1, 3)
    return oracle.cube_mips(cube.view(np.uint16), w)


@pytest.mark.parametrize("ew,pw,count", [(128, 64, 5), (16, 128, 8), (64, 1, 1), (64, 16, 5), (32, 2, 2), (128, 8, 3),
                                         (64, 256, 2)])
def test_prefilter_tables_match_oracle(ctx, ew, pw, count):
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
    print(f"{ok.mean():.6f} within 1 ulp / 1e-3, max rel {rel.max():.2e}")
    value = cube[:, :3].view(np.float16).astype(np.float64)
    assert ok.mean() >= 0.999 and rel.max() < (value.max() - value.min()) / 16.5 / value.min()
    e = np.abs(sh.download(np.float32, (9, 4)) - oracle.env_radiance_sh(cube, ew)[:, :4])[:, :3]
    assert e.max() < 1e-5 * np.abs(oracle.env_radiance_sh(cube, ew)[:, :3]).max()


@pytest.mark.parametrize("width", [1, 2, 8, 16, 32, 64, 512])
def test_environment_mips_bit_exact(ctx, width):
    _, _, env = _scene(ctx, width=width)
    gpu = env.texture.download(np.uint16, (cube_texels(width, env.levels), 4))
    assert gpu[: 6 * width * width, :3].any()
    assert np.array_equal(oracle.cube_mips(gpu, width), gpu)


def test_environment_mips_wider_than_the_tail(ctx):
    """4096: the first level below the tiles is 128 wide.  Levels 4 on are a 256 wide cube's chain."""
    _, _, env = _scene(ctx, width=4096)
    skip = cube_texels(4096, 4)
    n = cube_texels(4096, env.levels) - skip
    gpu = ctx.download_ptr(env.texture.ptr + 8 * skip, np.uint16, (n, 4))
    assert np.array_equal(oracle.cube_mips(gpu, 256), gpu)
