// The environment-luminance cube of the atmosphere renderer and its image-based-lighting
// precomputation:
//  - env_luminance_kernel: one thread per cube texel, the sky-view LUT pair looked up along
//    the texel's direction plus the lit ground (AtmosphereRenderer.glsl:248-275), stored as
//    RGBA16F (a = 0), and its tile's part of the mip chain, a 2x2 box per level
//    (glGenerateTextureMipmap, AtmosphereRenderer.cpp:242; the filter is the implementation's,
//    here a box); cube_mip_tail_kernel: the levels below a tile's, in one launch;
//  - prefilter_kernel: the 9 spherical-harmonic radiance coefficients (EnvRadianceSH.comp), one
//    workgroup per coefficient over 1024 stratified directions summed by the shader's halving
//    tree, and in the same launch the GGX-prefiltered radiance cube, one level per roughness
//    (PrefilterRadiance.comp, IBL.cpp:25-45).
#include "sky_env.h"

namespace skyhip {

int validate_atmosphere(const SkyhipAtmosphereBufferData* b);
int validate_render(const SkyhipAtmosphereRenderBufferData* b);
int validate_lut(const void* p, int w, int h, const char* what);

namespace {

__device__ inline ushort4 to_rgba16f(F3 c, float a) {
    ushort4 o;
    o.x = __half_as_ushort(__float2half_rn(c.x));
    o.y = __half_as_ushort(__float2half_rn(c.y));
    o.z = __half_as_ushort(__float2half_rn(c.z));
    o.w = __half_as_ushort(__float2half_rn(a));
    return o;
}

__device__ inline float h2f(uint16_t h) { return float(__builtin_bit_cast(_Float16, h)); }

bool is_pow2(int w) { return w > 0 && (w & (w - 1)) == 0; }
int log2i(int w) {
    int l = 0;
    while ((1 << (l + 1)) <= w) ++l;
    return l;
}

}  // namespace

// The mean of a 2x2 parent block per channel.
__device__ inline ushort4 box4(ushort4 a, ushort4 b, ushort4 c, ushort4 d) {
    ushort4 o;
    o.x = __half_as_ushort(__float2half_rn(((h2f(a.x) + h2f(b.x)) + (h2f(c.x) + h2f(d.x))) * 0.25f));
    o.y = __half_as_ushort(__float2half_rn(((h2f(a.y) + h2f(b.y)) + (h2f(c.y) + h2f(d.y))) * 0.25f));
    o.z = __half_as_ushort(__float2half_rn(((h2f(a.z) + h2f(b.z)) + (h2f(c.z) + h2f(d.z))) * 0.25f));
    o.w = __half_as_ushort(__float2half_rn(((h2f(a.w) + h2f(b.w)) + (h2f(c.w) + h2f(d.w))) * 0.25f));
    return o;
}

// A workgroup computes a tile of a face (16 x 16 texels, or the face if that is smaller) and, the
// tile's texels being in LDS, its part of the next levels down to one texel.  A launch of six
// workgroups, one a face, reading level 0 back for the whole chain took 10.3 us at 128^2; the levels left
// to it take 5.1 and the tiles 0.4 more.
constexpr int kEnvTile = 16, kEnvTileLog = 4;
__global__ __launch_bounds__(256) void env_luminance_kernel(AtmDev A, EnvFrame e, const float4* __restrict__ T,
                                                            int tw, int th, const float4* __restrict__ sv_l,
                                                            const float4* __restrict__ sv_t, int sw, int sh,
                                                            ushort4* __restrict__ out, int w, int tile_log) {
    __shared__ ushort4 s_a[kEnvTile * kEnvTile], s_b[kEnvTile * kEnvTile / 4];
    const int t = threadIdx.x, face = blockIdx.z;
    const int x0 = int(blockIdx.x) << tile_log, y0 = int(blockIdx.y) << tile_log;
    if (t < 1 << (2 * tile_log)) {
        const int x = x0 + (t & ((1 << tile_log) - 1)), y = y0 + (t >> tile_log);
        const ushort4 v =
            to_rgba16f(env_luminance(A, e, T, tw, th, sv_l, sv_t, sw, sh, cube_texel_dir(face, x, y, w)), 0.0f);
        out[(long long)face * w * w + (long long)y * w + x] = v;
        s_a[t] = v;
    }
    for (int l = 1; l <= tile_log; ++l) {  // a face of one texel is a chain of one level
        __syncthreads();
        const int lw = tile_log - l, wl = w >> l;
        const ushort4* src = (l & 1) ? s_a : s_b;
        ushort4* dst = (l & 1) ? s_b : s_a;
        if (t < 1 << (2 * lw)) {
            const int x = t & ((1 << lw) - 1), y = t >> lw, s = (2 * y << (lw + 1)) + 2 * x;
            const ushort4 v = box4(src[s], src[s + 1], src[s + (2 << lw)], src[s + (2 << lw) + 1]);
            out[cube_level_offset(w, l) + (long long)face * wl * wl + (long long)((y0 >> l) + y) * wl + (x0 >> l) + x] = v;
            dst[t] = v;
        }
    }
}

// Levels first_level .. levels - 1 of one face (blockIdx.x) in one workgroup: the first from the
// parent level in global memory, each later one from the previous level kept in LDS, every level
// also stored to the cube.  Levels after the first are at most kMipTailWidth / 2 wide (the launch's).
constexpr int kMipTailWidth = 64;
__global__ __launch_bounds__(1024) void cube_mip_tail_kernel(ushort4* cube, int w, int first_level, int levels) {
    __shared__ ushort4 s_a[kMipTailWidth * kMipTailWidth];
    __shared__ ushort4 s_b[(kMipTailWidth / 2) * (kMipTailWidth / 2)];
    const int face = blockIdx.x;
    for (int l = first_level; l < levels; ++l) {
        const int wl = max(w >> l, 1), wp = max(w >> (l - 1), 1);
        const bool from_global = l == first_level;
        const ushort4* gsrc = cube + cube_level_offset(w, l - 1) + (long long)face * wp * wp;
        const ushort4* lsrc = ((l - first_level) & 1) ? s_a : s_b;  // the previous level's buffer
        ushort4* ldst = ((l - first_level) & 1) ? s_b : s_a;
        ushort4* gdst = cube + cube_level_offset(w, l) + (long long)face * wl * wl;
        for (int t = threadIdx.x; t < wl * wl; t += 1024) {
            const int y = t / wl, x = t % wl;
            const int x0 = min(2 * x, wp - 1), x1 = min(2 * x + 1, wp - 1), y0 = min(2 * y, wp - 1),
                      y1 = min(2 * y + 1, wp - 1);
            const ushort4* src = from_global ? gsrc : lsrc;
            const ushort4 o = box4(src[y0 * wp + x0], src[y0 * wp + x1], src[y1 * wp + x0], src[y1 * wp + x1]);
            if (wl <= kMipTailWidth) ldst[t] = o;
            gdst[t] = o;
        }
        __syncthreads();
    }
}

// EnvRadianceSH.comp: coefficient `index` from 1024 directions on a 32 x 32 stratified grid
// (uniform in cos theta and phi, y up), each sample weighted 4 pi / 1024, summed by the shader's
// halving tree over the 1024 values (at half = 512, 256, ..., 1: s[i] += s[i + half]), the first
// level in registers: a 512-thread workgroup holds samples t and t + 512 in thread t.
__device__ inline F3 sh9_sample(const ushort4* __restrict__ cube, int w, int levels, int index, int li) {
    const float unit_theta = (0.5f + float(li >> 5)) / 32.0f;
    const float unit_phi = (0.5f + float(li & 31)) / 32.0f;
    const float cos_theta = 1.0f - 2.0f * unit_theta;
    const float sin_theta = sqrtf(clamp01(1.0f - cos_theta * cos_theta));
    const float phi = 2.0f * kPiF * unit_phi;
    const F3 dir = {cosf(phi) * sin_theta, cos_theta, sinf(phi) * sin_theta};
    const F3 radiance = cube_sample_lod(cube, w, levels, dir, 0.0f);
    const float Y00 = 0.282095f, Y1n = 0.488603f, Y2n = 1.092548f, Y20 = 0.315392f, Y22 = 0.546274f;
    float c;
    switch (index) {
        case 0: c = Y00; break;
        case 1: c = Y1n * dir.y; break;
        case 2: c = Y1n * dir.z; break;
        case 3: c = Y1n * dir.x; break;
        case 4: c = Y2n * dir.x * dir.y; break;
        case 5: c = Y2n * dir.y * dir.z; break;
        case 6: c = Y20 * (3.0f * dir.z * dir.z - 1.0f); break;
        case 7: c = Y2n * dir.x * dir.z; break;
        default: c = Y22 * (dir.x * dir.x - dir.y * dir.y); break;
    }
    return radiance * (c * (4.0f * kPiF / 1024.0f));
}
__device__ inline void sh9_block(const ushort4* __restrict__ cube, int w, int levels, int index,
                                 float4* __restrict__ out, F3* s) {
    const int t = threadIdx.x;
    s[t] = sh9_sample(cube, w, levels, index, t) + sh9_sample(cube, w, levels, index, t + 512);
    __syncthreads();
    for (int half = 256; half >= 1; half >>= 1) {
        if (t < half) s[t] = s[t] + s[t + half];
        __syncthreads();
    }
    if (t == 0) out[index] = make_float4(s[0].x, s[0].y, s[0].z, 0.0f);
}
constexpr int kSh9Blocks = 9;

__device__ inline uint32_t reverse_bits32(uint32_t b) {  // ReverseBits32 (shaders/Base/Noise.glsl:104-111)
    b = (b << 16) | (b >> 16);
    b = ((b & 0x00ff00ffu) << 8) | ((b & 0xff00ff00u) >> 8);
    b = ((b & 0x0f0f0f0fu) << 4) | ((b & 0xf0f0f0f0u) >> 4);
    b = ((b & 0x33333333u) << 2) | ((b & 0xccccccccu) >> 2);
    b = ((b & 0x55555555u) << 1) | ((b & 0xaaaaaaaau) >> 1);
    return b;
}

// CreateOrthonormalBasis (shaders/Base/Common.glsl:44-51, Duff et al. 2017)
__device__ inline void onb_frame(F3 N, F3& t0, F3& t1) {
    const float s = N.z >= 0.0f ? 1.0f : -1.0f;
    const float aa = -1.0f / (s + N.z);
    const float b = N.x * N.y * aa;
    t0 = {1.0f + s * N.x * N.x * aa, s * b, -s * N.x};
    t1 = {b, s + N.y * N.y * aa, -N.y};
}

constexpr int kMaxPrefilterLevels = 13;  // roughness_count <= log2(4096) + 1

// PrefilterRadiance.comp, all levels in one launch, after the kSh9Blocks workgroups that compute the
// SH9 coefficients (sh9_block; both read the environment cube only): workgroups kSh9Blocks +
// [block_start[l], block_start[l + 1]) build level l.
//
// The view direction is the normal, so a level's samples are the same in every texel's tangent frame:
// direction, cosine, density and mip level (H = (sin cos phi, sin sin phi, cos), L = 2 cos H - N).  A
// workgroup's first wave makes the table of those above the horizon; then a lane is a texel, the
// workgroup's kPrefilterWaves waves share its 64 texels' samples (wave v takes entries v,
// v + kPrefilterWaves, ..), and an entry's mip levels are wave-uniform.  Bound by the cube lookups'
// instructions.  128^2, 5 levels, with SH9: 11.4 us; 39.6 with a lane per sample of a texel, which
// evaluated the sample again in each texel.
struct PrefilterLevels {
    int count;
    int block_start[kMaxPrefilterLevels + 1];
    float roughness[kMaxPrefilterLevels];
    int samples[kMaxPrefilterLevels];  // at most 64; 1 at roughness 0
};

constexpr int kPrefilterWaves = 8;
// Whether a level of width wl is made by samples, a wave to a texel and a lane to a sample, rather than by tiles
// of 64 texels: where few texels leave CUs idle, a sample at a time is a chain of lookups (into the fine
// levels of the environment cube, the mip following the level's own texels).  us of the whole pass by samples
// up to a width of 4 / 8 / 16: 128^2 environment, 16^2 of 5 levels 7.8 / 4.7 / 4.7 (tiles alone 9.8), 32^2 of 5
// 7.8 / 7.0 / 5.1, 128^2 of 5 10.1 / 10.1 / 10.7; 1024^2 environment, 32^2 of 5 20.4 / 15.8 / 8.3.
__host__ __device__ inline bool prefilter_by_samples(int wl, int pw) { return wl <= 8 || pw <= 32; }
struct PrefilterSample {
    float x, y, z;  // direction in the texel's frame; z is also the weight
    float blend;    // of level + 1
    int level;
};

// Sample k of n (lane k < n) and whether it lies above the horizon.
__device__ inline bool prefilter_sample(uint32_t k, uint32_t n, float a2, float inv_sa_texel, int levels,
                                        PrefilterSample& s) {
    // Hammersley (shaders/Base/Noise.glsl:113-117) with no random offset
    const float q = float(k) / float(n);
    const float e1 = q - floorf(q);
    const float e2 = float(reverse_bits32(k)) * 2.3283064365386963e-10f;
    // ImportanceSampleGGX (shaders/Base/BRDF.glsl:48-67)
    const float phi = 2.0f * kPiF * e1;
    const float cos_t = sqrtf((1.0f - e2) / (1.0f + (a2 - 1.0f) * e2));
    const float sin_t = sqrtf(1.0f - cos_t * cos_t);
    s.x = 2.0f * cos_t * (sin_t * cosf(phi));
    s.y = 2.0f * cos_t * (sin_t * sinf(phi));
    s.z = fminf(2.0f * cos_t * cos_t - 1.0f, 1.0f);
    const float dg = (cos_t * a2 - cos_t) * cos_t + 1.0f;  // D_GGX (BRDF.glsl:36-40), NoH = HoV = cos_t
    const float D = a2 / (kPiF * dg * dg);
    const float pdf = fmaxf(D * cos_t / (4.0f * cos_t), 0.0001f);
    const float sa_sample = 1.0f / fmaxf(float(n) * pdf, 0.00001f);
    const float mip = 0.5f * log2f(sa_sample * inv_sa_texel) + 2.5f;
    const float lod = mip > 0.0f ? fminf(mip, float(levels - 1)) : 0.0f;
    s.level = int(lod);
    s.blend = lod - float(s.level);
    return s.z > 0.0f;
}

// Adds weight x (cube_level_bilinear's value) of a level of width 1 << log_w.
__device__ __forceinline__ void prefilter_add(const ushort4* __restrict__ level, int log_w, int face, float s, float t,
                                              float weight, F3& sum) {
    const int wl = 1 << log_w;
    const float top = float(wl - 1);
    const float fx = __builtin_amdgcn_fmed3f(fmaf(s, float(wl), -0.5f), 0.0f, top);
    const float fy = __builtin_amdgcn_fmed3f(fmaf(t, float(wl), -0.5f), 0.0f, top);
    const int x0 = int(fx), y0 = int(fy);
    const int dx = x0 < wl - 1 ? 1 : 0, dy = y0 < wl - 1 ? wl : 0;
    const unsigned at = (unsigned(face) << (2 * log_w)) + (unsigned(y0) << log_w) + unsigned(x0);
    const ushort4 a = level[at], b = level[at + dx], c = level[at + dy], d = level[at + dy + dx];
    const float ax = __builtin_amdgcn_fractf(fx), ay = __builtin_amdgcn_fractf(fy);
    const float wc = weight * ay, wa = weight * (1.0f - ay);
    const float w0 = wa * (1.0f - ax), w1 = wa * ax, w2 = wc * (1.0f - ax), w3 = wc * ax;
    sum = fma3(f3(w0), rgba16f_rgb(a), sum);
    sum = fma3(f3(w1), rgba16f_rgb(b), sum);
    sum = fma3(f3(w2), rgba16f_rgb(c), sum);
    sum = fma3(f3(w3), rgba16f_rgb(d), sum);
}

// The face of direction L and the position on it (cube_face_st, without its branches).
__device__ __forceinline__ int prefilter_face(F3 L, float& cs, float& ct) {
    const float ax = fabsf(L.x), ay = fabsf(L.y), az = fabsf(L.z);
    const bool mx = ax >= ay && ax >= az, my = !mx && ay >= az;
    const float major = mx ? L.x : my ? L.y : L.z;
    const bool neg = !(major >= 0.0f);
    const float sc0 = mx ? -L.z : L.x, tc0 = my ? L.z : -L.y;
    const float sc = neg && !my ? -sc0 : sc0, tc = neg && my ? -tc0 : tc0;
    const float ma = fabsf(major);
    float inv = __builtin_amdgcn_rcpf(ma);
    inv = fmaf(fmaf(-ma, inv, 1.0f), inv, inv);
    cs = fmaf(0.5f * sc, inv, 0.5f), ct = fmaf(0.5f * tc, inv, 0.5f);
    return (mx ? 0 : my ? 2 : 4) + (neg ? 1 : 0);
}
// Adds sample (x, y, z) of the frame (t0, t1, N) at level l0 + blend, l0 + 1 <= log_ew where blend > 0.
__device__ __forceinline__ void prefilter_lookup(const ushort4* __restrict__ env, int log_ew, F3 t0, F3 t1, F3 N, float x,
                                                 float y, float z, int l0, float blend, F3& sum) {
    float cs, ct;
    const int face = prefilter_face(fma3(t0, f3(x), fma3(t1, f3(y), N * z)), cs, ct);
    // Level l starts at 8 (w^2 - w_l^2) texels.
    const int log0 = log_ew - l0;
    const ushort4* base = env + 8ll * ((1ll << (2 * log_ew)) - (1ll << (2 * log0)));
    prefilter_add(base, log0, face, cs, ct, z * (1.0f - blend), sum);
    if (blend > 0.0f) {  // so there is a level l0 + 1
        const ushort4* next = env + 8ll * ((1ll << (2 * log_ew)) - (1ll << (2 * (log0 - 1))));
        prefilter_add(next, log0 - 1, face, cs, ct, z * blend, sum);
    }
}

__global__ __launch_bounds__(64 * kPrefilterWaves) void prefilter_kernel(const ushort4* __restrict__ env, int log_ew,
                                                                         float4* __restrict__ sh9_out,
                                                                         ushort4* __restrict__ out, int pw,
                                                                         PrefilterLevels lv) {
    constexpr int kThreads = 64 * kPrefilterWaves;
    __shared__ F3 s_sum[kThreads];
    __shared__ PrefilterSample s_sample[64];
    __shared__ float s_weight;
    __shared__ int s_count;
    const int ew = 1 << log_ew, elevels = log_ew + 1;
    if (int(blockIdx.x) < kSh9Blocks) {
        static_assert(kThreads == 512, "sh9_block's threads");
        sh9_block(env, ew, elevels, int(blockIdx.x), sh9_out, s_sum);
        return;
    }
    const int block = int(blockIdx.x) - kSh9Blocks;
    int level = 0;
    while (level + 1 < lv.count && block >= lv.block_start[level + 1]) ++level;
    const float roughness = lv.roughness[level];
    const int wl = max(pw >> level, 1);
    const int tile = block - lv.block_start[level];
    ushort4* dst = out + cube_level_offset(pw, level);
    if (roughness == 0.0f) {  // one sample, along the normal, at level 0
        const long long i = (long long)tile * kThreads + threadIdx.x;
        if (i >= 6ll * wl * wl) return;
        const int face = int(i / (wl * wl)), y = int(i / wl) % wl, x = int(i % wl);
        const F3 N = cube_texel_dir(face, x, y, wl);
        const F3 L = N * (2.0f * dot(N, N)) - N;
        const float NoL = clamp01(dot(N, L));
        const F3 c = cube_sample_lod(env, ew, elevels, L, 0.0f) * NoL;
        dst[i] = to_rgba16f(c * (1.0f / NoL), 0.0f);
        return;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float a = roughness * roughness, inv_sa_texel = (6.0f * float(wl) * float(wl)) / (4.0f * kPiF);
    if (prefilter_by_samples(wl, pw)) {  // a wave is a texel, a lane its sample
        const int p = tile * kPrefilterWaves + wave;
        if (p >= 6 * wl * wl) return;  // wave-uniform
        const F3 N = cube_texel_dir(p / (wl * wl), p % wl, (p / wl) % wl, wl);
        F3 t0, t1, sum = f3(0.0f);
        onb_frame(N, t0, t1);
        PrefilterSample s;
        const uint32_t n = uint32_t(lv.samples[level]);
        float weight = 0.0f;
        if (uint32_t(lane) < n && prefilter_sample(uint32_t(lane), n, a * a, inv_sa_texel, elevels, s)) {
            prefilter_lookup(env, log_ew, t0, t1, N, s.x, s.y, s.z, s.level, s.blend, sum);
            weight = s.z;
        }
        for (int m = 32; m >= 1; m >>= 1) {
            sum = sum + F3{__shfl_xor(sum.x, m, 64), __shfl_xor(sum.y, m, 64), __shfl_xor(sum.z, m, 64)};
            weight += __shfl_xor(weight, m, 64);
        }
        if (lane == 0) dst[p] = to_rgba16f(sum * (1.0f / weight), 0.0f);
        return;
    }
    // The workgroup's texels: 8 x 8 of a face.
    const long long p = (long long)tile * 64;
    const int face = int(p / (wl * wl)), q = int(p % (wl * wl)) >> 6, per_row = wl >> 3;
    const int x = (q % per_row) * 8 + (lane & 7), y = (q / per_row) * 8 + (lane >> 3);
    const F3 N = cube_texel_dir(face, x, y, wl);
    F3 t0, t1;
    onb_frame(N, t0, t1);
    if (wave == 0) {
        const uint32_t n = uint32_t(lv.samples[level]);
        PrefilterSample s;
        const bool up =
            uint32_t(lane) < n &&
            prefilter_sample(uint32_t(lane), n, a * a, inv_sa_texel, elevels, s);
        const uint64_t mask = __ballot(up);
        if (up) s_sample[__popcll(mask & ((1ull << lane) - 1))] = s;
        float weight = up ? s.z : 0.0f;
        for (int m = 32; m >= 1; m >>= 1) weight += __shfl_xor(weight, m, 64);
        if (lane == 0) s_weight = weight, s_count = __popcll(mask);
    }
    __syncthreads();
    const int count = s_count;
    F3 sum = f3(0.0f);
#pragma unroll 2
    for (int k = wave; k < count; k += kPrefilterWaves) {
        const PrefilterSample s = s_sample[k];
        const int l0 = __builtin_amdgcn_readfirstlane(s.level);
        const float blend = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, s.blend)));
        prefilter_lookup(env, log_ew, t0, t1, N, s.x, s.y, s.z, l0, blend, sum);
    }
    s_sum[threadIdx.x] = sum;
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int v = 1; v < kPrefilterWaves; ++v) sum = sum + s_sum[64 * v + lane];
    dst[(long long)face * wl * wl + y * wl + x] = to_rgba16f(sum * (1.0f / s_weight), 0.0f);
}

}  // namespace skyhip

using namespace skyhip;

extern "C" long long skyhip_cube_texels(int32_t width, int32_t levels) {
    if (width < 1 || levels < 0) return 0;
    return cube_level_offset(width, levels);
}

extern "C" int skyhip_environment_luminance(SkyhipContext* ctx, const SkyhipAtmosphereBufferData* atmosphere,
                                            const SkyhipAtmosphereRenderBufferData* render,
                                            const float* transmittance, int32_t transmittance_width,
                                            int32_t transmittance_height, const float* sky_view_luminance,
                                            const float* sky_view_transmittance, int32_t sky_view_width,
                                            int32_t sky_view_height, void* out_cube_rgba16f, int32_t width) {
    SKYHIP_CHECK(check_ctx(ctx));
    if (!atmosphere || !render || !out_cube_rgba16f) return fail(SKYHIP_ERR_INVALID_ARGUMENT, "NULL argument");
    SKYHIP_CHECK(validate_atmosphere(atmosphere));
    SKYHIP_CHECK(validate_render(render));
    SKYHIP_CHECK(validate_lut(transmittance, transmittance_width, transmittance_height, "transmittance"));
    SKYHIP_CHECK(validate_lut(sky_view_luminance, sky_view_width, sky_view_height, "sky-view luminance"));
    SKYHIP_CHECK(validate_lut(sky_view_transmittance, sky_view_width, sky_view_height, "sky-view transmittance"));
    if (!is_pow2(width) || width > 4096) return fail(SKYHIP_ERR_INVALID_SIZE, "cube width must be a power of two <= 4096");
    const AtmDev A = make_atm(*atmosphere);
    const EnvFrame e = make_env_frame(*render, *atmosphere);
    ushort4* cube = reinterpret_cast<ushort4*>(out_cube_rgba16f);
    const int levels = log2i(width) + 1, tile_log = std::min(kEnvTileLog, levels - 1), tiles = width >> tile_log;
    hipLaunchKernelGGL(env_luminance_kernel, dim3(tiles, tiles, 6), dim3(256), 0, ctx->stream, A, e,
                       reinterpret_cast<const float4*>(transmittance), transmittance_width, transmittance_height,
                       reinterpret_cast<const float4*>(sky_view_luminance),
                       reinterpret_cast<const float4*>(sky_view_transmittance), sky_view_width, sky_view_height, cube,
                       width, tile_log);
    SKYHIP_LAUNCH_CHECK("env_luminance_kernel");
    int l = tile_log + 1;
    while (l < levels) {
        const int last = (width >> l) > kMipTailWidth ? l + 1 : levels;  // a level too wide for the LDS by itself
        hipLaunchKernelGGL(cube_mip_tail_kernel, dim3(6), dim3(1024), 0, ctx->stream, cube, width, l, last);
        SKYHIP_LAUNCH_CHECK("cube_mip_tail_kernel");
        l = last;
    }
    return SKYHIP_OK;
}

extern "C" int skyhip_ibl_precompute(SkyhipContext* ctx, const void* environment_cube_rgba16f,
                                     int32_t environment_width, float* out_sh9_rgba, void* out_prefiltered_rgba16f,
                                     int32_t prefiltered_width, int32_t roughness_count) {
    SKYHIP_CHECK(check_ctx(ctx));
    if (!environment_cube_rgba16f || !out_sh9_rgba || !out_prefiltered_rgba16f)
        return fail(SKYHIP_ERR_INVALID_ARGUMENT, "NULL argument");
    if (!is_pow2(environment_width) || environment_width > 4096)
        return fail(SKYHIP_ERR_INVALID_SIZE, "environment width must be a power of two <= 4096");
    if (!is_pow2(prefiltered_width) || prefiltered_width > 4096)
        return fail(SKYHIP_ERR_INVALID_SIZE, "prefiltered width must be a power of two <= 4096");
    if (roughness_count < 1 || roughness_count > kMaxPrefilterLevels || (1 << (roughness_count - 1)) > prefiltered_width)
        return fail(SKYHIP_ERR_INVALID_SIZE, "roughness_count outside [1, log2(prefiltered_width) + 1]");
    const ushort4* env = reinterpret_cast<const ushort4*>(environment_cube_rgba16f);
    ushort4* out = reinterpret_cast<ushort4*>(out_prefiltered_rgba16f);
    PrefilterLevels lv{};
    lv.count = roughness_count;
    long long blocks = 0;
    for (int l = 0; l < roughness_count; ++l) {
        const int wl = prefiltered_width >> l;
        lv.roughness[l] = roughness_count > 1 ? float(l) / float(roughness_count - 1) : 0.0f;
        // The level's sample count uint(mix(1, 64, pow(roughness, 0.3))) in FP32 (1 at roughness 0,
        // 64 at 1; in between, for every level of up to 13, at least 0.011 from an integer, so no
        // powf rounding moves it).
        const float p = std::pow(lv.roughness[l], 0.3f);
        lv.samples[l] = std::min(std::max(int(uint32_t(1.0f * (1.0f - p) + 64.0f * p)), 1), 64);
        lv.block_start[l] = int(blocks);
        blocks += div_up(6LL * wl * wl, lv.roughness[l] == 0.0f ? 64 * kPrefilterWaves : prefilter_by_samples(wl, prefiltered_width) ? kPrefilterWaves : 64);
    }
    lv.block_start[roughness_count] = int(blocks);
    hipLaunchKernelGGL(prefilter_kernel, dim3(unsigned(kSh9Blocks + blocks)), dim3(64 * kPrefilterWaves), 0, ctx->stream,
                       env, log2i(environment_width), reinterpret_cast<float4*>(out_sh9_rgba), out, prefiltered_width, lv);
    SKYHIP_LAUNCH_CHECK("prefilter_kernel");
    return SKYHIP_OK;
}
