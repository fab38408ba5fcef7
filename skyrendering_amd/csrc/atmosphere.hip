// Atmosphere LUT kernels for gfx950: transmittance, multiple scattering,
// sky view and aerial perspective, plus their C-ABI entry points.
//
// Layout: every LUT is RGBA32F in GL texel order, neighbouring lanes at neighbouring texels so that
// stores coalesce.  Transmittance is a lane per texel, four in the one-call set; multiple scattering a
// wave64 per texel (its 64 sphere directions are the lanes), four waves in the set; the sky view a lane
// per texel over its row's shared steps (sky_rows.h), or marching for itself with dither or wide LUTs,
// two waves to 64 texels in the set; aerial perspective four waves to 64 froxels.
#include "sky_rows.h"

#include <algorithm>
#include <cmath>

namespace skyhip {

// ---------------------------------------------------------------------------
// Transmittance (Atmosphere.glsl:71-88, :311-337)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void transmittance_kernel(SkyhipAtmosphereBufferData b, float4* __restrict__ out,
                                                            int w, int h) {
    int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= w * h) return;
    out[t] = transmittance_texel_rgba(b, t % w, t / w, w, h);
}

// ---------------------------------------------------------------------------
// Multiple scattering (Atmosphere.glsl:344-438): one wave64 per texel, whose step tables (sky_rows.h)
// its workgroup's texels, of one row, share; marches of more than kMsMaxSteps steps integrate
// direction by direction.  32 x 32, 30 steps: 13.1 us, 21.3 with every direction evaluating its own
// densities and exponentials.
// ---------------------------------------------------------------------------
constexpr int kMsTexels = 4;  // texels (waves) of a workgroup
__global__ __launch_bounds__(64 * kMsTexels) void multiscattering_kernel(SkyhipAtmosphereBufferData b,
                                                                         const float4* __restrict__ T, int tw, int th,
                                                                         float4* __restrict__ out, int w, int h) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ MsTotals totals[kMsThetas];
    const AtmDev A = make_atm(b);
    const int n = row_step_count(A.ms_steps), ix = blockIdx.x * kMsTexels + (threadIdx.x >> 6), iy = blockIdx.y;
    const int lane = threadIdx.x & 63;
    if (n > kMsMaxSteps) {
        if (ix >= w) return;  // wave-uniform
        const float4 v = multiscattering_texel(A, T, tw, th, ix, iy, w, h, lane);
        if (lane == 0) out[iy * w + ix] = v;
        return;
    }
    MsStep* steps = reinterpret_cast<MsStep*>(smem);
    ms_row_tables(A, iy, h, tw, th, n, steps, totals);
    __syncthreads();
    if (ix >= w) return;
    const MsSun sun = ms_sun(ix, w, lane);
    const float4 v = ms_row_reduce<false>(A, T, tw, th, totals, sun, ms_row_steps<false>(T, tw, th, steps, n, sun, 0, n));
    if (lane == 0) out[iy * w + ix] = v;
}

// ---------------------------------------------------------------------------
// Sky view (AtmosphereRenderer.glsl:74-186)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void sky_view_kernel(SkyhipAtmosphereBufferData b,
                                                       SkyhipAtmosphereRenderBufferData rbd,
                                                       const float4* __restrict__ T, int tw, int th,
                                                       const float4* __restrict__ MS, int mw, int mh,
                                                       const uint16_t* __restrict__ blue_noise, int bn_size,
                                                       float4* __restrict__ out_l, float4* __restrict__ out_t, int w,
                                                       int h) {
    int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= w * h) return;
    const AtmDev A = make_atm(b);
    const RenderDev R = make_render(rbd);
    F3 L, Tr;
    sky_view_texel(A, R, T, tw, th, MS, mw, mh, blue_noise, bn_size, t % w, t / w, w, h, L, Tr);
    out_l[t] = make_float4(L.x, L.y, L.z, 0.0f);
    out_t[t] = make_float4(Tr.x, Tr.y, Tr.z, 0.0f);
}

// The same without dither, by rows: a wave takes 64 columns of a row.  A single LUT is latency-bound,
// so a lane takes one ray, where the batched builder's takes up to three.
__global__ __launch_bounds__(64) void sky_view_rows_kernel(SkyhipAtmosphereBufferData b,
                                                           SkyhipAtmosphereRenderBufferData rbd,
                                                           const float4* __restrict__ T, int tw, int th,
                                                           const float4* __restrict__ MS, int mw, int mh,
                                                           float4* __restrict__ out_l, float4* __restrict__ out_t,
                                                           int w, int h) {
    __shared__ RowLds lds;
    const AtmDev A = make_atm(b);
    const RenderDev R = make_render(rbd);
    sky_view_row<1>([&] { return A; }, R, sky_view_row_setup(A, R, blockIdx.y, h), T, tw, th, MS, mw, mh, blockIdx.y,
                    blockIdx.x * 64, w, lds, out_l, out_t);
}

// ---------------------------------------------------------------------------
// Aerial perspective (AtmosphereRenderer.glsl:191-243)
// ---------------------------------------------------------------------------
// Workgroup `block` of slice iz: P waves share 64 froxels (scattered_luminance_split).
template <int P>
__device__ __forceinline__ void aerial_perspective_block(const AtmDev& A, const RenderDev& R,
                                                         const float* inv_view_projection, const float4* __restrict__ T,
                                                         int tw, int th, const float4* __restrict__ MS, int mw, int mh,
                                                         const uint16_t* __restrict__ blue_noise, int bn_size,
                                                         float4* __restrict__ out_l, float4* __restrict__ out_t, int w,
                                                         int h, int d, int block, int iz, SplitLds& lds) {
    const int wave = threadIdx.x >> 6;
    const int texel = block * (256 / P) + 64 * (wave / P) + int(threadIdx.x & 63);
    const bool valid = texel < w * h;
    const int t = valid ? texel : 0;
    const AerialRay ray = aerial_ray(A, R, inv_view_projection, blue_noise, bn_size, t % w, t / w, iz, w, h, d);
    F3 L, Tr;
    scattered_luminance_split<P>(A, T, tw, th, MS, mw, mh, ray.s, ray.marching_distance, R.ap_steps,
                                 ray.start_i, ray.marching_distance > 0.0f, lds, L, Tr);
    if (wave % P == 0 && valid) {
        const long long o = (long long)iz * w * h + t;
        out_l[o] = make_float4(L.x, L.y, L.z, 0.0f);
        out_t[o] = make_float4(Tr.x, Tr.y, Tr.z, 0.0f);
    }
}

// Bound by the steps' instructions, the lookups' latency and the rays' set-up, which every part repeats.
// A 32^3 LUT at 51 steps: 12.6 us; 26.1 with four consecutive lanes to a froxel, whose lookups at four
// distances touch four times the lines per load.  The frame around it with 1, 2 and 4 waves to 64
// froxels takes 83.8, 72.3 and 68.8 us (consecutive lanes: 83.4, 73.3 and 78.8 with 1, 2 and 4).
constexpr int kApParts = 4;
struct ViewProjectionInverse {
    float m[16];
};
__global__ __launch_bounds__(256) void aerial_perspective_kernel(
    AtmDev A, RenderDev R, ViewProjectionInverse m, const float4* __restrict__ T, int tw, int th,
    const float4* __restrict__ MS, int mw, int mh, const uint16_t* __restrict__ blue_noise, int bn_size,
    float4* __restrict__ out_l, float4* __restrict__ out_t, int w, int h, int d) {
    __shared__ SplitLds lds;
    aerial_perspective_block<kApParts>(A, R, m.m, T, tw, th, MS, mw, mh, blue_noise, bn_size, out_l, out_t, w, h, d,
                                       blockIdx.x, blockIdx.y, lds);
}
ViewProjectionInverse view_projection_inverse(const SkyhipAtmosphereRenderBufferData& r) {
    ViewProjectionInverse m;
    std::copy(r.inv_view_projection, r.inv_view_projection + 16, m.m);
    return m;
}

// ---------------------------------------------------------------------------
// Latency-bound form of one frame's LUT set (skyhip_atmosphere_lut_set).  A single set has
// too few texels to fill 256 CUs one lane per texel (the 256x64 transmittance LUT is one wave
// per CU, the 192x108 sky view 1.3), so each texel's march is split over lanes or waves
// and the parts combined in order, and the sky-view and aerial-perspective passes, which read
// only T and MS, run as one launch.  Same quantities as the per-pass kernels; the FP32 sums
// associate differently (parts add in order), which is why the batched builder, which must
// match the per-pass kernels bit for bit, does not use these.
// ---------------------------------------------------------------------------
constexpr int kSetTransmittanceParts = 4;
// Waves of a sky-view and of an aerial-perspective ray: the set takes 32.2 us with 2 and 4, 34.8 with 2
// and 2, 32.8 with 4 and 4, 38.4 with 1 and 2, and 44.3 with 3 and 8 consecutive lanes.
constexpr int kSetSkyViewParts = 2;
constexpr int kSetAerialParts = 4;

template <class S, int kParts>
__device__ inline F3 transmittance_texel_split(const SkyhipAtmosphereBufferData& b, int ix, int iy, int w, int h,
                                               int part) {
    const int n = transmittance_step_count(b);
    const int c = (n + kParts - 1) / kParts, first = min(part * c, n);
    S od[3], dx;
    transmittance_od<S>(b, ix, iy, w, h, first, max(0, min(c, n - first)), od, dx);
    S acc[3] = {od[0], od[1], od[2]};
    for (int p = 1; p < kParts; ++p)
        for (int k = 0; k < 3; ++k) acc[k] += __shfl_down(od[k], p, 64);
    return transmittance_from_od<S>(b, acc, dx);
}

__global__ __launch_bounds__(256) void set_transmittance_kernel(SkyhipAtmosphereBufferData b,
                                                                float4* __restrict__ out, int w, int h) {
    constexpr int P = kSetTransmittanceParts;
    const int g = blockIdx.x * 256 + threadIdx.x;
    const int t = g / P, part = g % P;
    if (t >= w * h) return;  // whole groups of P lanes leave together
    const int ix = t % w, iy = t / w;
    const F3 v = ix >= transmittance_fp64_column(w) ? transmittance_texel_split<double, P>(b, ix, iy, w, h, part)
                                                    : transmittance_texel_split<float, P>(b, ix, iy, w, h, part);
    if (part == 0) out[t] = make_float4(v.x, v.y, v.z, 1.0f);
}

// Multiple scattering with the steps of a texel's 64 directions split over kSetMsParts waves: the
// workgroup builds the step tables (whose weights hold the transmittance up to each step, so parts
// simply add), kMsMaxSteps steps at a time, wave p marches part p of them, and wave 0 adds the parts in
// order and reduces over the directions as the per-pass kernel does.  (One chunk is a kernel of its own: the
// march kept between chunks takes 106 registers for 73.)  The set at 128 steps: 50.9 us, 83.9 with the
// per-pass kernel's march direction by direction; an 8 x 8 LUT 39.0 against 90.8.
constexpr int kSetMsParts = 4;
template <bool kChunks>
__global__ __launch_bounds__(64 * kSetMsParts) void set_multiscattering_kernel(SkyhipAtmosphereBufferData b,
                                                                               const float4* __restrict__ T, int tw,
                                                                               int th, float4* __restrict__ out,
                                                                               int w, int h) {
    constexpr int P = kSetMsParts;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ MsTotals totals[kMsThetas];
    __shared__ float part_sums[P - 1][3][64];
    MsStep* steps = reinterpret_cast<MsStep*>(smem);
    const AtmDev A = make_atm(b);
    const int ix = blockIdx.x, iy = blockIdx.y, part = threadIdx.x >> 6, lane = threadIdx.x & 63;
    static_assert(64 * P == kMsThetas * kRowSteps, "half a wave per polar angle");
    const int n = row_step_count(A.ms_steps), theta = int(threadIdx.x) / kRowSteps;
    const MsSun sun = ms_sun(ix, w, lane);
    MsMarch m = ms_march(A, iy, h, theta);
    F3 L = f3(0.0f);
    if (n == 0 && (threadIdx.x & 31) == 0) totals[theta] = ms_totals(m);
    for (int first = 0; first < n; first += kMsMaxSteps) {  // workgroup-uniform
        const int count = min(kMsMaxSteps, n - first), c = (count + P - 1) / P;
        if (kChunks && first > 0) __syncthreads();  // the previous steps' reads
        ms_march_steps(A, m, n, first, first + count, tw, th, steps + theta * count);
        if (first + count == n && (threadIdx.x & 31) == 0) totals[theta] = ms_totals(m);
        __syncthreads();
        L += ms_row_steps<false>(T, tw, th, steps, count, sun, min(part * c, count), min(part * c + c, count));
        if (!kChunks) break;
    }
    if (part > 0) {
        part_sums[part - 1][0][lane] = L.x;
        part_sums[part - 1][1][lane] = L.y;
        part_sums[part - 1][2][lane] = L.z;
    }
    __syncthreads();
    if (part != 0) return;
    for (int p = 0; p < P - 1; ++p) L += F3{part_sums[p][0][lane], part_sums[p][1][lane], part_sums[p][2][lane]};
    const float4 v = ms_row_reduce<false>(A, T, tw, th, totals, sun, L);
    if (lane == 0) out[iy * w + ix] = v;
}

// Blocks [0, sv_blocks) build the sky view, kSetSkyViewParts waves to a texel; the rest the aerial
// perspective, ap_blocks to a slice, kSetAerialParts waves to a froxel (no blue-noise dither, as the set's per-pass calls).
__global__ __launch_bounds__(256) void set_sky_aerial_kernel(
    AtmDev A, RenderDev R, ViewProjectionInverse m, const float4* __restrict__ T, int tw, int th,
    const float4* __restrict__ MS, int mw, int mh, float4* __restrict__ sv_l, float4* __restrict__ sv_t, int sw,
    int sh, int sv_blocks, float4* __restrict__ ap_l, float4* __restrict__ ap_t, int aw, int ah, int ad,
    int ap_blocks) {
    __shared__ SplitLds lds;
    if (int(blockIdx.x) < sv_blocks) {
        F3 L, Tr;
        constexpr int P = kSetSkyViewParts;
        const int wave = threadIdx.x >> 6;
        const int texel = int(blockIdx.x) * (256 / P) + 64 * (wave / P) + int(threadIdx.x & 63);
        const bool valid = texel < sw * sh;
        const int t = valid ? texel : 0;
        const SkyViewRay ray = sky_view_ray(A, R, nullptr, 1, t % sw, t / sw, sw, sh);
        scattered_luminance_split<P>(A, T, tw, th, MS, mw, mh, ray.s, ray.dist, R.sv_steps, ray.start_i,
                                     ray.dist > 0.0f, lds, L, Tr);
        if (wave % P == 0 && valid) {
            sv_l[t] = make_float4(L.x, L.y, L.z, 0.0f);
            sv_t[t] = make_float4(Tr.x, Tr.y, Tr.z, 0.0f);
        }
        return;
    }
    const int block = int(blockIdx.x) - sv_blocks, iz = block / ap_blocks;
    aerial_perspective_block<kSetAerialParts>(A, R, m.m, T, tw, th, MS, mw, mh, nullptr, 1, ap_l, ap_t, aw, ah, ad,
                                              block - iz * ap_blocks, iz, lds);
}

// ---------------------------------------------------------------------------
// Validation and launch helpers
// ---------------------------------------------------------------------------
constexpr int kMaxLutDim = 8192;

int validate_atmosphere(const SkyhipAtmosphereBufferData* b) {
    SKYHIP_CHECK(require(b != nullptr, SKYHIP_ERR_INVALID_ARGUMENT, "atmosphere block is NULL"));
    SKYHIP_CHECK(require(finite_block(reinterpret_cast<const float*>(b), sizeof(*b) / 4), SKYHIP_ERR_NON_FINITE,
                         "atmosphere block has a non-finite field"));
    SKYHIP_CHECK(require(b->bottom_radius > 0.0f && b->top_radius > b->bottom_radius, SKYHIP_ERR_NON_FINITE,
                         "atmosphere needs 0 < bottom_radius < top_radius"));
    SKYHIP_CHECK(require(b->transmittance_steps > 0.0f && b->transmittance_steps <= 4096.0f &&
                             b->multiscattering_steps > 0.0f && b->multiscattering_steps <= 4096.0f,
                         SKYHIP_ERR_INVALID_SIZE, "step counts must be in (0, 4096]"));
    return SKYHIP_OK;
}

int validate_render(const SkyhipAtmosphereRenderBufferData* r) {
    SKYHIP_CHECK(require(r != nullptr, SKYHIP_ERR_INVALID_ARGUMENT, "render block is NULL"));
    SKYHIP_CHECK(require(finite_block(reinterpret_cast<const float*>(r), sizeof(*r) / 4), SKYHIP_ERR_NON_FINITE,
                         "render block has a non-finite field"));
    SKYHIP_CHECK(require(r->sky_view_lut_steps >= 0.0f && r->sky_view_lut_steps <= 4096.0f &&
                             r->aerial_perspective_lut_steps >= 0.0f && r->aerial_perspective_lut_steps <= 4096.0f,
                         SKYHIP_ERR_INVALID_SIZE, "step counts must be in [0, 4096]"));
    return SKYHIP_OK;
}

int validate_lut(const void* p, int w, int h, const char* what) {
    if (p == nullptr) return fail(SKYHIP_ERR_INVALID_ARGUMENT, "%s pointer is NULL", what);
    if (w < 2 || h < 2 || w > kMaxLutDim || h > kMaxLutDim)
        return fail(SKYHIP_ERR_INVALID_SIZE, "%s size %dx%d outside [2, %d]", what, w, h, kMaxLutDim);
    return SKYHIP_OK;
}

int validate_blue_noise(const uint16_t* bn, int size) {
    if (bn == nullptr) return SKYHIP_OK;
    if (size < 1 || size > 4096 || (size & (size - 1)) != 0)
        return fail(SKYHIP_ERR_INVALID_SIZE, "blue-noise tile size %d is not a power of two in [1, 4096]", size);
    return SKYHIP_OK;
}

int launch_transmittance(hipStream_t st, const SkyhipAtmosphereBufferData& b, float* out, int w, int h) {
    hipLaunchKernelGGL(transmittance_kernel, dim3(div_up(w * h, 256)), dim3(256), 0, st, b,
                       reinterpret_cast<float4*>(out), w, h);
    SKYHIP_LAUNCH_CHECK("transmittance_kernel");
    return SKYHIP_OK;
}

int launch_multiscattering(hipStream_t st, const SkyhipAtmosphereBufferData& b, const float* T, int tw, int th,
                           float* out, int w, int h) {
    hipLaunchKernelGGL(multiscattering_kernel, dim3(div_up(w, kMsTexels), h), dim3(64 * kMsTexels),
                       ms_table_bytes(b.multiscattering_steps), st, b, reinterpret_cast<const float4*>(T), tw, th,
                       reinterpret_cast<float4*>(out), w, h);
    SKYHIP_LAUNCH_CHECK("multiscattering_kernel");
    return SKYHIP_OK;
}

int launch_sky_view(hipStream_t st, const SkyhipAtmosphereBufferData& b, const SkyhipAtmosphereRenderBufferData& r,
                    const float* T, int tw, int th, const float* MS, int mw, int mh, const uint16_t* bn, int bn_size,
                    float* L, float* Tr, int w, int h) {
    // Rows share their march unless the dither starts every texel's elsewhere, or the LUTs are wider
    // than a wave's entries.  128 x 128, 30 steps: 12.7 us by rows, 31.6 texel by texel with the longer
    // step and 18 with scatter_step (256 + 32 columns 13.1 against 257 + 32 18.3; 2048 x 1024 132 and
    // 268).
    if (bn == nullptr && row_luts_fit(tw, mw)) {
        hipLaunchKernelGGL(sky_view_rows_kernel, dim3(div_up(w, 64), h), dim3(64), 0, st, b, r,
                           reinterpret_cast<const float4*>(T), tw, th, reinterpret_cast<const float4*>(MS), mw, mh,
                           reinterpret_cast<float4*>(L), reinterpret_cast<float4*>(Tr), w, h);
        SKYHIP_LAUNCH_CHECK("sky_view_rows_kernel");
        return SKYHIP_OK;
    }
    hipLaunchKernelGGL(sky_view_kernel, dim3(div_up(w * h, 256)), dim3(256), 0, st, b, r,
                       reinterpret_cast<const float4*>(T), tw, th, reinterpret_cast<const float4*>(MS), mw, mh, bn,
                       bn_size, reinterpret_cast<float4*>(L), reinterpret_cast<float4*>(Tr), w, h);
    SKYHIP_LAUNCH_CHECK("sky_view_kernel");
    return SKYHIP_OK;
}

int launch_aerial_perspective(hipStream_t st, const SkyhipAtmosphereBufferData& b,
                              const SkyhipAtmosphereRenderBufferData& r, const float* T, int tw, int th,
                              const float* MS, int mw, int mh, const uint16_t* bn, int bn_size, float* L, float* Tr,
                              int w, int h, int d) {
    hipLaunchKernelGGL(aerial_perspective_kernel, dim3(div_up((long long)w * h * kApParts, 256), d), dim3(256), 0, st,
                       make_atm(b), make_render(r), view_projection_inverse(r),
                       reinterpret_cast<const float4*>(T), tw, th, reinterpret_cast<const float4*>(MS), mw, mh, bn,
                       bn_size, reinterpret_cast<float4*>(L), reinterpret_cast<float4*>(Tr), w, h, d);
    SKYHIP_LAUNCH_CHECK("aerial_perspective_kernel");
    return SKYHIP_OK;
}

}  // namespace skyhip

using namespace skyhip;

extern "C" int skyhip_transmittance_lut(SkyhipContext* ctx, const SkyhipAtmosphereBufferData* atmosphere,
                                        float* transmittance_rgba, int32_t width, int32_t height) {
    SKYHIP_CHECK(check_ctx(ctx));
    SKYHIP_CHECK(validate_atmosphere(atmosphere));
    SKYHIP_CHECK(validate_lut(transmittance_rgba, width, height, "transmittance"));
    return launch_transmittance(ctx->stream, *atmosphere, transmittance_rgba, width, height);
}

extern "C" int skyhip_multiscattering_lut(SkyhipContext* ctx, const SkyhipAtmosphereBufferData* atmosphere,
                                          const float* transmittance_rgba, int32_t transmittance_width,
                                          int32_t transmittance_height, float* multiscattering_rgba, int32_t width,
                                          int32_t height) {
    SKYHIP_CHECK(check_ctx(ctx));
    SKYHIP_CHECK(validate_atmosphere(atmosphere));
    SKYHIP_CHECK(validate_lut(transmittance_rgba, transmittance_width, transmittance_height, "transmittance"));
    SKYHIP_CHECK(validate_lut(multiscattering_rgba, width, height, "multiscattering"));
    return launch_multiscattering(ctx->stream, *atmosphere, transmittance_rgba, transmittance_width,
                                  transmittance_height, multiscattering_rgba, width, height);
}

extern "C" int skyhip_atmosphere_update_luts(SkyhipContext* ctx, const SkyhipAtmosphereParameters* parameters,
                                             float* transmittance_rgba, int32_t transmittance_width,
                                             int32_t transmittance_height, float* multiscattering_rgba,
                                             int32_t multiscattering_width, int32_t multiscattering_height) {
    SKYHIP_CHECK(check_ctx(ctx));
    SkyhipAtmosphereBufferData b;
    SKYHIP_CHECK(skyhip_atmosphere_assign_buffer_data(parameters, &b));
    SKYHIP_CHECK(validate_atmosphere(&b));
    SKYHIP_CHECK(validate_lut(transmittance_rgba, transmittance_width, transmittance_height, "transmittance"));
    SKYHIP_CHECK(validate_lut(multiscattering_rgba, multiscattering_width, multiscattering_height, "multiscattering"));
    SKYHIP_CHECK(launch_transmittance(ctx->stream, b, transmittance_rgba, transmittance_width, transmittance_height));
    return launch_multiscattering(ctx->stream, b, transmittance_rgba, transmittance_width, transmittance_height,
                                  multiscattering_rgba, multiscattering_width, multiscattering_height);
}

extern "C" int skyhip_sky_view_lut(SkyhipContext* ctx, const SkyhipAtmosphereBufferData* atmosphere,
                                   const SkyhipAtmosphereRenderBufferData* render, const float* transmittance_rgba,
                                   int32_t transmittance_width, int32_t transmittance_height,
                                   const float* multiscattering_rgba, int32_t multiscattering_width,
                                   int32_t multiscattering_height, const uint16_t* blue_noise, int32_t blue_noise_size,
                                   float* luminance_rgba, float* sky_transmittance_rgba, int32_t width,
                                   int32_t height) {
    SKYHIP_CHECK(check_ctx(ctx));
    SKYHIP_CHECK(validate_atmosphere(atmosphere));
    SKYHIP_CHECK(validate_render(render));
    SKYHIP_CHECK(validate_lut(transmittance_rgba, transmittance_width, transmittance_height, "transmittance"));
    SKYHIP_CHECK(validate_lut(multiscattering_rgba, multiscattering_width, multiscattering_height, "multiscattering"));
    SKYHIP_CHECK(validate_blue_noise(blue_noise, blue_noise_size));
    SKYHIP_CHECK(validate_lut(luminance_rgba, width, height, "sky-view luminance"));
    SKYHIP_CHECK(validate_lut(sky_transmittance_rgba, width, height, "sky-view transmittance"));
    return launch_sky_view(ctx->stream, *atmosphere, *render, transmittance_rgba, transmittance_width,
                           transmittance_height, multiscattering_rgba, multiscattering_width, multiscattering_height,
                           blue_noise, blue_noise_size, luminance_rgba, sky_transmittance_rgba, width, height);
}

extern "C" int skyhip_aerial_perspective_lut(SkyhipContext* ctx, const SkyhipAtmosphereBufferData* atmosphere,
                                             const SkyhipAtmosphereRenderBufferData* render,
                                             const float* transmittance_rgba, int32_t transmittance_width,
                                             int32_t transmittance_height, const float* multiscattering_rgba,
                                             int32_t multiscattering_width, int32_t multiscattering_height,
                                             const uint16_t* blue_noise, int32_t blue_noise_size,
                                             float* luminance_rgba, float* ap_transmittance_rgba, int32_t width,
                                             int32_t height, int32_t depth) {
    SKYHIP_CHECK(check_ctx(ctx));
    SKYHIP_CHECK(validate_atmosphere(atmosphere));
    SKYHIP_CHECK(validate_render(render));
    SKYHIP_CHECK(validate_lut(transmittance_rgba, transmittance_width, transmittance_height, "transmittance"));
    SKYHIP_CHECK(validate_lut(multiscattering_rgba, multiscattering_width, multiscattering_height, "multiscattering"));
    SKYHIP_CHECK(validate_blue_noise(blue_noise, blue_noise_size));
    SKYHIP_CHECK(validate_lut(luminance_rgba, width, height, "aerial-perspective luminance"));
    SKYHIP_CHECK(validate_lut(ap_transmittance_rgba, width, height, "aerial-perspective transmittance"));
    if (depth < 2 || depth > 1024) return fail(SKYHIP_ERR_INVALID_SIZE, "aerial-perspective depth %d outside [2, 1024]", depth);
    return launch_aerial_perspective(ctx->stream, *atmosphere, *render, transmittance_rgba, transmittance_width,
                                     transmittance_height, multiscattering_rgba, multiscattering_width,
                                     multiscattering_height, blue_noise, blue_noise_size, luminance_rgba,
                                     ap_transmittance_rgba, width, height, depth);
}

extern "C" int skyhip_atmosphere_lut_set(SkyhipContext* ctx, const SkyhipAtmosphereBufferData* atmosphere,
                                         const SkyhipAtmosphereRenderBufferData* render, float* transmittance_rgba,
                                         int32_t transmittance_width, int32_t transmittance_height,
                                         float* multiscattering_rgba, int32_t multiscattering_width,
                                         int32_t multiscattering_height, float* sky_view_luminance_rgba,
                                         float* sky_view_transmittance_rgba, int32_t sky_view_width,
                                         int32_t sky_view_height, float* ap_luminance_rgba,
                                         float* ap_transmittance_rgba, int32_t ap_width, int32_t ap_height,
                                         int32_t ap_depth) {
    SKYHIP_CHECK(check_ctx(ctx));
    SKYHIP_CHECK(validate_atmosphere(atmosphere));
    SKYHIP_CHECK(validate_render(render));
    const int tw = transmittance_width, th = transmittance_height, mw = multiscattering_width,
              mh = multiscattering_height;
    SKYHIP_CHECK(validate_lut(transmittance_rgba, tw, th, "transmittance"));
    SKYHIP_CHECK(validate_lut(multiscattering_rgba, mw, mh, "multiscattering"));
    SKYHIP_CHECK(validate_lut(sky_view_luminance_rgba, sky_view_width, sky_view_height, "sky-view luminance"));
    SKYHIP_CHECK(validate_lut(sky_view_transmittance_rgba, sky_view_width, sky_view_height, "sky-view transmittance"));
    SKYHIP_CHECK(validate_lut(ap_luminance_rgba, ap_width, ap_height, "aerial-perspective luminance"));
    SKYHIP_CHECK(validate_lut(ap_transmittance_rgba, ap_width, ap_height, "aerial-perspective transmittance"));
    if (ap_depth < 2 || ap_depth > 1024) return fail(SKYHIP_ERR_INVALID_SIZE, "aerial-perspective depth outside [2, 1024]");
    hipStream_t st = ctx->stream;
    hipLaunchKernelGGL(set_transmittance_kernel, dim3(div_up((long long)tw * th * kSetTransmittanceParts, 256)),
                       dim3(256), 0, st, *atmosphere, reinterpret_cast<float4*>(transmittance_rgba), tw, th);
    SKYHIP_LAUNCH_CHECK("set_transmittance_kernel");
    const int ms_steps = row_step_count(atmosphere->multiscattering_steps);
    hipLaunchKernelGGL(ms_steps > kMsMaxSteps ? set_multiscattering_kernel<true> : set_multiscattering_kernel<false>,
                       dim3(mw, mh), dim3(64 * kSetMsParts),
                       size_t(kMsThetas) * std::min(ms_steps, kMsMaxSteps) * sizeof(MsStep), st, *atmosphere,
                       reinterpret_cast<const float4*>(transmittance_rgba), tw, th,
                       reinterpret_cast<float4*>(multiscattering_rgba), mw, mh);
    SKYHIP_LAUNCH_CHECK("set_multiscattering_kernel");
    const int sv_blocks = int(div_up((long long)sky_view_width * sky_view_height * kSetSkyViewParts, 256));
    const int ap_blocks = int(div_up((long long)ap_width * ap_height * kSetAerialParts, 256));
    hipLaunchKernelGGL(set_sky_aerial_kernel, dim3(sv_blocks + ap_blocks * ap_depth), dim3(256), 0, st,
                       make_atm(*atmosphere), make_render(*render), view_projection_inverse(*render),
                       reinterpret_cast<const float4*>(transmittance_rgba), tw, th,
                       reinterpret_cast<const float4*>(multiscattering_rgba), mw, mh,
                       reinterpret_cast<float4*>(sky_view_luminance_rgba),
                       reinterpret_cast<float4*>(sky_view_transmittance_rgba), sky_view_width, sky_view_height,
                       sv_blocks, reinterpret_cast<float4*>(ap_luminance_rgba),
                       reinterpret_cast<float4*>(ap_transmittance_rgba), ap_width, ap_height, ap_depth,
                       ap_blocks);
    SKYHIP_LAUNCH_CHECK("set_sky_aerial_kernel");
    return SKYHIP_OK;
}
