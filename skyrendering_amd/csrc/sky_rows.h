// The atmosphere integrator (ComputeScatteredLuminance, Atmosphere.glsl:220-295) for rows of rays that
// leave one point at one zenith angle towards different azimuths: the rows of the sky-view LUT and of a
// panorama, and the directions of one polar angle in the multiple-scattering LUT.
//
// Along such a row the altitude, the densities, the extinction, the transmittance so far and the LUT
// rows that a step reads are the same for every ray; only the sun's zenith cosine at the step differs,
// mu_s = (r mu_s0 + d nu) / r_d, linear in the ray's own sun-view cosine nu.  So a step's exponentials,
// divisions and densities are evaluated once per row, and its weights
//   w_r = T (1 - T_i) / sigma * sigma_Rayleigh,  w_m likewise for Mie
// kept; a ray adds w V and w MS, V the sun's visibility and MS the multiple scattering at its mu_s, and
// multiplies by its phases at the end.  A ray's step is about 50 vector instructions instead of about
// 160.  The sums associate differently from the ray-by-ray form (scattered_luminance); both are within
// 4e-7 (relative 2-norm) of 64-bit arithmetic.
#pragma once

#include <type_traits>

#include "lut_texels.h"

namespace skyhip {

// What a step has in common for its row.
struct RowStep {
    float a0, a1;                 // mu_s = a0 + a1 nu
    float r, r2, h2q;             // radius, its square, R_t^2 - r^2
    float d_min, kx;              // transmittance column = (d_sun - d_min) kx
    float fade_c, fade_k;         // the sun's limb at the horizon: clamp((mu_s + fade_c) fade_k)
    float ty, my;                 // transmittance and multiple-scattering rows (texel space)
    F3 wr, wm;                    // weights of the Rayleigh and Mie in-scattering
};

// A row's ray: r_mu_s0 + (near + d) nu is r_d mu_s at distance d (near: the part of the ray above the
// atmosphere).
struct RowRay {
    float r, alt0, mu, dist, r_mu_s0, near;
};
constexpr int kRowSteps = 32;

// The product over the half wave's lanes before this one, and over all of them.
__device__ __forceinline__ float half_wave_product(float x, float& all) {
    const int k = threadIdx.x & 31;
    for (int off = 1; off < 32; off <<= 1) {
        const float y = __shfl_up(x, off, 32);
        if (k >= off) x *= y;
    }
    all = __shfl(x, 31, 32);
    const float before = __shfl_up(x, 1, 32);
    return k == 0 ? 1.0f : before;
}

// Steps [first, first + 32) of the row's n over the 32 lanes of each half wave (lane k: step
// first + k); carry is the transmittance up to step `first`, and becomes the one after these steps.
__device__ inline RowStep row_step(const AtmDev& A, const RowRay& ray, float dx, int n, int first, int tw, int th,
                                   int mh, F3& carry) {
    const int j = first + (threadIdx.x & 31);
    const float d = (0.5f + float(j)) * dx;  // the shader's float counter 0.5, 1.5, ...
    const float q = fmaf(d, d + 2.0f * ray.r * ray.mu, ray.alt0 * (ray.r + A.rb));  // r_d^2 - R_b^2
    RowStep s;
    s.r = fsqrt_fast(fmaxf(q + A.rb * A.rb, 0.0f));
    const float alt = fdiv_fast(q, s.r + A.rb);
    const float inv_r = __builtin_amdgcn_rcpf(s.r);
    s.a0 = ray.r_mu_s0 * inv_r;
    s.a1 = (ray.near + d) * inv_r;
    s.r2 = s.r * s.r;
    s.h2q = fmaxf(A.H2 - q, 0.0f);  // below 0 only by rounding, at the top
    const float rho = fsqrt_fast(fmaxf(q, 0.0f));
    s.d_min = A.thickness - alt;
    s.kx = fdiv_fast(float(tw - 1), rho + A.H - s.d_min);
    const float e = A.rb * inv_r * A.sun_angular_radius;
    s.fade_c = e + rho * inv_r;  // -cos of the horizon's zenith angle = rho / r
    s.fade_k = __builtin_amdgcn_rcpf(2.0f * e);
    s.ty = fminf(fmaxf(rho * A.inv_H * float(th - 1), 0.0f), float(th - 1));
    s.my = fminf(fmaxf(alt * A.inv_thickness * float(mh - 1), 0.0f), float(mh - 1));
    const Densities dn = densities(A, alt);
    const F3 sr = A.rayleigh * dn.rayleigh, sm = A.mie_s * dn.mie;
    const F3 ext = sr + A.mie_ext * dn.mie + A.ozone * dn.ozone;
    const F3 tr = {__expf(-ext.x * dx), __expf(-ext.y * dx), __expf(-ext.z * dx)};
    const bool in = j < n;
    F3 all;
    const F3 before = {half_wave_product(in ? tr.x : 1.0f, all.x), half_wave_product(in ? tr.y : 1.0f, all.y),
                       half_wave_product(in ? tr.z : 1.0f, all.z)};
    const F3 w = carry * before *
                 F3{step_weight(dx, ext.x, ext.x * dx, tr.x), step_weight(dx, ext.y, ext.y * dx, tr.y),
                    step_weight(dx, ext.z, ext.z * dx, tr.z)};
    s.wr = w * sr;
    s.wm = w * sm;
    carry *= all;
    return s;
}

// Trip count of the float counter (0.5, 1.5, ... < steps).
__host__ __device__ inline int row_step_count(float steps) { return steps > 0.5f ? int(ceilf(steps - 0.5f)) : 0; }

// The transmittance LUT's column (texel space, before clamping to the LUT) for the sun at mu_s from a
// step's radius.
__device__ __forceinline__ float sun_column(float r, float r2, float h2q, float d_min, float kx, float mu_s) {
    return (fmaf(-r, mu_s, fsqrt_fast(fmaf(r2 * mu_s, mu_s, h2q))) - d_min) * kx;
}
// smoothstep of the sun's disc crossing the horizon.
__device__ __forceinline__ float sun_fade(float fade_c, float fade_k, float mu_s) {
    const float s = clamp01((mu_s + fade_c) * fade_k);
    return s * s * fmaf(-2.0f, s, 3.0f);
}
// x clamped to [lo, hi] in one instruction (lo for a NaN).
__device__ __forceinline__ float clamp_med3(float x, float lo, float hi) { return __builtin_amdgcn_fmed3f(x, lo, hi); }

// ---------------------------------------------------------------------------
// A wave marches P rays per lane of one row.  The two LUT rows of each step are blended once (the
// vertical half of the bilinear filter) into LDS, over the columns the wave's rays can reach at that
// step, usually a few, so that a ray reads one entry of each.  The columns of several steps are
// blended together, one entry per lane.
// ---------------------------------------------------------------------------
// Entries of a step: its transmittance columns, then its multiple-scattering columns, each range with
// two more than it spans, so the row kernels take LUTs of up to kRowColumns columns together.  An entry
// keeps its colour and the difference to the next entry's: c.x c.y, c.z d.x, d.y d.z.
constexpr int kRowColumns = 288, kRowEntries = kRowColumns + 4;
constexpr int kRowFirst = kRowEntries + 4 * 63;  // what row_entries' last round reads
struct RowLds {
    float4 step[kRowSteps][5];
    int4 fetch[kRowSteps][2];
    float2 entry[kRowEntries][3];
    alignas(4) uint8_t first[(kRowFirst + 3) / 4 * 4];  // 1 at a step's first entry
};
__host__ __device__ inline bool row_luts_fit(int tw, int mw) { return tw + mw <= kRowColumns; }

// The next lane's value (lane 63 keeps its own).
__device__ __forceinline__ float next_lane(float x) {
    const int v = __float_as_int(x);
    return __int_as_float(__builtin_amdgcn_update_dpp(v, v, 0x130 /* wave_shl:1 */, 0xf, 0xf, false));
}

// An LDS address, in bytes, and what lies there.
typedef __attribute__((address_space(3))) char LdsByte;
typedef float LdsPair __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) const LdsPair LdsFloat2;
__device__ __forceinline__ unsigned lds_address(const void* p) { return unsigned(uintptr_t((LdsByte*)p)); }

// The blended rows at position x of the entries at LDS address `base`.
__device__ __forceinline__ F3 row_lookup(unsigned base, float x) {
    static_assert(sizeof(RowLds::entry[0]) == 24, "the stride below");
    unsigned at;  // base + 24 x at full rate (the compiler takes the quarter-rate 64-bit form)
    asm("v_mad_u32_u24 %0, %1, 24, %2" : "=v"(at) : "v"(unsigned(x)), "s"(base));
    LdsFloat2* e = (LdsFloat2*)uintptr_t(at);
    const float t = __builtin_amdgcn_fractf(x);
    const LdsPair a = e[0], b = e[1], c = e[2];
    return {fmaf(t, b.y, a.x), fmaf(t, c.x, a.y), fmaf(t, c.y, b.x)};
}

// A step whose sun is down for every ray of the wave, up for every ray, or in between.
enum { kSunDown = 0, kSunCrossing = 1, kSunUp = 2 };

// One step of P rays; et and em are the LDS addresses of its two entry ranges.
template <int P, int kSun>
__device__ __forceinline__ void row_march(const RowLds& lds, int k, unsigned et, unsigned em, float half_mw,
                                          const float (&nu)[P], F3 (&Sr)[P], F3 (&Sm)[P], F3 (&Sx)[P]) {
    const float4 c0 = lds.step[k][0], c1 = lds.step[k][1], c2 = lds.step[k][2], c3 = lds.step[k][3],
                 c4 = lds.step[k][4];
    const F3 wr = {c3.x, c3.y, c3.z}, wm = {c4.x, c4.y, c4.z}, ws = wr + wm;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const float mu_s = fmaf(c0.y, nu[p], c0.x);
        Sx[p] = fma3(ws, row_lookup(em, clamp_med3(fmaf(mu_s, half_mw, half_mw), c2.z, c2.w) - c2.z), Sx[p]);
        if constexpr (kSun != kSunDown) {  // (down: the fade is 0)
            const float tx = clamp_med3(sun_column(c1.x, c0.z, c0.w, c1.y, c1.z, mu_s), c2.x, c2.y) - c2.x;
            F3 V = row_lookup(et, tx);
            if constexpr (kSun == kSunCrossing) V = V * sun_fade(c1.w, c3.w, mu_s);
            Sr[p] = fma3(wr, V, Sr[p]);
            Sm[p] = fma3(wm, V, Sm[p]);
        }
    }
}

// Blends entries [g0, g0 + 63 N) of the steps whose `fetch` records and `first` marks are in lds, N
// entries per lane with all their texels on the way together; before is the step of entry g0 - 1,
// and becomes the one of the last entry.  Lanes past `total` read the last step's texels and store
// nothing.
template <int N>
__device__ __forceinline__ void row_entry_round(const float4* __restrict__ T, int tw, int th,
                                                const float4* __restrict__ MS, int mw, int mh, int g0, int total,
                                                int& before, RowLds& lds) {
    const int lane = threadIdx.x & 63;
    float4 v0[N], v1[N];
    float t[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int g = g0 + 63 * i + lane;  // lane 63's entry is only there as lane 62's neighbour
        const unsigned long long marks = __ballot(lds.first[g] != 0);
        const int k = before + __popcll(marks & (~0ull >> (63 - lane)));
        before += __popcll(marks & (~0ull >> 1));
        const int4 a = lds.fetch[k][0], b = lds.fetch[k][1];
        const int e = g - a.x;
        const bool is_t = e < a.y;
        const int w = is_t ? tw : mw, h = is_t ? th : mh, row = is_t ? a.z : b.x;
        const int c = row + min(e + (is_t ? a.w : b.y), w - 1);
        const float4* lut = is_t ? T : MS;
        v0[i] = lut[c];
        v1[i] = lut[c + (row + w < w * h ? w : 0)];  // the last row has no next one
        t[i] = __int_as_float(is_t ? b.z : b.w);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int g = g0 + 63 * i + lane;
        const F3 m = {fmaf(t[i], v1[i].x - v0[i].x, v0[i].x), fmaf(t[i], v1[i].y - v0[i].y, v0[i].y),
                      fmaf(t[i], v1[i].z - v0[i].z, v0[i].z)};
        const F3 d = {next_lane(m.x) - m.x, next_lane(m.y) - m.y, next_lane(m.z) - m.z};
        if (lane < 63 && g < total) {
            lds.entry[g][0] = make_float2(m.x, m.y);
            lds.entry[g][1] = make_float2(m.z, d.x);
            lds.entry[g][2] = make_float2(d.y, d.z);
        }
    }
}
__device__ inline void row_entries(const float4* __restrict__ T, int tw, int th, const float4* __restrict__ MS, int mw,
                                   int mh, int first_step, int total, RowLds& lds) {
    int before = first_step - 1;
    for (int g0 = 0; g0 < total;) {  // wave-uniform
        if (total - g0 > 2 * 63) {
            row_entry_round<4>(T, tw, th, MS, mw, mh, g0, total, before, lds);
            g0 += 4 * 63;
        } else {
            row_entry_round<2>(T, tw, th, MS, mw, mh, g0, total, before, lds);
            g0 += 2 * 63;
        }
    }
}

// Luminance of the rays nu[p] of a row (0 < ray.dist), and the row's transmittance.  All 64 lanes call
// it with the same row; nu_lo and nu_hi bound every lane's nu.
// `atm` gives the atmosphere each time it is called for.
template <int P, class Atm>
__device__ inline void row_scatter(const Atm& atm, const float4* __restrict__ T, int tw, int th,
                                   const float4* __restrict__ MS, int mw, int mh, const RowRay& ray, float steps,
                                   const float (&nu)[P], float nu_lo, float nu_hi, RowLds& lds, F3 (&L)[P], F3& Tr) {
    const int lane = threadIdx.x & 63;
    const int n = row_step_count(steps);
    const float dx = ray.dist / steps;
    const float half_mw = 0.5f * float(mw - 1);
    const unsigned entries = __builtin_amdgcn_readfirstlane(lds_address(lds.entry));
    F3 Sr[P], Sm[P], Sx[P];  // Rayleigh, Mie and multiple-scattering sums
#pragma unroll
    for (int p = 0; p < P; ++p) Sr[p] = Sm[p] = Sx[p] = f3(0.0f);
    Tr = f3(1.0f);
    for (int first = 0; first < n; first += kRowSteps) {
        const RowStep s = row_step(atm(), ray, dx, n, first, tw, th, mh, Tr);
        const int count = min(kRowSteps, n - first);
        // The columns that nu_lo .. nu_hi reach: the column falls and the multiple-scattering column
        // rises with mu_s.  A sixteenth of a texel covers the rounding.
        const float mu0 = fmaf(s.a1, nu_lo, s.a0), mu1 = fmaf(s.a1, nu_hi, s.a0);
        const float t0 = sun_column(s.r, s.r2, s.h2q, s.d_min, s.kx, mu1),
                    t1 = sun_column(s.r, s.r2, s.h2q, s.d_min, s.kx, mu0);
        const float t_max = float(tw - 1), m_max = float(mw - 1), eps = 0.0625f;
        const int t_lo = int(fminf(fmaxf(fminf(t0, t1) - eps, 0.0f), t_max));
        const int t_hi = int(fminf(fmaxf(fmaxf(t0, t1) + eps, 0.0f), t_max));
        const int m_lo = int(fminf(fmaxf(fmaf(mu0, half_mw, half_mw) - eps, 0.0f), m_max));
        const int m_hi = int(fminf(fmaxf(fmaf(mu1, half_mw, half_mw) + eps, 0.0f), m_max));
        const int n_t = max(t_hi - t_lo, 0) + 3, n_m = max(m_hi - m_lo, 0) + 3;
        const int ty0 = int(s.ty), my0 = int(s.my);
        // The sun is up for every ray, or down for every ray, where the fade is 1, or 0, at both ends.
        const float lit = mu0 + s.fade_c, dark = mu1 + s.fade_c;
        const int sun = lit * s.fade_k >= 1.0f ? kSunUp : dark * s.fade_k <= 0.0f ? kSunDown : kSunCrossing;
        wave_lds_fence();  // the previous steps' reads
        if (lane < kRowSteps) {
            lds.step[lane][0] = make_float4(s.a0, s.a1, s.r2, s.h2q);
            lds.step[lane][1] = make_float4(s.r, s.d_min, s.kx, s.fade_c);
            lds.step[lane][2] = make_float4(float(t_lo), float(min(t_lo + n_t - 2, tw - 1)), float(m_lo),
                                            float(min(m_lo + n_m - 2, mw - 1)));
            lds.step[lane][3] = make_float4(s.wr.x, s.wr.y, s.wr.z, s.fade_k);
            lds.step[lane][4] = make_float4(s.wm.x, s.wm.y, s.wm.z, 0.0f);
        }
        int end = lane < count ? n_t + n_m : 0;  // inclusive sums of the steps' entries
        for (int off = 1; off < kRowSteps; off <<= 1) {
            const int v = __shfl_up(end, off, 64);
            if (lane >= off && lane < kRowSteps) end += v;
        }
        for (int k0 = 0; k0 < count;) {  // as many steps at a time as the entries hold
            const int base0 = k0 > 0 ? __builtin_amdgcn_readlane(end, k0 - 1) : 0;
            const int k1 = __popcll(__ballot(lane < count && end - base0 <= kRowEntries));
            const int total = __builtin_amdgcn_readlane(end, k1 - 1) - base0;
            wave_lds_fence();
            for (int g = lane; g < (kRowFirst + 3) / 4; g += 64) reinterpret_cast<uint32_t*>(lds.first)[g] = 0u;
            wave_lds_fence();
            if (lane >= k0 && lane < k1) {
                const int base = end - base0 - n_t - n_m;
                lds.fetch[lane][0] = make_int4(base, n_t, ty0 * tw, t_lo);
                lds.fetch[lane][1] = make_int4(my0 * mw, m_lo - n_t, __float_as_int(s.ty - float(ty0)),
                                               __float_as_int(s.my - float(my0)));
                lds.first[base] = 1;
            }
            wave_lds_fence();
            row_entries(T, tw, th, MS, mw, mh, k0, total, lds);
            wave_lds_fence();
            // Runs of steps of one kind, so that the sums stay in their registers.
            const auto run = [&](int k, auto kind) {
                const int stop = min(k1, k + __builtin_ctzll(~(__ballot(sun == kind.value) >> k) | (1ull << 63)));
                for (; k < stop; ++k) {
                    const int nt = __builtin_amdgcn_readlane(n_t, k);
                    const int at = __builtin_amdgcn_readlane(end, k) - base0 - nt - __builtin_amdgcn_readlane(n_m, k);
                    const unsigned et = entries + unsigned(at) * unsigned(sizeof(lds.entry[0])),
                                   em = et + unsigned(nt) * unsigned(sizeof(lds.entry[0]));
                    row_march<P, kind.value>(lds, k, et, em, half_mw, nu, Sr, Sm, Sx);
                }
                return k;
            };
            for (int k = k0; k < k1;) {
                k = run(k, std::integral_constant<int, kSunUp>());
                k = run(k, std::integral_constant<int, kSunCrossing>());
                k = run(k, std::integral_constant<int, kSunDown>());
            }
            k0 = k1;
        }
    }
    const AtmDev A = atm();
#pragma unroll
    for (int p = 0; p < P; ++p)
        L[p] = (rayleigh_phase(nu[p]) * Sr[p] + mie_phase(A.g, nu[p]) * Sm[p] + A.ms_mask * Sx[p]) * A.solar;
}

// Rays per lane for a row of w in a throughput-bound launch: of 1 to 3, the count that leaves the
// fewest lanes idle (the larger at a tie, which shares a step's set-up among more rays).
__host__ __device__ inline int row_rays_per_lane(int w) {
    const int idle2 = (w + 127) / 128 * 128, idle3 = (w + 191) / 192 * 192;
    return w <= 64 ? 1 : idle3 <= idle2 ? 3 : 2;
}

// A pointer the compiler takes for a new one, so that what is read through it is not kept from before.
template <class B>
__device__ __forceinline__ const B* reload(const B* p) {
    asm volatile("" : "+s"(p));
    return p;
}

// The wave's bounds of P values per lane.
template <int P>
__device__ inline void wave_bounds(const float (&v)[P], float& lo, float& hi) {
    lo = hi = v[0];
#pragma unroll
    for (int p = 1; p < P; ++p) {
        lo = fminf(lo, v[p]);
        hi = fmaxf(hi, v[p]);
    }
    for (int off = 32; off >= 1; off >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, off, 64));
        hi = fmaxf(hi, __shfl_xor(hi, off, 64));
    }
}

// The row of rays at zenith cosine mu from radius r (altitude alt0) under a sun at zenith cosine
// mu_s0: its start and length (0: nothing to integrate), with the part above the atmosphere skipped
// (start_from_space).
__device__ inline RowRay row_ray(const AtmDev& A, float r, float alt0, float mu, float mu_s0) {
    const bool hit = ray_hits_ground(A, r, alt0, mu);
    RowRay ray{r, alt0, mu, hit ? distance_to_bottom(A, r, alt0, mu) : distance_to_top(A, r, alt0, mu), r * mu_s0, 0.0f};
    if (r > A.rt) {
        const float disc = r * r * (mu * mu - 1.0f) + A.rt * A.rt;
        if (mu < 0.0f && disc >= 0.0f) {
            ray.near = fmaxf(-r * mu - sqrtf(fmaxf(disc, 0.0f)), 0.0f);
            ray.r = sqrtf(ray.near * ray.near + 2.0f * r * mu * ray.near + r * r);
            ray.mu = (r * mu + ray.near) / ray.r;
            ray.alt0 = ray.r - A.rb;
            ray.dist -= ray.near;
        } else {
            ray.dist = 0.0f;
        }
    }
    return ray;
}

// ---------------------------------------------------------------------------
// Sky view: row iy of the LUT, columns [x0, x0 + 64 P), by one wave.
// ---------------------------------------------------------------------------
struct SkyViewRow {
    SkyViewLatitude lat;
    RowRay ray;
};
__device__ inline SkyViewRow sky_view_row_setup(const AtmDev& A, const RenderDev& R, int iy, int h) {
    const SkyViewLatitude lat = sky_view_latitude(A, R, iy, h);
    return {lat, row_ray(A, R.r, R.r - A.rb, lat.cos_lat, dot(R.sun, R.up))};
}
template <int P, class Atm>
__device__ inline void sky_view_row(const Atm& atm, const RenderDev& R, const SkyViewRow& row,
                                    const float4* __restrict__ T, int tw, int th, const float4* __restrict__ MS, int mw,
                                    int mh, int iy, int x0, int w, RowLds& lds, float4* __restrict__ out_l,
                                    float4* __restrict__ out_t) {
    const int lane = threadIdx.x & 63;
    float nu[P];
#pragma unroll
    for (int p = 0; p < P; ++p) nu[p] = sky_view_nu(R, row.lat, min(x0 + 64 * p + lane, w - 1), w);
    F3 L[P], Tr = f3(1.0f);
    if (row.ray.dist > 0.0f) {  // wave-uniform
        float lo, hi;
        wave_bounds<P>(nu, lo, hi);
        row_scatter<P>(atm, T, tw, th, MS, mw, mh, row.ray, R.sv_steps, nu, lo, hi, lds, L, Tr);
    } else {
#pragma unroll
        for (int p = 0; p < P; ++p) L[p] = f3(0.0f);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int x = x0 + 64 * p + lane;
        if (x < w) {
            out_l[iy * w + x] = make_float4(L[p].x, L[p].y, L[p].z, 0.0f);
            out_t[iy * w + x] = make_float4(Tr.x, Tr.y, Tr.z, 0.0f);
        }
    }
}

// ---------------------------------------------------------------------------
// Multiple scattering: the 64 directions of a texel are 8 polar angles by 8 azimuths, so a row of the
// LUT (one altitude) marches 8 rows of rays, whatever its texel's sun.
// ---------------------------------------------------------------------------
constexpr int kMsThetas = 8;
constexpr int kMsMaxSteps = 64;  // steps the table holds
struct MsStep {                  // one step of one polar angle
    float4 c[4];
};
// Dynamic LDS of a workgroup's tables (none for marches too long for them).
inline size_t ms_table_bytes(float ms_steps) {
    const int n = row_step_count(ms_steps);
    return n > kMsMaxSteps ? 0 : size_t(kMsThetas) * n * sizeof(MsStep);
}
struct MsTotals {                // per polar angle: transmittance, multiple-scattering transfer, the ray
    F3 tr, lf;
    float r, dist;
    bool hit;
};

// The zenith cosine of polar angle t (ms_ray's, for lanes 8 t .. 8 t + 7).
__device__ __forceinline__ float ms_cos_theta(int t) { return 1.0f - 2.0f * ((0.5f + float(t)) / 8.0f); }

// The march of one polar angle, by half a wave.
struct MsMarch {
    RowRay ray;
    bool hit;
    F3 tr, lf;  // so far
};
__device__ inline MsMarch ms_march(const AtmDev& A, int iy, int h, int theta) {
    const float alt0 = (float(iy) / float(h - 1)) * A.thickness, r = alt0 + A.rb, mu = ms_cos_theta(theta);
    const bool hit = ray_hits_ground(A, r, alt0, mu);
    // mu_s at a step is a0 mu_s0 + a1 nu: r_mu_s0 stands for r alone.
    return {RowRay{r, alt0, mu, hit ? distance_to_bottom(A, r, alt0, mu) : distance_to_top(A, r, alt0, mu), r, 0.0f}, hit,
            f3(1.0f), f3(0.0f)};
}
// Steps [first, last) of its n, into row[0] onwards.
__device__ inline void ms_march_steps(const AtmDev& A, MsMarch& m, int n, int first, int last, int tw, int th, MsStep* row) {
    const float iso = 1.0f / (4.0f * kPiF), dx = m.ray.dist / A.ms_steps;
    for (int f = first; f < last; f += kRowSteps) {
        const RowStep s = row_step(A, m.ray, dx, n, f, tw, th, 2, m.tr);
        const int j = f + int(threadIdx.x & 31);
        const F3 ws = s.wr + s.wm;
        F3 sum = j < n ? ws : f3(0.0f);
        for (int off = 16; off >= 1; off >>= 1)
            sum = sum + F3{__shfl_xor(sum.x, off, 32), __shfl_xor(sum.y, off, 32), __shfl_xor(sum.z, off, 32)};
        m.lf += sum;
        if (j < n) {
            MsStep& d = row[j - first];
            d.c[0] = make_float4(s.a0, s.a1, s.r2, s.h2q);
            d.c[1] = make_float4(s.r, s.d_min, s.kx, s.fade_c);
            d.c[2] = make_float4(ws.x * iso, ws.y * iso, ws.z * iso, s.fade_k);
            d.c[3] = make_float4(s.ty, 0.0f, 0.0f, 0.0f);
        }
    }
}
__device__ __forceinline__ MsTotals ms_totals(const MsMarch& m) { return {m.tr, m.lf, m.ray.r, m.ray.dist, m.hit}; }

// Fills `steps` (kMsThetas x n) and `totals` for the altitude of row iy: one (angle, step) per thread.
// Every thread of the workgroup calls it; the caller synchronises.
__device__ inline void ms_row_tables(const AtmDev& A, int iy, int h, int tw, int th, int n, MsStep* steps,
                                     MsTotals* totals) {
    for (int e = threadIdx.x; e < kMsThetas * kRowSteps; e += blockDim.x) {  // half a wave per angle
        const int t = e / kRowSteps;
        MsMarch m = ms_march(A, iy, h, t);
        ms_march_steps(A, m, n, 0, n, tw, th, steps + t * n);
        if ((e & 31) == 0) totals[t] = ms_totals(m);
    }
}

// Steps [first, last) of a texel's 64 directions (the lane's): the luminance they add.
template <bool kCells>
__device__ __forceinline__ F3 ms_row_steps(const float4* __restrict__ T, int tw, int th, const MsStep* steps, int n,
                                           const MsSun& sun, int first, int last) {
    F3 L = f3(0.0f);
    const MsStep* row = steps + ((threadIdx.x & 63) >> 3) * n;
#pragma unroll 2
    for (int j = first; j < last; ++j) {
        const float4 c0 = row[j].c[0], c1 = row[j].c[1], c2 = row[j].c[2];
        const float mu_s = fmaf(c0.y, sun.nu, c0.x * sun.mu_s0);
        const float tx = sun_column(c1.x, c0.z, c0.w, c1.y, c1.z, mu_s);
        const F3 V = lut_bilinear<kCells>(T, tw, th, tx, row[j].c[3].x) * sun_fade(c1.w, c2.w, mu_s);
        L = fma3(F3{c2.x, c2.y, c2.z}, V, L);
    }
    return L;
}

// A row texel from the luminance of its 64 directions (ms_row_steps'; the lane's).  Valid in lane 0.
template <bool kCells>
__device__ __forceinline__ float4 ms_row_reduce(const AtmDev& A, const float4* __restrict__ T, int tw, int th,
                                                const MsTotals* totals, const MsSun& sun, F3 L) {
    const MsTotals t = totals[(threadIdx.x & 63) >> 3];
    const MsRay ray{RayStart{t.r, 0.0f, 0.0f, sun.mu_s0, sun.nu}, t.dist, t.hit};
    return multiscattering_reduce<kCells>(A, T, tw, th, ray, L, t.tr, t.lf);
}

}  // namespace skyhip
