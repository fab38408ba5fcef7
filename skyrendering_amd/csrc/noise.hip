// Cloud-texture generators for gfx950 (NoiseGen.comp + shaders/Base/Noise.glsl):
// the 2D cloud map (RG8: Perlin-FBM coverage, Worley-FBM type), the 3D detail
// volume (R8 Perlin-Worley), the 3D Worley detail volume (R8 Worley-FBM) and the 2D
// displacement map (RGBA8 Perlin-FBM),
// plus the box-filter mip chain builder.  One lane per texel, workgroups over tiles of texels that
// share their octaves' hashes.  Hashes are
// exact uint32 arithmetic; FBM sums run in FP32 as in the shader.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "common.h"

namespace skyhip {

__device__ __forceinline__ uint32_t wang_hash(uint32_t seed) {
    seed = (seed ^ 61u) ^ (seed >> 16);
    seed *= 9u;
    seed = seed ^ (seed >> 4);
    seed *= 0x27d4eb2du;
    seed = seed ^ (seed >> 15);
    return seed;
}

// A gradient of Noise.glsl:17-22 dotted with (x, y, z).  The table's 16 entries are 12 distinct
// gradients, +-u +-v with (u, v) = (x, y) for 0..3, (x, z) for 4..7 and (y, z) for 8..11, the signs
// in bits 0 and 1; entries 12..15 repeat 0, 1, 9 and 11 (perlin_gradient).
__device__ __forceinline__ uint32_t perlin_gradient(uint32_t h) {
    const uint32_t i = h & 15u;
    return i < 12u ? i : (0xb910u >> (4u * (i - 12u))) & 15u;
}
__device__ __forceinline__ float perlin_grad_dot(uint32_t g, float x, float y, float z) {
    const float u = g < 8u ? x : y, v = g < 4u ? y : z;
    return __uint_as_float(__float_as_uint(u) ^ (g << 31)) + __uint_as_float(__float_as_uint(v) ^ ((g & 2u) << 30));
}

__device__ __forceinline__ float gmixf(float a, float b, float t) { return a * (1.0f - t) + b * t; }

// ---------------------------------------------------------------------------
// Octaves by tile.  A workgroup covers a TX x TY x TZ tile of texels, and an octave's hashes depend
// on lattice cells, which neighbouring texels share: the tile's cells are hashed once into LDS and
// the texels read them there.  The reference's chains are H(seed + H(x + H(y + H(z)))), so their
// (y, z) parts are a table of their own (`hash`), filled first; where the whole cell table does not
// fit (an octave finer than the texels, whose texels share no cells) the texels finish the chain from
// the (y, z) table, and where that does not fit either they hash for themselves.
// Calls whose octaves share too little go by texels throughout (tiles_pay).
// Bound by the integer hashes (a 3D Worley octave is 198 per texel without sharing, each about 10
// instructions with a quarter-rate multiply).  Same hashes and float operations as the reference's
// texel-by-texel form, so the same bytes.  Measured: detail 128^3 1,090 -> 520 us (its two finest
// octaves, whose texels share no cells, are half of what is left), cloud map 512^2 130 -> 59 us,
// Worley 32^3 35 -> 28 us; all textures of the default material 1,331 -> 665 us.
// The tables hold 1,024 columns and 1,536 cells (30 KiB, five workgroups per CU): a 256-texel tile
// of a 128^3 volume fits them up to one octave beyond the texels' own density, past which filling the
// table would hash as many cells as the texels do themselves.
// ---------------------------------------------------------------------------
constexpr int kMaxPairs = 1024;   // (y, z) columns of a tile's cells
constexpr int kMaxCells = 1536;
template <bool kTiles>
struct NoiseTables {
    uint32_t hash[3][kMaxPairs];
    float cell[3][kMaxCells];  // Worley feature points; Perlin keeps its gradients in cell[0]
};
// By texels: no tables, and the gradients as they are, a read and three products each (14 instructions of
// perlin_grad_dot, which latency hides better, in the tiles).
template <>
struct NoiseTables<false> {
    float4 gradient[16];
};
__device__ __forceinline__ void fill_gradients(float4 (&g)[16]) {
    if (threadIdx.x < 16) {
        const uint32_t i = perlin_gradient(threadIdx.x);
        g[threadIdx.x] = make_float4(perlin_grad_dot(i, 1.0f, 0.0f, 0.0f), perlin_grad_dot(i, 0.0f, 1.0f, 0.0f),
                                     perlin_grad_dot(i, 0.0f, 0.0f, 1.0f), 0.0f);
    }
    __syncthreads();
}
__device__ __forceinline__ float gradient_dot(const float4 (&g)[16], uint32_t h, float x, float y, float z) {
    const float4 v = g[h & 15u];
    return fmaf(v.z, z, fmaf(v.y, y, v.x * x));
}

// One octave's cells over the tile along each axis: base[a] + [0, n[a]), from the cell coordinates
// of the tile's first and last texels (the texels' own float operations, monotonic in the texel).
struct CellRange {
    uint32_t base[3], n[3];
    bool pairs, cells;
};
struct NoiseTile {
    float lo[3], hi[3];  // coordinates of the tile's first and last texel
    float p[3];          // this thread's texel
};

__device__ __forceinline__ CellRange cell_range(const NoiseTile& t, uint32_t freq, uint32_t extra) {
    CellRange r;
    for (int a = 0; a < 3; ++a) {
        r.base[a] = uint32_t(floorf(t.lo[a] * float(freq)));
        r.n[a] = uint32_t(floorf(t.hi[a] * float(freq))) - r.base[a] + extra;
    }
    r.pairs = r.n[1] <= uint32_t(kMaxPairs) && r.n[2] <= uint32_t(kMaxPairs) && r.n[1] * r.n[2] <= uint32_t(kMaxPairs);
    r.cells = r.pairs && r.n[0] <= uint32_t(kMaxCells) && r.n[0] * r.n[1] * r.n[2] <= uint32_t(kMaxCells);
    return r;
}

// v % freq for v < 2 freq.
__device__ __forceinline__ uint32_t wrap_once(uint32_t v, uint32_t freq) { return min(v, v - freq); }
// v % freq for v < 3 freq (a division below frequency 4, where v can be larger).
__device__ __forceinline__ uint32_t wrap_cell(uint32_t v, uint32_t freq) {
    if (freq < 4u) return v % freq;
    if (v >= freq) v -= freq;
    return v >= freq ? v - freq : v;
}

// The noise at (tx, ty, tz) of a cell; dot(c, x, y, z) dots the gradient of corner c = x + 2 y + 4 z.
template <class Dot>
__device__ __forceinline__ float perlin_mix(const Dot& dot, float tx, float ty, float tz) {
    const float u = tx * tx * tx * (tx * (tx * 6.0f - 15.0f) + 10.0f);
    const float v = ty * ty * ty * (ty * (ty * 6.0f - 15.0f) + 10.0f);
    const float w = tz * tz * tz * (tz * (tz * 6.0f - 15.0f) + 10.0f);
    const float x1 = tx - 1.0f, y1 = ty - 1.0f, z1 = tz - 1.0f;
    const float n000 = dot(0, tx, ty, tz), n100 = dot(1, x1, ty, tz);
    const float n010 = dot(2, tx, y1, tz), n110 = dot(3, x1, y1, tz);
    const float n001 = dot(4, tx, ty, z1), n101 = dot(5, x1, ty, z1);
    const float n011 = dot(6, tx, y1, z1), n111 = dot(7, x1, y1, z1);
    return gmixf(gmixf(gmixf(n000, n100, u), gmixf(n010, n110, u), v),
                 gmixf(gmixf(n001, n101, u), gmixf(n011, n111, u), v), w);
}

// PerlinNoise, Noise.glsl:28-60 (p >= 0 here: texture coordinates in [0, 1)).  The far corner is
// cell + 1 where the reference takes ceil: they differ only at integer coordinates, where the
// corner's weight is 0.
template <bool kTiles>
__device__ inline float perlin_octave(NoiseTables<kTiles>& s, const NoiseTile& t, uint32_t freq, uint32_t seed) {
    const float px = t.p[0] * float(freq), py = t.p[1] * float(freq), pz = t.p[2] * float(freq);
    const float fx = floorf(px), fy = floorf(py), fz = floorf(pz);
    const float tx = px - fx, ty = py - fy, tz = pz - fz;
    const uint32_t ix = uint32_t(int(fx)), iy = uint32_t(int(fy)), iz = uint32_t(int(fz));
    const uint32_t x0 = wrap_once(ix, freq), x1 = wrap_once(x0 + 1u, freq);
    uint32_t hjk[4];  // column y + 2 z
    const auto columns = [&] {
        const uint32_t y0 = wrap_once(iy, freq), z0 = wrap_once(iz, freq), y1 = wrap_once(y0 + 1u, freq);
        const uint32_t hk0 = wang_hash(z0), hk1 = wang_hash(wrap_once(z0 + 1u, freq));
        hjk[0] = wang_hash(y0 + hk0), hjk[1] = wang_hash(y1 + hk0);
        hjk[2] = wang_hash(y0 + hk1), hjk[3] = wang_hash(y1 + hk1);
    };
    const auto corner = [&](int c) { return wang_hash(seed + wang_hash((c & 1 ? x1 : x0) + hjk[c >> 1])); };
    if constexpr (!kTiles) {
        columns();
        return perlin_mix([&](int c, float x, float y, float z) { return gradient_dot(s.gradient, corner(c), x, y, z); },
                          tx, ty, tz);
    } else {
        const CellRange r = cell_range(t, freq, 2u);
        uint8_t* grad = reinterpret_cast<uint8_t*>(s.cell[0]);
        if (r.pairs) {
            __syncthreads();  // the previous octave's reads
            for (uint32_t k = threadIdx.x; k < r.n[1] * r.n[2]; k += 256) {
                const uint32_t cz = k / r.n[1], cy = k - cz * r.n[1];
                s.hash[0][k] = wang_hash(wrap_cell(r.base[1] + cy, freq) + wang_hash(wrap_cell(r.base[2] + cz, freq)));
            }
            __syncthreads();
        }
        if (r.cells) {
            for (uint32_t k = threadIdx.x; k < r.n[0] * r.n[1] * r.n[2]; k += 256) {
                const uint32_t pair = k / r.n[0], cx = k - pair * r.n[0];
                grad[k] = uint8_t(perlin_gradient(
                    wang_hash(seed + wang_hash(wrap_cell(r.base[0] + cx, freq) + s.hash[0][pair]))));
            }
            __syncthreads();
        }
        uint32_t g[8];
        if (r.cells) {
            const uint32_t at = ((iz - r.base[2]) * r.n[1] + (iy - r.base[1])) * r.n[0] + (ix - r.base[0]);
            const uint32_t sy = r.n[0], sz = r.n[0] * r.n[1];
            for (uint32_t c = 0; c < 8; ++c) g[c] = grad[at + (c & 1u) + ((c >> 1) & 1u) * sy + (c >> 2) * sz];
        } else {
            if (r.pairs) {
                const uint32_t at = (iz - r.base[2]) * r.n[1] + (iy - r.base[1]);
                for (uint32_t c = 0; c < 4; ++c) hjk[c] = s.hash[0][at + (c & 1u) + (c >> 1) * r.n[1]];
            } else {
                columns();
            }
#pragma unroll
            for (int c = 0; c < 8; ++c) g[c] = perlin_gradient(corner(c));
        }
        return perlin_mix([&](int c, float x, float y, float z) { return perlin_grad_dot(g[c], x, y, z); }, tx, ty, tz);
    }
}

// The reference's random float of a hash.
__device__ __forceinline__ float hash_to_unit(uint32_t h) { return float(h) * 2.3283064365386963e-10f; }

// WorleyNoise (3D), Noise.glsl:81-101: the nearest feature point of the 27 cells around p, shifted
// up by one period as the reference shifts it (the feature point of cell g is g + a fraction).
template <bool kTiles>
__device__ inline float worley_octave(NoiseTables<kTiles>& s, const NoiseTile& t, uint32_t freq, uint32_t seed) {
    const uint32_t off = freq - 1u;
    float px = t.p[0] * float(freq), py = t.p[1] * float(freq), pz = t.p[2] * float(freq);
    const uint32_t ix = uint32_t(floorf(px)), iy = uint32_t(floorf(py)), iz = uint32_t(floorf(pz));
    px += float(freq);
    py += float(freq);
    pz += float(freq);
    float min_d2 = 1e20f;
    const uint32_t sx0 = wrap_once(ix + off, freq), sx1 = wrap_once(sx0 + 1u, freq),
                   sx[3] = {sx0, sx1, wrap_once(sx1 + 1u, freq)};
    const auto column = [&](uint32_t dj, uint32_t dk, const uint32_t (&hy)[3]) {
#pragma unroll
        for (uint32_t di = 0; di < 3; ++di) {
            const float dx = px - (float(ix + off + di) + hash_to_unit(wang_hash(seed + wang_hash(sx[di] + hy[0]))));
            const float dy = py - (float(iy + off + dj) + hash_to_unit(wang_hash(seed + wang_hash(sx[di] + hy[1]))));
            const float dz = pz - (float(iz + off + dk) + hash_to_unit(wang_hash(seed + wang_hash(sx[di] + hy[2]))));
            min_d2 = fminf(min_d2, dx * dx + dy * dy + dz * dz);
        }
    };
    if constexpr (kTiles) {
        const CellRange r = cell_range(t, freq, 3u);  // cells base - 1 .. of the shifted coordinates
        if (r.pairs) {
            __syncthreads();  // the previous octave's reads
            for (uint32_t k = threadIdx.x; k < r.n[1] * r.n[2]; k += 256) {
                const uint32_t cz = k / r.n[1], cy = k - cz * r.n[1];
                const uint32_t sz = wrap_cell(r.base[2] + off + cz, freq), sy = wrap_cell(r.base[1] + off + cy, freq);
                for (uint32_t c = 0; c < 3; ++c) s.hash[c][k] = wang_hash(sy + wang_hash(sz + c));
            }
            __syncthreads();
        }
        const uint32_t lx = ix - r.base[0], ly = iy - r.base[1], lz = iz - r.base[2];
        if (r.cells) {
            for (uint32_t k = threadIdx.x; k < r.n[0] * r.n[1] * r.n[2]; k += 256) {
                const uint32_t pair = k / r.n[0], cx = k - pair * r.n[0];
                const uint32_t cell = wrap_cell(r.base[0] + off + cx, freq);
                for (uint32_t c = 0; c < 3; ++c)
                    s.cell[c][k] = hash_to_unit(wang_hash(seed + wang_hash(cell + s.hash[c][pair])));
            }
            __syncthreads();
            const uint32_t at0 = (lz * r.n[1] + ly) * r.n[0] + lx;
#pragma unroll
            for (uint32_t dk = 0; dk < 3; ++dk)
#pragma unroll
                for (uint32_t dj = 0; dj < 3; ++dj) {
                    const uint32_t at = at0 + (dk * r.n[1] + dj) * r.n[0];
#pragma unroll
                    for (uint32_t di = 0; di < 3; ++di) {
                        const float dx = px - (float(ix + off + di) + s.cell[0][at + di]);
                        const float dy = py - (float(iy + off + dj) + s.cell[1][at + di]);
                        const float dz = pz - (float(iz + off + dk) + s.cell[2][at + di]);
                        min_d2 = fminf(min_d2, dx * dx + dy * dy + dz * dz);
                    }
                }
            return sqrtf(min_d2);
        }
        if (r.pairs) {
            for (uint32_t dk = 0; dk < 3; ++dk)
                for (uint32_t dj = 0; dj < 3; ++dj) {
                    const uint32_t at = (lz + dk) * r.n[1] + ly + dj;
                    const uint32_t hy[3] = {s.hash[0][at], s.hash[1][at], s.hash[2][at]};
                    column(dj, dk, hy);
                }
            return sqrtf(min_d2);
        }
    }
    uint32_t sz = wrap_once(iz + off, freq);
    for (uint32_t dk = 0; dk < 3; ++dk) {
        const uint32_t hz[3] = {wang_hash(sz), wang_hash(sz + 1u), wang_hash(sz + 2u)};
        uint32_t sy = wrap_once(iy + off, freq);
        for (uint32_t dj = 0; dj < 3; ++dj) {
            const uint32_t hy[3] = {wang_hash(sy + hz[0]), wang_hash(sy + hz[1]), wang_hash(sy + hz[2])};
            column(dj, dk, hy);
            sy = wrap_once(sy + 1u, freq);
        }
        sz = wrap_once(sz + 1u, freq);
    }
    return sqrtf(min_d2);
}

__device__ __forceinline__ float remap_to01(float x, float x0, float x1) {
    return fminf(fmaxf((x - x0) / (x1 - x0), 0.0f), 1.0f);
}

// PerlinFBM / WorleyFBM, NoiseGen.comp:20-50 (8 octaves).  Every thread of the workgroup calls them.
template <bool kTiles>
__device__ inline float perlin_fbm(NoiseTables<kTiles>& s, const NoiseTile& t, const SkyhipNoiseCreateInfo& ci) {
    float res = 0.0f, a = 0.5f, sum_a = 0.0f;
    uint32_t f = ci.base_frequency;
    for (int c = 0; c < 8; ++c) {
        float n = perlin_octave<kTiles>(s, t, f, ci.seed) * 0.5f + 0.5f;
        res += remap_to01(n, ci.remap_min, ci.remap_max) * a;
        sum_a += a;
        f *= 2u;
        a *= 0.5f;
    }
    return res / sum_a;
}
template <bool kTiles>
__device__ inline float worley_fbm(NoiseTables<kTiles>& s, const NoiseTile& t, const SkyhipNoiseCreateInfo& ci) {
    float res = 0.0f, a = 0.5f, sum_a = 0.0f;
    uint32_t f = ci.base_frequency;
    for (int c = 0; c < 8; ++c) {
        float n = worley_octave<kTiles>(s, t, f, ci.seed);
        res += remap_to01(n, ci.remap_min, ci.remap_max) * a;
        sum_a += a;
        f *= 2u;
        a *= 0.5f;
    }
    return res / sum_a;
}

__device__ __forceinline__ uint8_t to_unorm8(float f) {
    return uint8_t(floorf(fminf(fmaxf(f, 0.0f), 1.0f) * 255.0f + 0.5f));
}

// The tile of a workgroup of TX x TY x TZ threads, x fastest, at `tile` tiles of a dims-sized texture,
// and this thread's texel.  Threads past the edge take the coordinates of the last texel (they still
// hash and synchronise) and store nothing.  Coordinates are texel centres; an axis of size 0 is the
// plane 0 of a 2D texture.
struct TexelPos {
    int x, y, z;
    bool in;
};
template <int TX, int TY, int TZ>
__device__ inline TexelPos noise_tile(int tx, int ty, int tz, const int dims[3], NoiseTile& t) {
    const int id = threadIdx.x;
    const int first[3] = {tx * TX, ty * TY, tz * TZ}, edge[3] = {TX, TY, TZ};
    const int at[3] = {first[0] + id % TX, first[1] + (id / TX) % TY, first[2] + id / (TX * TY)};
    TexelPos p{at[0], at[1], at[2], true};
    for (int a = 0; a < 3; ++a) {
        if (dims[a] == 0) {
            t.lo[a] = t.hi[a] = t.p[a] = 0.0f;
            continue;
        }
        const int last = min(first[a] + edge[a], dims[a]) - 1;
        t.lo[a] = (float(first[a]) + 0.5f) / float(dims[a]);
        t.hi[a] = (float(last) + 0.5f) / float(dims[a]);
        t.p[a] = (float(min(at[a], last)) + 0.5f) / float(dims[a]);
        p.in = p.in && at[a] < dims[a];
    }
    return p;
}

// Tiles of 256 texels: 16 x 16 of an image, 8 x 8 x 4 of a volume.
constexpr int kImageTile = 16, kVolumeTileXY = 8, kVolumeTileZ = 4;
__device__ inline TexelPos image_tile(int size, NoiseTile& t) {
    const int dims[3] = {size, size, 0};
    return noise_tile<kImageTile, kImageTile, 1>(blockIdx.x, blockIdx.y, 0, dims, t);
}
__device__ inline TexelPos volume_tile(int nx, int ny, int nz, NoiseTile& t) {
    const int dims[3] = {nx, ny, nz};
    return noise_tile<kVolumeTileXY, kVolumeTileXY, kVolumeTileZ>(blockIdx.x, blockIdx.y, blockIdx.z, dims, t);
}

// The image kernels give each channel its own workgroups (blockIdx.z): an image has few tiles, and a
// tile's octaves follow one another through barriers.  128^2 displacement: 13.6 us, 47.8 with a tile's
// four channels in one workgroup (17.5 with every texel hashing for itself).
template <bool kTiles>
__global__ __launch_bounds__(256) void cloud_map_kernel(SkyhipNoiseCreateInfo density, SkyhipNoiseCreateInfo height,
                                                        uint8_t* __restrict__ out, int size) {
    __shared__ NoiseTables<kTiles> s;
    if constexpr (!kTiles) fill_gradients(s.gradient);
    NoiseTile t;
    const TexelPos p = image_tile(size, t);
    const float v = blockIdx.z == 0 ? perlin_fbm<kTiles>(s, t, density) : worley_fbm<kTiles>(s, t, height);
    if (p.in) out[2ll * (p.y * size + p.x) + blockIdx.z] = to_unorm8(v);
}

template <bool kTiles>
__global__ __launch_bounds__(256) void detail_kernel(SkyhipNoiseCreateInfo perlin, SkyhipNoiseCreateInfo worley,
                                                     uint8_t* __restrict__ out, int size) {
    __shared__ NoiseTables<kTiles> s;
    if constexpr (!kTiles) fill_gradients(s.gradient);
    NoiseTile t;
    const TexelPos at = volume_tile(size, size, size, t);
    float p = perlin_fbm<kTiles>(s, t, perlin);
    float w = worley_fbm<kTiles>(s, t, worley);
    if (at.in)  // RemapFrom01(p, w, 1)
        out[((long long)at.z * size + at.y) * size + at.x] = to_unorm8(fminf(fmaxf(w + p * (1.0f - w), 0.0f), 1.0f));
}

// The Worley detail volume: WorleyFBM alone at texel centres, UNORM8.
template <bool kTiles>
__global__ __launch_bounds__(256) void worley_kernel(SkyhipNoiseCreateInfo worley, uint8_t* __restrict__ out,
                                                     int size) {
    __shared__ NoiseTables<kTiles> s;
    NoiseTile t;
    const TexelPos at = volume_tile(size, size, size, t);
    const uint8_t v = to_unorm8(worley_fbm<kTiles>(s, t, worley));
    if (at.in) out[((long long)at.z * size + at.y) * size + at.x] = v;
}

__global__ __launch_bounds__(256) void displacement_kernel(SkyhipNoiseCreateInfo perlin, uint8_t* __restrict__ out,
                                                           int size) {
    __shared__ NoiseTables<true> s;
    NoiseTile t;
    const TexelPos p = image_tile(size, t);
    perlin.seed += blockIdx.z;
    const uint8_t v = to_unorm8(perlin_fbm<true>(s, t, perlin));
    if (p.in) out[4ll * (p.y * size + p.x) + blockIdx.z] = v;
}

// The same by texels: the channels' seeds enter in the last hash alone, so a texel's four channels share the
// chains before it.
__global__ __launch_bounds__(256) void displacement_texels_kernel(SkyhipNoiseCreateInfo perlin,
                                                                  uint8_t* __restrict__ out, int size) {
    __shared__ float4 gradient[16];
    fill_gradients(gradient);
    const int i = int(blockIdx.x * 256 + threadIdx.x);
    if (i >= size * size) return;
    const float x = (float(i % size) + 0.5f) / float(size), y = (float(i / size) + 0.5f) / float(size);
    float res[4] = {0.0f, 0.0f, 0.0f, 0.0f}, a = 0.5f, sum_a = 0.0f;
    uint32_t f = perlin.base_frequency;
    for (int o = 0; o < 8; ++o) {
        const float px = x * float(f), py = y * float(f), fx = floorf(px), fy = floorf(py);
        const float tx = px - fx, ty = py - fy;
        const uint32_t x0 = wrap_once(uint32_t(int(fx)), f), y0 = wrap_once(uint32_t(int(fy)), f);
        const uint32_t x1 = wrap_once(x0 + 1u, f), y1 = wrap_once(y0 + 1u, f);
        const uint32_t hk0 = wang_hash(0u), hk1 = wang_hash(wrap_once(1u, f));
        const uint32_t hjk[4] = {wang_hash(y0 + hk0), wang_hash(y1 + hk0), wang_hash(y0 + hk1), wang_hash(y1 + hk1)};
        uint32_t h[8];  // corner x + 2 y + 4 z
#pragma unroll
        for (int c = 0; c < 4; ++c) h[2 * c] = wang_hash(x0 + hjk[c]), h[2 * c + 1] = wang_hash(x1 + hjk[c]);
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const auto dot = [&](int c, float gx, float gy, float gz) {
                return gradient_dot(gradient, wang_hash(perlin.seed + k + h[c]), gx, gy, gz);
            };
            res[k] += remap_to01(perlin_mix(dot, tx, ty, 0.0f) * 0.5f + 0.5f, perlin.remap_min, perlin.remap_max) * a;
        }
        sum_a += a;
        f *= 2u;
        a *= 0.5f;
    }
    reinterpret_cast<uchar4*>(out)[i] = make_uchar4(to_unorm8(res[0] / sum_a), to_unorm8(res[1] / sum_a),
                                                    to_unorm8(res[2] / sum_a), to_unorm8(res[3] / sum_a));
}

// One mip step of a UNORM8 texture: box over 2x2(x2) source texels (indices clamped to the source level),
// (sum + n/2) / n.  A lane per byte of the level, neighbouring lanes at neighbouring bytes.
template <int kDims, int kChannels>
__global__ __launch_bounds__(256) void downsample_level_kernel(const uint8_t* __restrict__ src, int sx, int sy, int sz,
                                                               uint8_t* __restrict__ dst, int dx, int dy, int dz) {
    constexpr int kBox = kDims == 3 ? 8 : 4;
    const unsigned t = blockIdx.x * 256u + threadIdx.x;  // the level's bytes fit 32 bits (the launch's)
    if (t >= unsigned(dx) * unsigned(dy) * unsigned(dz) * unsigned(kChannels)) return;
    const unsigned texel = t / kChannels, c = t - texel * kChannels, row = texel / unsigned(dx);
    const int x = int(texel - row * unsigned(dx));
    const unsigned uz = kDims == 3 ? row / unsigned(dy) : 0u;
    const int z = int(uz), y = int(row - uz * unsigned(dy));
    int sum = 0;
#pragma unroll
    for (int k = 0; k < kBox; ++k) {
        const int xx = min(2 * x + (k & 1), sx - 1), yy = min(2 * y + ((k >> 1) & 1), sy - 1);
        const int zz = kDims == 3 ? min(2 * z + ((k >> 2) & 1), sz - 1) : 0;
        sum += src[(((long long)zz * sy + yy) * sx + xx) * kChannels + c];
    }
    dst[t] = uint8_t((sum + kBox / 2) / kBox);
}

// Up to kMipLevels mip steps in one launch.  A workgroup computes a tile of the first level (2^kTileLog texels
// a side) from the source in memory, and, a tile's edge being even, its part of the next levels from
// the one before in LDS.  Bound by launches: an edit's four chains (512^2, two of 128
// and 32 a side) are 11 launches of 4.4 to 4.9 us; a launch per level made 28 of 1 to 4 us, and the edit
// 664 against 619 us.  (Tiles of 32 x 32 texels and a run-time channel count: 650 us.)
constexpr int kMipLevels = 3;
template <int kDims, int kChannels>
__global__ __launch_bounds__(256) void downsample_kernel(const uint8_t* __restrict__ src, int sx, int sy, int sz,
                                                         uint8_t* __restrict__ dst, int levels) {
    constexpr int channels = kChannels, kTileLog = kDims == 3 ? 3 : 4, kTexels = 1 << (kTileLog * kDims), kBox = kDims == 3 ? 8 : 4;
    __shared__ uint8_t s_a[kTexels * channels], s_b[kTexels * channels / kBox];
    int ox = int(blockIdx.x) << kTileLog, oy = int(blockIdx.y) << kTileLog, oz = int(blockIdx.z) << kTileLog;
    if (kDims == 2) oz = 0;
    for (int l = 0; l < levels; ++l) {
        const int dx = max(sx / 2, 1), dy = max(sy / 2, 1), dz = max(sz / 2, 1);
        const int log = kTileLog - l;  // the tile's texels a side: 2^log here, 2^(log + 1) in the source
        const uint8_t* from = (l & 1) ? s_a : s_b;
        uint8_t* to = (l & 1) ? s_b : s_a;
        for (int t = threadIdx.x; t < (channels << (log * kDims)); t += 256) {
            const int texel = t / channels, c = t - texel * channels;
            const int tx = texel & ((1 << log) - 1), ty = (texel >> log) & ((1 << log) - 1),
                      tz = kDims == 3 ? texel >> (2 * log) : 0;
            const int x = ox + tx, y = oy + ty, z = oz + tz;
            if (x >= dx || y >= dy || z >= dz) continue;
            int sum = 0;
            for (int k = 0; k < kBox; ++k) {
                int xx = min(2 * x + (k & 1), sx - 1), yy = min(2 * y + ((k >> 1) & 1), sy - 1);
                int zz = kDims == 3 ? min(2 * z + ((k >> 2) & 1), sz - 1) : 0;
                if (l == 0) {
                    sum += src[(((long long)zz * sy + yy) * sx + xx) * channels + c];
                } else {
                    xx -= 2 * ox, yy -= 2 * oy, zz -= 2 * oz;
                    sum += from[((((zz << (log + 1)) + yy) << (log + 1)) + xx) * channels + c];
                }
            }
            const uint8_t v = uint8_t((sum + kBox / 2) / kBox);
            dst[(((long long)z * dy + y) * dx + x) * channels + c] = v;
            to[t] = v;
        }
        dst += (long long)dx * dy * dz * channels;
        sx = dx, sy = dy, sz = dz;
        ox >>= 1, oy >>= 1, oz >>= 1;
        __syncthreads();
    }
}

// The path-tracing workload's voxel-cloud density (see SkyhipVoxelGridCreateInfo):
// fBm of PerlinNoise (unremapped), lognormal transform, ellipsoidal falloff,
// threshold, FP16 round-to-nearest-even.  One lane per texel.
template <bool kTiles>
__global__ __launch_bounds__(256) void voxel_grid_kernel(SkyhipVoxelGridCreateInfo ci, uint16_t* __restrict__ out,
                                                         int nx, int ny, int nz) {
    __shared__ NoiseTables<kTiles> s;
    if constexpr (!kTiles) fill_gradients(s.gradient);
    NoiseTile t;
    const TexelPos at = volume_tile(nx, ny, nz, t);
    float res = 0.0f, a = 1.0f, sum_a = 0.0f;
    uint32_t f = ci.base_frequency;
    for (int o = 0; o < ci.octaves; ++o) {
        res += perlin_octave<kTiles>(s, t, f, ci.seed) * a;
        sum_a += a;
        f *= 2u;
        a *= 0.5f;
    }
    float fbm = res / sum_a;
    float e = 0.0f;
    for (int k = 0; k < 3; ++k) {
        float q = (t.p[k] - ci.ellipsoid_center[k]) / ci.ellipsoid_radii[k];
        e += q * q;
    }
    float falloff = fmaxf(1.0f - e, 0.0f);
    float density = fmaxf(expf(ci.lognormal_sigma * ci.fbm_inv_std * fbm) * falloff - ci.threshold, 0.0f);
    if (at.in)
        out[((long long)at.z * ny + at.y) * nx + at.x] = __builtin_bit_cast(uint16_t, __float2half_rn(density));
}

dim3 image_grid(int size, int channels) {
    return dim3(div_up(size, kImageTile), div_up(size, kImageTile), unsigned(channels));
}
dim3 volume_grid(int nx, int ny, int nz) {
    return dim3(div_up(nx, kVolumeTileXY), div_up(ny, kVolumeTileXY), div_up(nz, kVolumeTileZ));
}

// Levels the next launch of a chain makes by tiles, or 0 for one level by bytes: tiles save launches (3.1 us
// each), bytes are read and stored faster, and a thin level fills little of a tile.  us, level by level /
// by tiles: one level of 512^2 3.6 / 3.6, three 9.6 / 3.8; three of 2048^2 (4,096 tiles) 9.8 / 7.5, of
// 4096^2 17.1 / 21.5 and with four channels 39.3 / 35.8, of 1 x 2^20 texels of four bytes (32,768 tiles)
// 10.5 / 60.9; three of 128^3 (512) 9.8 / 5.3, of 256^3 (4,096) 14.7 / 24.0; two of 64^3 with four channels
// 6.7 / 7.5.  (Below 4 GiB no grid of tiles has more than 8,192 in y or z.)
int mip_tile_levels(int dims, int channels, int dx, int dy, int dz, int remaining) {
    const int edge = dims == 3 ? 8 : 16;
    const bool full = dx >= edge && dy >= edge;
    if ((long long)dx * dy * dz * channels > (1ll << 32) - 256) return std::min(kMipLevels, remaining);  // the bytes' index
    if (dims == 2 && channels == 4 && full && std::max(dx, dy) <= 1 << 14) return std::min(kMipLevels, remaining);
    const long long tiles = (long long)div_up(dx, edge) * div_up(dy, edge) * div_up(dz, dims == 3 ? edge : 1);
    const int most = dims == 3 ? 1024 : full ? 8192 : remaining > 2 ? 4096 : 2048;
    return tiles <= most && remaining >= (dims == 3 && channels > 2 ? 3 : 2) ? std::min(kMipLevels, remaining) : 0;
}

// Hashes per texel of a call's octaves, by tiles and by texels.
struct NoiseCost {
    double tiles = 0.0, texels = 0.0;
};
void add_octaves(NoiseCost& c, const int (&edge)[3], const int (&dims)[3], uint32_t base_frequency, int octaves, bool worley) {
    const double pair_hashes = worley ? 6.0 : 2.0, texel_hashes = worley ? 198.0 : 22.0, after_pairs = worley ? 162.0 : 16.0;
    for (int o = 0; o < octaves; ++o) {
        double n[3];  // mean cells of a tile along each axis (cell_range)
        for (int a = 0; a < 3; ++a)
            n[a] = (dims[a] > 0 ? std::ldexp(double(base_frequency), o) * (std::min(edge[a], dims[a]) - 1) / dims[a] : 0.0) +
                   (worley ? 3.0 : 2.0);
        const double pairs = n[1] * n[2], cells = n[0] * pairs;
        if (pairs <= kMaxPairs && cells <= kMaxCells)
            c.tiles += (pairs + cells) * pair_hashes / 256.0;
        else
            c.tiles += pairs <= kMaxPairs ? pairs * pair_hashes / 256.0 + after_pairs : texel_hashes;
        c.texels += texel_hashes;
    }
}
// Whether a call's tiles save enough hashes for their barriers and 30 KiB of LDS.  us by tiles / by texels, and
// the share of the hashes that tiles leave: detail 128^3 at base frequency 1 277 / 990 (0.02), 8 550 / 991
// (0.28), 100 922 / 990 (0.74); 64^3 at 100 140 / 130 (0.96); in small textures, whose tiles wait at
// their barriers, 32^3 at 1 33.5 / 38.9 (0.25), 8 39.6 / 39.0 (0.54), 100 45.2 / 39.0 (0.97).  A Perlin octave alone has
// a ninth of the hashes to save: voxel grids of 512^3 at 4 3,348 / 4,691 (0.01), 64 4,283 / 4,690
// (0.22), of 128^3 at 64 92.3 / 76.9 (0.6), of 8^3 at 1 7.2 / 4.6.
bool tiles_pay(const NoiseCost& c, bool worley, long long texels) {
    const bool large = texels > 1 << 16;
    return c.tiles < c.texels * (worley ? (large ? 0.85 : 0.6) : large ? 0.3 : 0.0);
}
bool image_tiles_pay(const SkyhipNoiseCreateInfo& perlin, const SkyhipNoiseCreateInfo& worley, int size) {
    NoiseCost c;
    add_octaves(c, {kImageTile, kImageTile, 1}, {size, size, 0}, perlin.base_frequency, 8, false);
    add_octaves(c, {kImageTile, kImageTile, 1}, {size, size, 0}, worley.base_frequency, 8, true);
    return tiles_pay(c, true, (long long)size * size);
}
bool volume_tiles_pay(const SkyhipNoiseCreateInfo* perlin, const SkyhipNoiseCreateInfo& worley, int size) {
    NoiseCost c;
    if (perlin) add_octaves(c, {kVolumeTileXY, kVolumeTileXY, kVolumeTileZ}, {size, size, size}, perlin->base_frequency, 8, false);
    add_octaves(c, {kVolumeTileXY, kVolumeTileXY, kVolumeTileZ}, {size, size, size}, worley.base_frequency, 8, true);
    return tiles_pay(c, true, (long long)size * size * size);
}

int validate_noise(const SkyhipNoiseCreateInfo* ci) {
    if (ci == nullptr) return fail(SKYHIP_ERR_INVALID_ARGUMENT, "noise create info is NULL");
    if (ci->base_frequency == 0 || ci->base_frequency > (1u << 20))
        return fail(SKYHIP_ERR_INVALID_SIZE, "base_frequency %u outside [1, 2^20]", ci->base_frequency);
    if (!std::isfinite(ci->remap_min) || !std::isfinite(ci->remap_max))
        return fail(SKYHIP_ERR_NON_FINITE, "non-finite remap range");
    return SKYHIP_OK;
}

}  // namespace skyhip

using namespace skyhip;

extern "C" int skyhip_mip_levels(int32_t width, int32_t height, int32_t depth) {
    int m = width > height ? width : height;
    m = m > depth ? m : depth;
    if (m <= 0) return 0;
    int levels = 1;
    while ((m >> levels) > 0) ++levels;  // floor(log2(max)) + 1, ImageLoader.h:8-14
    return levels;
}

extern "C" size_t skyhip_mip_chain_bytes(int32_t width, int32_t height, int32_t depth, int32_t channels,
                                         int32_t levels) {
    size_t total = 0;
    for (int l = 0; l < levels; ++l) {
        size_t w = size_t(width >> l > 0 ? width >> l : 1), h = size_t(height >> l > 0 ? height >> l : 1),
               d = size_t(depth >> l > 0 ? depth >> l : 1);
        total += w * h * d * size_t(channels);
    }
    return total;
}

extern "C" int skyhip_noise_cloud_map(SkyhipContext* ctx, const SkyhipNoiseCreateInfo* density,
                                      const SkyhipNoiseCreateInfo* height, uint8_t* out_rg8, int32_t size) {
    SKYHIP_CHECK(check_ctx(ctx));
    SKYHIP_CHECK(validate_noise(density));
    SKYHIP_CHECK(validate_noise(height));
    if (out_rg8 == nullptr) return fail(SKYHIP_ERR_INVALID_ARGUMENT, "output is NULL");
    if (size < 1 || size > 16384) return fail(SKYHIP_ERR_INVALID_SIZE, "cloud map size %d outside [1, 16384]", size);
    if (image_tiles_pay(*density, *height, size))
        hipLaunchKernelGGL(cloud_map_kernel<true>, image_grid(size, 2), dim3(256), 0, ctx->stream,
                       *density, *height, out_rg8, size);
    else
        hipLaunchKernelGGL(cloud_map_kernel<false>, image_grid(size, 2), dim3(256), 0, ctx->stream,
                       *density, *height, out_rg8, size);
    SKYHIP_LAUNCH_CHECK("cloud_map_kernel");
    return SKYHIP_OK;
}

extern "C" int skyhip_noise_detail(SkyhipContext* ctx, const SkyhipNoiseCreateInfo* perlin,
                                   const SkyhipNoiseCreateInfo* worley, uint8_t* out_r8, int32_t size) {
    SKYHIP_CHECK(check_ctx(ctx));
    SKYHIP_CHECK(validate_noise(perlin));
    SKYHIP_CHECK(validate_noise(worley));
    if (out_r8 == nullptr) return fail(SKYHIP_ERR_INVALID_ARGUMENT, "output is NULL");
    if (size < 1 || size > 1024) return fail(SKYHIP_ERR_INVALID_SIZE, "detail size %d outside [1, 1024]", size);
    if (volume_tiles_pay(perlin, *worley, size))
        hipLaunchKernelGGL(detail_kernel<true>, volume_grid(size, size, size), dim3(256), 0, ctx->stream,
                       *perlin, *worley, out_r8, size);
    else
        hipLaunchKernelGGL(detail_kernel<false>, volume_grid(size, size, size), dim3(256), 0, ctx->stream,
                       *perlin, *worley, out_r8, size);
    SKYHIP_LAUNCH_CHECK("detail_kernel");
    return SKYHIP_OK;
}

extern "C" int skyhip_noise_displacement(SkyhipContext* ctx, const SkyhipNoiseCreateInfo* perlin, uint8_t* out_rgba8,
                                         int32_t size) {
    SKYHIP_CHECK(check_ctx(ctx));
    SKYHIP_CHECK(validate_noise(perlin));
    if (out_rgba8 == nullptr) return fail(SKYHIP_ERR_INVALID_ARGUMENT, "output is NULL");
    if (size < 1 || size > 16384) return fail(SKYHIP_ERR_INVALID_SIZE, "displacement size %d outside [1, 16384]", size);
    // Tiles by channel while they leave CUs idle: us by tiles / by texels 128^2 11.6 / 13.5, 160^2 15.4 / 13.6,
    // 2,048^2 654 / 487.
    if (image_grid(size, 4).x * image_grid(size, 4).y * 4u <= unsigned(std::max(ctx->cu_count, 1)))
        hipLaunchKernelGGL(displacement_kernel, image_grid(size, 4), dim3(256), 0, ctx->stream, *perlin, out_rgba8, size);
    else
        hipLaunchKernelGGL(displacement_texels_kernel, dim3(div_up((long long)size * size, 256)), dim3(256), 0,
                           ctx->stream, *perlin, out_rgba8, size);
    SKYHIP_LAUNCH_CHECK("displacement_kernel");
    return SKYHIP_OK;
}

extern "C" int skyhip_noise_worley(SkyhipContext* ctx, const SkyhipNoiseCreateInfo* worley, uint8_t* out_r8,
                                   int32_t size) {
    SKYHIP_CHECK(check_ctx(ctx));
    SKYHIP_CHECK(validate_noise(worley));
    if (out_r8 == nullptr) return fail(SKYHIP_ERR_INVALID_ARGUMENT, "output is NULL");
    if (size < 1 || size > 1024) return fail(SKYHIP_ERR_INVALID_SIZE, "Worley volume size %d outside [1, 1024]", size);
    if (volume_tiles_pay(nullptr, *worley, size))
        hipLaunchKernelGGL(worley_kernel<true>, volume_grid(size, size, size), dim3(256), 0, ctx->stream,
                       *worley, out_r8, size);
    else
        hipLaunchKernelGGL(worley_kernel<false>, volume_grid(size, size, size), dim3(256), 0, ctx->stream,
                       *worley, out_r8, size);
    SKYHIP_LAUNCH_CHECK("worley_kernel");
    return SKYHIP_OK;
}

// Cell-corner copies of a REPEAT texture's level 0 (size s a power of two, indices mod s):
// a 2D RG8 cell (x, y) packs texels (x, y), (x + 1, y) in .x and (x, y + 1), (x + 1, y + 1) in
// .y, two bytes each; a 3D R8 cell (x, y, z) packs the eight texels (x + a, y + b, z + c) as
// byte a + 2b + 4c.
__global__ __launch_bounds__(256) void cells_2d_rg8_kernel(const uint16_t* __restrict__ t, int ls,
                                                           uint2* __restrict__ out) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x, s = 1u << ls, m = s - 1u;
    if (i >= s * s) return;
    const uint32_t x = i & m, y = i >> ls, x1 = (x + 1u) & m, y1 = (y + 1u) & m;
    const uint32_t r0 = y << ls, r1 = y1 << ls;
    out[i] = make_uint2(uint32_t(t[r0 | x]) | (uint32_t(t[r0 | x1]) << 16), uint32_t(t[r1 | x]) | (uint32_t(t[r1 | x1]) << 16));
}

__global__ __launch_bounds__(256) void cells_3d_r8_kernel(const uint8_t* __restrict__ t, int ls,
                                                          uint2* __restrict__ out) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x, s = 1u << ls, m = s - 1u;
    if (i >= s * s * s) return;
    const uint32_t x = i & m, y = (i >> ls) & m, z = i >> (2 * ls);
    uint32_t w[2] = {0u, 0u};
    for (int k = 0; k < 8; ++k) {
        const uint32_t xx = (x + uint32_t(k & 1)) & m, yy = (y + uint32_t((k >> 1) & 1)) & m,
                       zz = (z + uint32_t(k >> 2)) & m;
        w[k >> 2] |= uint32_t(t[(zz << (2 * ls)) | (yy << ls) | xx]) << (8 * (k & 3));
    }
    out[i] = make_uint2(w[0], w[1]);
}

static int cells_args(SkyhipContext* ctx, const uint8_t* level0, int32_t size, uint8_t* out, int max_size,
                      int align_in, int& ls) {
    SKYHIP_CHECK(check_ctx(ctx));
    if (!level0 || !out) return fail(SKYHIP_ERR_INVALID_ARGUMENT, "NULL argument");
    if (size < 2 || size > max_size || (size & (size - 1)) != 0)
        return fail(SKYHIP_ERR_INVALID_SIZE, "texture size %d is not a power of two in [2, %d]", size, max_size);
    if (reinterpret_cast<uintptr_t>(out) % 8 != 0 || reinterpret_cast<uintptr_t>(level0) % align_in != 0)
        return fail(SKYHIP_ERR_INVALID_ARGUMENT, "misaligned texture or cell buffer");
    ls = 0;
    while ((1 << ls) < size) ++ls;
    return SKYHIP_OK;
}

extern "C" int skyhip_texture_cells_2d_rg8(SkyhipContext* ctx, const uint8_t* level0, int32_t size,
                                           uint8_t* out_cells) {
    int ls;
    SKYHIP_CHECK(cells_args(ctx, level0, size, out_cells, 16384, 2, ls));
    hipLaunchKernelGGL(cells_2d_rg8_kernel, dim3(div_up((long long)size * size, 256)), dim3(256), 0, ctx->stream,
                       reinterpret_cast<const uint16_t*>(level0), ls, reinterpret_cast<uint2*>(out_cells));
    SKYHIP_LAUNCH_CHECK("cells_2d_rg8_kernel");
    return SKYHIP_OK;
}

extern "C" int skyhip_texture_cells_3d_r8(SkyhipContext* ctx, const uint8_t* level0, int32_t size,
                                          uint8_t* out_cells) {
    int ls;
    SKYHIP_CHECK(cells_args(ctx, level0, size, out_cells, 1024, 1, ls));
    hipLaunchKernelGGL(cells_3d_r8_kernel, dim3(div_up((long long)size * size * size, 256)), dim3(256), 0,
                       ctx->stream, level0, ls, reinterpret_cast<uint2*>(out_cells));
    SKYHIP_LAUNCH_CHECK("cells_3d_r8_kernel");
    return SKYHIP_OK;
}

extern "C" int skyhip_generate_mipmaps(SkyhipContext* ctx, uint8_t* texture, int32_t dims, int32_t channels,
                                       int32_t width, int32_t height, int32_t depth, int32_t levels) {
    SKYHIP_CHECK(check_ctx(ctx));
    if (texture == nullptr) return fail(SKYHIP_ERR_INVALID_ARGUMENT, "texture is NULL");
    if ((dims != 2 && dims != 3) || channels < 1 || channels > 4)
        return fail(SKYHIP_ERR_INVALID_ARGUMENT, "dims must be 2 or 3 and channels 1..4");
    if (dims == 2) depth = 1;
    if (width < 1 || height < 1 || depth < 1 || levels < 1 || levels > skyhip_mip_levels(width, height, depth))
        return fail(SKYHIP_ERR_INVALID_SIZE, "bad texture size or level count");
    size_t off = 0;
    int sx = width, sy = height, sz = depth;
    for (int l = 1; l < levels;) {
        const int dx = std::max(sx / 2, 1), dy = std::max(sy / 2, 1), dz = std::max(sz / 2, 1);
        const int n = mip_tile_levels(dims, channels, dx, dy, dz, levels - l);
        auto launch = [&](auto d, auto c) {
            constexpr int kD = decltype(d)::value, kC = decltype(c)::value, kEdge = kD == 3 ? 8 : 16;
            uint8_t *src = texture + off, *dst = src + size_t(sx) * sy * sz * kC;
            if (n == 0)
                hipLaunchKernelGGL((downsample_level_kernel<kD, kC>), dim3(div_up((long long)dx * dy * dz * kC, 256)),
                                   dim3(256), 0, ctx->stream, src, sx, sy, sz, dst, dx, dy, dz);
            else
                hipLaunchKernelGGL((downsample_kernel<kD, kC>),
                                   dim3(div_up(dx, kEdge), div_up(dy, kEdge), kD == 3 ? div_up(dz, kEdge) : 1), dim3(256),
                                   0, ctx->stream, src, sx, sy, sz, dst, n);
        };
        auto channel = [&](auto d) {
            if (channels == 1) launch(d, std::integral_constant<int, 1>());
            else if (channels == 2) launch(d, std::integral_constant<int, 2>());
            else if (channels == 3) launch(d, std::integral_constant<int, 3>());
            else launch(d, std::integral_constant<int, 4>());
        };
        if (dims == 3) channel(std::integral_constant<int, 3>());
        else channel(std::integral_constant<int, 2>());
        SKYHIP_LAUNCH_CHECK("downsample_kernel");
        for (int k = 0; k < std::max(n, 1); ++k, ++l) {
            off += size_t(sx) * sy * sz * channels;
            sx = std::max(sx / 2, 1), sy = std::max(sy / 2, 1), sz = std::max(sz / 2, 1);
        }
    }
    return SKYHIP_OK;
}

extern "C" int skyhip_voxel_grid_generate(SkyhipContext* ctx, const SkyhipVoxelGridCreateInfo* info,
                                          uint16_t* out_grid, int32_t dim_x, int32_t dim_y, int32_t dim_z) {
    SKYHIP_CHECK(check_ctx(ctx));
    if (info == nullptr || out_grid == nullptr) return fail(SKYHIP_ERR_INVALID_ARGUMENT, "NULL argument");
    if (dim_x < 8 || dim_y < 8 || dim_z < 8 || dim_x > 1024 || dim_y > 1024 || dim_z > 1024)
        return fail(SKYHIP_ERR_INVALID_SIZE, "grid dims outside [8, 1024]");
    if (info->base_frequency < 1 || info->base_frequency > (1u << 16) || info->octaves < 1 || info->octaves > 12)
        return fail(SKYHIP_ERR_INVALID_SIZE, "base_frequency outside [1, 65536] or octaves outside [1, 12]");
    if (!finite_block(&info->fbm_inv_std, 9)) return fail(SKYHIP_ERR_NON_FINITE, "non-finite grid parameter");
    for (int k = 0; k < 3; ++k)
        if (!(info->ellipsoid_radii[k] > 0.0f)) return fail(SKYHIP_ERR_INVALID_ARGUMENT, "ellipsoid radii must be > 0");
    NoiseCost c;
    add_octaves(c, {kVolumeTileXY, kVolumeTileXY, kVolumeTileZ}, {dim_x, dim_y, dim_z}, info->base_frequency, info->octaves, false);
    if (tiles_pay(c, false, (long long)dim_x * dim_y * dim_z))
        hipLaunchKernelGGL(voxel_grid_kernel<true>, volume_grid(dim_x, dim_y, dim_z), dim3(256), 0, ctx->stream, *info, out_grid,
                       dim_x, dim_y, dim_z);
    else
        hipLaunchKernelGGL(voxel_grid_kernel<false>, volume_grid(dim_x, dim_y, dim_z), dim3(256), 0, ctx->stream, *info, out_grid,
                       dim_x, dim_y, dim_z);
    SKYHIP_LAUNCH_CHECK("voxel_grid_kernel");
    return SKYHIP_OK;
}
