// upf_material.hpp -- the per-texel / per-tile material stack of the reference
// (coloringDefault / coloringBarren / coloringDebug, sources/coloringModes.cpp:905-966)
// on gfx950: elevation, precipitation, temperature, slope from 8 elevation probes,
// biome, type, then the layers bedrock, cliffs, mica, dirt, sand, grass, boulders,
// water, flowers, ice and snow, and the final saturation.
//
// The noise objects the reference configures are evaluated in place with their
// configurations written at the call (constants fold into the code).  Object k is seeded
// seed + 16 k and its octaves add 0..7 (the reference draws every seed from noiseSeed(),
// sources/math.cpp:73-77; objects that share `seed` in the reference share an index
// here).  cage's noise kinds map as follows (cage is not in the reference's checkout; the
// definitions are this library's, documented at upf_material_spec):
//   Perlin -> lattice gradient noise; Value -> lattice value noise; Cubic -> value noise
//   with cubic interpolation over the 4^3 lattice values around the sample; Simplex and
//   SimplexReduced -> simplex noise; Cellular -> F1 / F2 over the 27 cells around the
//   sample with a distance (Euclidean, Manhattan, Hybrid) and an operation (Cell value,
//   Subtract, Multiply, Divide).
// Everything is plain FP32 (no fused operations) and pow / atan are the library's own
// (upf_math.hpp): the CPU restatement rounds alike.
#pragma once

#include "upf_device.hpp"
#include "upf_modes.hpp"

namespace upf {

struct DMaterial {
  DSpec field;
  int32_t coloring, purpose, poles, flowers;
  uint32_t seed;
  int32_t pad[3];
};

// Tile (sources/planets.h:63-83), the fields the material stack reads and writes.
struct MTile {
  float px, py, pz, nx, ny, nz;
  float r, g, b;
  float roughness, metallic, height, elevation, slope, temperature, precipitation, opacity;
  int biome, type;
};

enum { kDistManhattan = 1, kDistHybrid = 2 };
enum { kBiomeBare = 0, kBiomeTundra, kBiomeTaiga, kBiomeShrubland, kBiomeGrassland, kBiomeTemperateSeasonal,
       kBiomeTemperateRain, kBiomeDesert, kBiomeSavanna, kBiomeTropicalSeasonal, kBiomeTropicalRain, kBiomeWater };
enum { kTypeRoad = 0, kTypeFlat = 1, kTypeRough = 2, kTypeCliffs = 3, kTypeWater = 4 };

// ------------------------------------------------------------------ base noises
__device__ __forceinline__ float m_lerp(float a, float b, float t) { return a + t * (b - a); }
__device__ __forceinline__ float m_fade(float t) { return t * t * t * (t * (t * 6.0f - 15.0f) + 10.0f); }
__device__ __forceinline__ uint32_t m_hash(uint32_t seed, int32_t x, int32_t y, int32_t z) {
  return (seed ^ ((uint32_t)x * kPX) ^ ((uint32_t)y * kPY) ^ ((uint32_t)z * kPZ)) * kHM;
}
__device__ __forceinline__ float m_lattice(uint32_t h) { return (float)(int32_t)h * 4.656612873077393e-10f; }

typedef __attribute__((address_space(3))) float lds_float;
typedef float v4f __attribute__((ext_vector_type(4)));  // plain vector: loads from address space 3
typedef __attribute__((address_space(3))) v4f lds_v4;

// gdot with the 16 gradient vectors in LDS: their components are -1, 0 and 1, two of them
// not 0, so the products are exact and the sum rounds once, as gdot's +-u +- v does; one
// 16-byte read (16 entries over the 64 banks) in place of 9 of gdot's 14 instructions.
__device__ __forceinline__ float m_gdot(const lds_v4* gtab, uint32_t h, float x, float y, float z) {
  const v4f g = gtab[h >> 28];
  return fmaf(g.z, z, fmaf(g.y, y, g.x * x));
}
__device__ __forceinline__ v4f m_gtab_entry(int g) {
  v4f e;
  float gx, gy, gz;
  gvec((uint32_t)g << 28, gx, gy, gz);
  e.x = gx; e.y = gy; e.z = gz; e.w = 0.0f;
  return e;
}

// Noise octaves out of line: a texel evaluates ~45 of them, and inlined they would make
// a kernel of several instruction caches.
__device__ __noinline__ float m_perlin(const lds_v4* gtab, uint32_t seed, float x, float y, float z) {
  const float fx = floorf(x), fy = floorf(y), fz = floorf(z);
  const float tx = x - fx, ty = y - fy, tz = z - fz;
  const float sx = tx - 1.0f, sy = ty - 1.0f, sz = tz - 1.0f;
  const float ux = m_fade(tx), uy = m_fade(ty), uz = m_fade(tz);
  uint32_t h[8];
  cell_hashes(seed, (int)fx, (int)fy, (int)fz, h);
  const float n000 = m_gdot(gtab, h[0], tx, ty, tz), n100 = m_gdot(gtab, h[1], sx, ty, tz);
  const float n010 = m_gdot(gtab, h[2], tx, sy, tz), n110 = m_gdot(gtab, h[3], sx, sy, tz);
  const float n001 = m_gdot(gtab, h[4], tx, ty, sz), n101 = m_gdot(gtab, h[5], sx, ty, sz);
  const float n011 = m_gdot(gtab, h[6], tx, sy, sz), n111 = m_gdot(gtab, h[7], sx, sy, sz);
  const float y0 = m_lerp(m_lerp(n000, n100, ux), m_lerp(n010, n110, ux), uy);
  const float y1 = m_lerp(m_lerp(n001, n101, ux), m_lerp(n011, n111, ux), uy);
  return m_lerp(y0, y1, uz);
}

__device__ __noinline__ float m_value(uint32_t seed, float x, float y, float z) {
  return noise_value<true>(seed, x, y, z);
}

// noise_simplex with the gradients in LDS; a corner out of reach adds 0
__device__ __noinline__ float m_simplex(const lds_v4* gtab, uint32_t seed, float x, float y, float z) {
  SimplexCell c;
  simplex_cell(x, y, z, c);
  float n = 0.0f;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const float dx = c.d[q][0], dy = c.d[q][1], dz = c.d[q][2];
    const float t = 0.5f - (dx * dx + dy * dy + dz * dz);
    const float t2 = t * t;
    const float v = n + t2 * t2 * m_gdot(gtab, simplex_hash(seed, c, q), dx, dy, dz);
    n = t > 0.0f ? v : n;
  }
  return 72.0f * n;
}

// ------------------------------------------------------------------ lattices shared by a wave
// The cubic and cellular noises and the Voronoi read 64 lattice values, 27 feature points
// or 27 cells of impact points around a sample: nearly all of a tile's arithmetic when
// every lane makes its own.  The lanes of a wave sit on neighbouring texels (8 x 8), so
// their neighbourhoods are few or overlap, and the 64 lanes make them together in the
// wave's LDS:
//   slots   one per different neighbourhood (m_share), filled by the whole wave, the lanes
//           of a neighbourhood reading the same addresses;
//   box     every lattice point that some lane reads, when the wave's bounding box (m_box)
//           holds more than kBoxCells neighbourhoods and its points fit the LDS;
//   lane    each lane makes its own (scattered points: a wave whose first two
//           neighbourhoods serve under kShareMin lanes, or that fits neither).
// The values, and so the results, are the same bit for bit.  Called by all 64 lanes; `need`
// marks the lanes whose result is used.  2048^2 lakes textures, VALU instructions per wave
// and time of the whole call: per lane 23,150, 1.89 ms; slots alone 10,200, 0.976 ms (the
// finest octaves' attempts failed); with the boxes 10,130, 0.969 ms; with the rows'
// polynomials in the slots and the gradients in LDS 9,360, 0.924 ms.  kBoxCells: a slot
// costs ~30 instructions a neighbourhood and ~180 to read, a box ~110 and ~290.
constexpr int kWaveLds = 1024;  // floats of LDS per wave
constexpr int kShareMin = 12;
constexpr int kBoxCells = 4;

__device__ __forceinline__ int m_lane() { return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

__device__ __forceinline__ void m_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Gives every needed lane's neighbourhood (ix, iy, iz) a slot, make(slot, x, y, z) filling
// it (called by all lanes with uniform arguments); -1 when the wave shares too little.
template <int kCells, class Make>
__device__ __forceinline__ int m_share(int ix, int iy, int iz, bool need, Make make) {
  uint64_t todo = __ballot(need);
  int slot = 0;
  m_wave_sync();  // earlier readers of the slots are done
  for (int s = 0; todo; s++) {
    if (s == kCells) return -1;
    const int lead = __builtin_ctzll(todo);
    const int x = __builtin_amdgcn_readlane(ix, lead), y = __builtin_amdgcn_readlane(iy, lead),
              z = __builtin_amdgcn_readlane(iz, lead);
    const bool same = ix == x && iy == y && iz == z;
    const uint64_t mask = __ballot(same);
    if (same) slot = s;
    todo &= ~mask;
    if (s == 1 && __popcll(__ballot(need) & ~todo) < kShareMin && todo) return -1;
    make(s, x, y, z);
  }
  m_wave_sync();
  return slot;
}

// The lattice cells floor(p f) .. of a wave: the smallest and the extent per axis, from the
// bounding box of its positions (products and roundings are monotone, so every lane's cell
// lies inside).  points(margin) is the number of lattice points with `margin` more per axis.
struct MBounds {
  float lo[3], hi[3];  // wave-uniform; hi < lo when no lane holds a tile
};
struct MBox {
  int x, y, z, nx, ny, nz;
  float cells;
};
template <bool ROUND>
__device__ __forceinline__ MBox m_box(const MBounds& b, float f) {
  float l[3], e[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    l[a] = ROUND ? rintf(b.lo[a] * f) : floorf(b.lo[a] * f);
    e[a] = (ROUND ? rintf(b.hi[a] * f) : floorf(b.hi[a] * f)) - l[a] + 1.0f;
  }
  MBox r;
  r.x = (int)l[0]; r.y = (int)l[1]; r.z = (int)l[2];
  r.cells = e[0] * e[1] * e[2];  // NaN and infinities compare false against any limit below
  r.nx = (int)e[0]; r.ny = (int)e[1]; r.nz = (int)e[2];
  return r;
}
// a / b for 0 <= a < 1024, 1 <= b <= 1024, rb = 1 / b: (a + 1/2) / b lies at least 1 / (2 b)
// from an integer, the roundings move it by under a 2^-23
__device__ __forceinline__ int m_small_div(int a, float rb) { return (int)(((float)a + 0.5f) * rb); }
// Calls make(e, i, j, k) for the points e = i + nx (j + ny k) of an nx x ny x nz box, one
// per lane.
template <class Make>
__device__ __forceinline__ void m_fill_box(int nx, int ny, int nz, Make make) {
  const float rx = 1.0f / (float)nx, ry = 1.0f / (float)ny;
  const int n = nx * ny * nz;
  m_wave_sync();  // earlier readers are done
  for (int e = m_lane(); e < n; e += 64) {
    const int q = m_small_div(e, rx), k = m_small_div(q, ry);
    make(e, e - q * nx, q - k * ny, k);
  }
  m_wave_sync();
}
__device__ __forceinline__ int m_clamp(int v, int hi) { return min(max(v, 0), hi); }

// cubic through b (t = 0) and c (t = 1) with neighbours a, d: t^3 p + t^2 ((a - b) - p)
// + t (c - a) + b, p = (d - c) - (a - b)
__device__ __forceinline__ float m_cubic(float a, float b, float c, float d, float t) {
  const float p = (d - c) - (a - b);
  return t * t * t * p + t * t * ((a - b) - p) + t * (c - a) + b;
}

// lane i of each quad of lanes: CTRL = i * 0x55
template <int CTRL>
__device__ __forceinline__ float m_quad(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}

// Value noise with cubic interpolation over the 4^3 lattice values, at p f; b bounds the
// wave's p.
__device__ __noinline__ float m_value_cubic(lds_float* lds, const MBounds b, uint32_t seed, float f, float px, float py,
                                            float pz, bool need) {
  constexpr int kStride = 68;  // 64 values; neighbourhoods 4 banks apart
  const float x = px * f, y = py * f, z = pz * f;
  const float fx = floorf(x), fy = floorf(y), fz = floorf(z);
  const int ix = (int)fx, iy = (int)fy, iz = (int)fz;
  const float tx = x - fx, ty = y - fy, tz = z - fz;
  const MBox box = m_box<false>(b, f);
  const int nx = box.nx + 3, ny = box.ny + 3, nz = box.nz + 3;
  float zs[4];
  if (box.cells > (float)kBoxCells && box.cells < (float)kWaveLds && nx * ny * nz <= kWaveLds) {
    m_fill_box(nx, ny, nz, [&](int e, int i, int j, int k) {
      lds[e] = m_lattice(m_hash(seed, box.x + i - 1, box.y + j - 1, box.z + k - 1));
    });
    const int o = m_clamp(ix - box.x, box.nx - 1) + nx * (m_clamp(iy - box.y, box.ny - 1) + ny * m_clamp(iz - box.z, box.nz - 1));
#pragma unroll
    for (int k = 0; k < 4; k++) {
      float ys[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const lds_float* q = lds + o + nx * (j + ny * k);
        ys[j] = m_cubic(q[0], q[1], q[2], q[3], tx);
      }
      zs[k] = m_cubic(ys[0], ys[1], ys[2], ys[3], ty);
    }
    return m_cubic(zs[0], zs[1], zs[2], zs[3], tz) * (1.0f / 3.375f);
  }
  const int lane = m_lane();
  // a slot holds its 16 rows' polynomials (p, (a - b) - p, c - a, b) in tx, which are the
  // same for all its lanes: lane 4 row + i has lattice value i of the row, and takes the
  // others of its quad
  const int slot = m_share<kWaveLds / kStride>(ix, iy, iz, need, [&](int s, int cx, int cy, int cz) {
    const float v = m_lattice(m_hash(seed, cx + (lane & 3) - 1, cy + ((lane >> 2) & 3) - 1, cz + (lane >> 4) - 1));
    const float va = m_quad<0x00>(v), vb = m_quad<0x55>(v), vc = m_quad<0xAA>(v), vd = m_quad<0xFF>(v);
    const float p = (vd - vc) - (va - vb);
    const int i = lane & 3;
    lds[s * kStride + lane] = i == 0 ? p : (i == 1 ? (va - vb) - p : (i == 2 ? vc - va : vb));
  });
  if (slot >= 0) {
    const lds_v4* q = (const lds_v4*)(lds + slot * kStride);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      float ys[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const v4f v = q[4 * k + j];
        ys[j] = tx * tx * tx * v.x + tx * tx * v.y + tx * v.z + v.w;  // m_cubic of the row
      }
      zs[k] = m_cubic(ys[0], ys[1], ys[2], ys[3], ty);
    }
  } else {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      float ys[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        float xs[4];
#pragma unroll
        for (int i = 0; i < 4; i++) xs[i] = m_lattice(m_hash(seed, ix + i - 1, iy + j - 1, iz + k - 1));
        ys[j] = m_cubic(xs[0], xs[1], xs[2], xs[3], tx);
      }
      zs[k] = m_cubic(ys[0], ys[1], ys[2], ys[3], ty);
    }
  }
  return m_cubic(zs[0], zs[1], zs[2], zs[3], tz) * (1.0f / 3.375f);
}

// Cellular over the 27 cells around rint(q), one point per cell at k - 0.5 + r (r from
// three 10-bit fields of h ^ (h >> 15), scaled by 1/1023): F1 d0, F2 d1 and the hash of
// the nearest cell; the operations read from them.
struct MCell {
  float d0, d1;
  uint32_t best;
};
__device__ __forceinline__ v4f m_cell_point(uint32_t seed, int kx, int ky, int kz) {
  const uint32_t h = m_hash(seed, kx, ky, kz);
  const uint32_t m = h ^ (h >> 15);
  v4f p;
  p.x = ((float)kx - 0.5f) + (float)(m & 1023u) * (1.0f / 1023.0f);
  p.y = ((float)ky - 0.5f) + (float)((m >> 10) & 1023u) * (1.0f / 1023.0f);
  p.z = ((float)kz - 0.5f) + (float)((m >> 20) & 1023u) * (1.0f / 1023.0f);
  p.w = __uint_as_float(h);
  return p;
}
// At p f; b bounds the wave's p, or is empty (hi < lo) where that is not known.
template <int DIST>
__device__ __noinline__ MCell m_cellular(lds_float* lds, const MBounds b, uint32_t seed, float f, float px, float py,
                                         float pz, bool need) {
  constexpr int kStride = 28;  // float4: 27 points; neighbourhoods 16 banks apart
  const float x = px * f, y = py * f, z = pz * f;
  const int cx = (int)rintf(x), cy = (int)rintf(y), cz = (int)rintf(z);
  MCell r = {__builtin_inff(), __builtin_inff(), 0u};
  const auto add = [&](const v4f p) {
    const float ex = p.x - x, ey = p.y - y, ez = p.z - z;
    float d;
    const float l1 = fabsf(ex) + fabsf(ey) + fabsf(ez);
    d = DIST == kDistHybrid ? l1 + (ex * ex + ey * ey + ez * ez) : l1;
    if (d < r.d0) { r.d1 = r.d0; r.d0 = d; r.best = __float_as_uint(p.w); }
    else if (d < r.d1) r.d1 = d;
  };
  lds_v4* const pts = (lds_v4*)lds;
  const MBox box = m_box<true>(b, f);
  const int nx = box.nx + 2, ny = box.ny + 2, nz = box.nz + 2;
  if (b.lo[0] <= b.hi[0] && box.cells > (float)kBoxCells && box.cells < (float)kWaveLds && nx * ny * nz <= kWaveLds / 4) {
    m_fill_box(nx, ny, nz, [&](int e, int i, int j, int k) { pts[e] = m_cell_point(seed, box.x + i - 1, box.y + j - 1, box.z + k - 1); });
    const int o = m_clamp(cx - box.x, box.nx - 1) + nx * (m_clamp(cy - box.y, box.ny - 1) + ny * m_clamp(cz - box.z, box.nz - 1));
    for (int k = 0; k < 3; k++)
#pragma unroll
      for (int j = 0; j < 3; j++)
#pragma unroll
        for (int i = 0; i < 3; i++) add(pts[o + i + nx * (j + ny * k)]);
    return r;
  }
  const int lane = m_lane();
  const int slot = m_share<kWaveLds / (4 * kStride)>(cx, cy, cz, need, [&](int s, int ux, int uy, int uz) {
    if (lane < 27)
      pts[s * kStride + lane] = m_cell_point(seed, ux + lane % 3 - 1, uy + lane / 3 % 3 - 1, uz + lane / 9 - 1);
  });
  if (slot >= 0) {
    const lds_v4* q = pts + slot * kStride;
#pragma unroll 9
    for (int i = 0; i < 27; i++) add(q[i]);
  } else {
    for (int dz = -1; dz <= 1; dz++)
      for (int dy = -1; dy <= 1; dy++)
#pragma unroll
        for (int dx = -1; dx <= 1; dx++) add(m_cell_point(seed, cx + dx, cy + dy, cz + dz));
  }
  return r;
}
__device__ __forceinline__ float m_ret_cell(const MCell& c) { return m_lattice(c.best); }
__device__ __forceinline__ float m_ret_sub(const MCell& c) { return c.d1 - c.d0 - 1.0f; }
__device__ __forceinline__ float m_ret_mul(const MCell& c) { return c.d1 * c.d0 * 0.5f - 1.0f; }
__device__ __forceinline__ float m_ret_div(const MCell& c) { return c.d0 / c.d1 - 1.0f; }

// A noise object's fractal sum: octaves at freq lac^k with amplitudes bounded by
// 1 / sum |gain|^k, octave k seeded seed + k; RIDGED sums 1 - 2 |n|.  The octave counts,
// frequencies and gains are constants at every call and fold.
template <bool RIDGED, int OCT, class F>
__device__ __forceinline__ float m_fractal(float freq, float lac, float gain, F octave) {
  const float ag = fabsf(gain);
  float s = 1.0f, a = ag;
#pragma unroll
  for (int i = 1; i < OCT; i++) { s = s + a; a = a * ag; }
  float sum = 0.0f, amp = 1.0f / s, f = freq;
#pragma unroll
  for (int k = 0; k < OCT; k++) {
    const float n = octave((uint32_t)k, f);
    if (RIDGED) sum = sum + (1.0f - 2.0f * fabsf(n)) * amp;
    else sum = sum + n * amp;
    amp = amp * gain;
    f = f * lac;
  }
  return sum;
}

// ------------------------------------------------------------------ helpers
__device__ __forceinline__ float m_sat(float x) { return fminf(fmaxf(x, 0.0f), 1.0f); }
__device__ __forceinline__ float m_smoothstep(float x) { return x * x * (3.0f - 2.0f * x); }
__device__ __forceinline__ float m_smootherstep(float x) { return x * x * x * (x * (x * 6.0f - 15.0f) + 10.0f); }
__device__ __forceinline__ float m_rescale(float v, float ia, float ib, float oa, float ob) {
  return (v - ia) / (ib - ia) * (ob - oa) + oa;
}
__device__ __forceinline__ float m_sharp_edge(float v, float p = 0.05f) {  // sources/math.cpp:13-16
  return m_rescale(fminf(fmaxf(v, 0.5f - p), 0.5f + p), 0.5f - p, 0.5f + p, 0.0f, 1.0f);
}
__device__ __forceinline__ float m_range_mask(float v, float zero_at, float one_at) {  // :29-32
  return m_sat((v - zero_at) / (one_at - zero_at));
}
constexpr float kRadToDeg = 57.29577951308232f;
constexpr float kPi = 3.14159265358979f;
// slope in radians, thresholds in degrees (:22-27)
__device__ __forceinline__ float m_steepness(float slope_rad, float threshold, float smoothing) {
  return m_sat((threshold + smoothing - slope_rad * kRadToDeg) / (2.0f * smoothing));
}

// fmodf(v, 1): the subtraction is exact, so the quotient loop of fmodf is not needed
__device__ __forceinline__ float m_mod1(float v) { return v - truncf(v); }

// RGB <-> HSV (h, s, v in [0, 1]), the textbook hexcone model.
__device__ __forceinline__ void m_rgb_to_hsv(float r, float g, float b, float& h, float& s, float& v) {
  const float mx = fmaxf(r, fmaxf(g, b)), mn = fminf(r, fminf(g, b));
  const float d = mx - mn;
  v = mx;
  s = mx > 0.0f ? d / mx : 0.0f;
  if (d <= 0.0f) { h = 0.0f; return; }
  float hh;
  if (mx == r) hh = (g - b) / d + (g < b ? 6.0f : 0.0f);
  else if (mx == g) hh = (b - r) / d + 2.0f;
  else hh = (r - g) / d + 4.0f;
  h = hh / 6.0f;
}
__device__ __forceinline__ void m_hsv_to_rgb(float h, float s, float v, float& r, float& g, float& b) {
  const float h6 = (h - floorf(h)) * 6.0f;
  const int i = min((int)h6, 5);
  const float f = h6 - (float)i;
  const float p = v * (1.0f - s), q = v * (1.0f - s * f), t = v * (1.0f - s * (1.0f - f));
  switch (i) {
    case 0: r = v; g = t; b = p; break;
    case 1: r = q; g = v; b = p; break;
    case 2: r = p; g = v; b = t; break;
    case 3: r = p; g = q; b = v; break;
    case 4: r = t; g = p; b = v; break;
    default: r = v; g = p; b = q; break;
  }
}
// colorHueShift, sources/math.cpp:47-52
__device__ __forceinline__ void m_hue_shift(float& r, float& g, float& b, float shift) {
  float h, s, v;
  m_rgb_to_hsv(r, g, b, h, s, v);
  h = m_mod1(h + shift + 1.0f);
  m_hsv_to_rgb(h, s, v, r, g, b);
}
// interpolateColor: HSV with the hue along the shorter arc
__device__ __forceinline__ void m_mix_color(float ar, float ag, float ab, float br, float bg, float bb, float t,
                                            float& r, float& g, float& b) {
  float h0, s0, v0, h1, s1, v1;
  m_rgb_to_hsv(ar, ag, ab, h0, s0, v0);
  m_rgb_to_hsv(br, bg, bb, h1, s1, v1);
  float dh = h1 - h0;
  if (dh > 0.5f) dh = dh - 1.0f;
  else if (dh < -0.5f) dh = dh + 1.0f;
  const float h = m_mod1(h0 + t * dh + 1.0f);
  m_hsv_to_rgb(h, m_lerp(s0, s1, t), m_lerp(v0, v1, t), r, g, b);
}
// colorDeviation (sources/math.cpp:40-45) without the global RNG: the deviation vector
// (three 10-bit fractions minus 0.5) is hashed from the position's float bits, and the
// colour moves in HSV.
__device__ __forceinline__ void m_deviation(float& r, float& g, float& b, float dev, uint32_t seed, float px,
                                            float py, float pz) {
  const uint32_t hsh = fmix32(m_hash(seed, (int32_t)__float_as_uint(px), (int32_t)__float_as_uint(py),
                                     (int32_t)__float_as_uint(pz)));
  const float u0 = (float)(hsh & 1023u) * (1.0f / 1023.0f) - 0.5f;
  const float u1 = (float)((hsh >> 10) & 1023u) * (1.0f / 1023.0f) - 0.5f;
  const float u2 = (float)((hsh >> 20) & 1023u) * (1.0f / 1023.0f) - 0.5f;
  float h, s, v;
  m_rgb_to_hsv(r, g, b, h, s, v);
  h = m_mod1(h + u0 * dev + 1.0f);
  s = m_sat(s + u1 * dev);
  v = m_sat(v + u2 * dev);
  m_hsv_to_rgb(h, s, v, r, g, b);
}

// Voronoi nearest with the points projected into the plane through p with normal n
// (sources/voronoi.cpp:58-66; closestPoint(plane, q) = q - dot(q - p, n) n).  PPC points
// per cell, the chain of states of upf_modes.hpp; called by all lanes.
template <int PPC>
__device__ __forceinline__ void m_voronoi_cell(uint32_t h0, uint32_t h1, uint32_t h2, int kx, int ky, int kz, float cell,
                                               v4f q[PPC]) {
  uint32_t s0 = (uint32_t)kx, s1 = (uint32_t)ky, s2 = (uint32_t)kz;
#pragma unroll
  for (int i = 0; i <= PPC; i++) {
    const uint32_t t0 = h0 + s0 + s1 + fmix32(s0);
    const uint32_t t1 = h1 + s1 + s2 + fmix32(s1);
    const uint32_t t2 = h2 + s2 + s0 + fmix32(s2);
    s0 = t0; s1 = t1; s2 = t2;
    if (i == 0) continue;
    q[i - 1].x = ((float)((int32_t)s0 % 65536) / 65535.0f + (float)kx) * cell;
    q[i - 1].y = ((float)((int32_t)s1 % 65536) / 65535.0f + (float)ky) * cell;
    q[i - 1].z = ((float)((int32_t)s2 % 65536) / 65535.0f + (float)kz) * cell;
    q[i - 1].w = 0.0f;
  }
}
template <int PPC>
__device__ __noinline__ v4f m_voronoi_plane(lds_float* lds, uint32_t seed, float cell, float px, float py, float pz,
                                            float nx, float ny, float nz, bool need) {
  constexpr int kStride = 27 * PPC + 1;  // float4
  constexpr int kCells = kWaveLds / (4 * kStride);
  const uint32_t h0 = fmix32(seed), h1 = fmix32(h0), h2 = fmix32(h1);
  const float freq = 1.0f / cell;
  const int32_t cx = cell_index(px * freq), cy = cell_index(py * freq), cz = cell_index(pz * freq);
  const int lane = m_lane();
  const int slot = m_share<kCells>(cx, cy, cz, need, [&](int s, int ux, int uy, int uz) {
    if (lane < 27) {
      v4f q[PPC];
      m_voronoi_cell<PPC>(h0, h1, h2, ux + lane % 3 - 1, uy + lane / 3 % 3 - 1, uz + lane / 9 - 1, cell, q);
#pragma unroll
      for (int i = 0; i < PPC; i++) ((lds_v4*)lds)[s * kStride + lane * PPC + i] = q[i];
    }
  });
  v4f c = {0.0f, 0.0f, 0.0f, 0.0f};
  float best = __builtin_inff();
  const auto add = [&](const v4f q) {
    const float dd = (q.x - px) * nx + (q.y - py) * ny + (q.z - pz) * nz;
    const float qx = q.x - dd * nx, qy = q.y - dd * ny, qz = q.z - dd * nz;
    const float ex = qx - px, ey = qy - py, ez = qz - pz;
    const float d2 = ex * ex + ey * ey + ez * ez;
    if (d2 < best) { best = d2; c.x = qx; c.y = qy; c.z = qz; }
  };
  if (slot >= 0) {
    const lds_v4* q = (const lds_v4*)lds + slot * kStride;
#pragma unroll 3
    for (int i = 0; i < 27 * PPC; i++) add(q[i]);
  } else {
    for (int dz = -1; dz <= 1; dz++)
      for (int dy = -1; dy <= 1; dy++)
        for (int dx = -1; dx <= 1; dx++) {
          v4f q[PPC];
          m_voronoi_cell<PPC>(h0, h1, h2, cx + dx, cy + dy, cz + dz, cell, q);
#pragma unroll
          for (int i = 0; i < PPC; i++) add(q[i]);
        }
  }
  return c;
}

__device__ __forceinline__ float m_dist(float ax, float ay, float az, float bx, float by, float bz) {
  const float dx = ax - bx, dy = ay - by, dz = az - bz;
  return sqrtf(dx * dx + dy * dy + dz * dz);
}
__device__ __forceinline__ void m_blend(MTile& t, float r, float g, float b, float rough, float metal, float height,
                                        float bf) {
  t.r = m_lerp(t.r, r, bf); t.g = m_lerp(t.g, g, bf); t.b = m_lerp(t.b, b, bf);
  t.roughness = m_lerp(t.roughness, rough, bf);
  t.metallic = m_lerp(t.metallic, metal, bf);
  t.height = m_lerp(t.height, height, bf);
}

// out of line: ~100 instructions each, used by most steps
__device__ __noinline__ float m_pow(float x, float e) { return upf_math::powf_(x, e); }
__device__ __noinline__ float m_atan(float x) { return upf_math::atanf_(x); }

// ------------------------------------------------------------------ the stack
// Every step runs with the whole wave: a step that some lane needs is run by all of them
// (it would run for the wave either way), the lanes that do not need it leave their tile
// as it is.  `on` marks the lanes that hold a tile.
struct MCtx {
  const lds_v4* gtab;  // the 16 gradient vectors
  lds_float* lds;  // the wave's kWaveLds floats
  bool on;
  MBounds bounds;  // of the positions of the lanes that are on
};
// the context of a wave whose lanes sit at (x, y, z)
__device__ __forceinline__ MCtx m_ctx(const lds_v4* gtab, lds_float* lds, bool on, float x, float y, float z) {
  MCtx c;
  c.gtab = gtab;
  c.lds = lds;
  c.on = on;
  const float p[3] = {x, y, z};
#pragma unroll
  for (int a = 0; a < 3; a++) {
    float lo = on ? p[a] : __builtin_inff(), hi = on ? p[a] : -__builtin_inff();
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
      lo = fminf(lo, __shfl_xor(lo, d));
      hi = fmaxf(hi, __shfl_xor(hi, d));
    }
    c.bounds.lo[a] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__float_as_int(lo)));
    c.bounds.hi[a] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__float_as_int(hi)));
  }
  return c;
}
// one octave, fBm and ridged sums of the lattice noises
__device__ __forceinline__ float m_perlin1(const MCtx& c, uint32_t seed, float f, float x, float y, float z) { return m_perlin(c.gtab, seed, x * f, y * f, z * f); }
__device__ __forceinline__ float m_value1(uint32_t seed, float f, float x, float y, float z) { return m_value(seed, x * f, y * f, z * f); }
template <int OCT> __device__ __forceinline__ float m_perlin_fbm(const MCtx& c, uint32_t seed, float freq, float lac, float gain, float x, float y, float z) {
  return m_fractal<false, OCT>(freq, lac, gain, [&](uint32_t k, float f) { return m_perlin1(c, seed + k, f, x, y, z); });
}
template <int OCT> __device__ __forceinline__ float m_value_fbm(uint32_t seed, float freq, float lac, float gain, float x, float y, float z) {
  return m_fractal<false, OCT>(freq, lac, gain, [&](uint32_t k, float f) { return m_value1(seed + k, f, x, y, z); });
}
template <bool RIDGED, int OCT> __device__ __forceinline__ float m_simplex_sum(const MCtx& c, uint32_t seed, float freq, float lac, float gain, float x, float y, float z) {
  return m_fractal<RIDGED, OCT>(freq, lac, gain, [&](uint32_t k, float f) { return m_simplex(c.gtab, seed + k, x * f, y * f, z * f); });
}
// the shared noises at the tile's position, and at warped positions (no bounds); all lanes
template <int OCT> __device__ __forceinline__ float m_cubic_fbm(const MCtx& c, uint32_t seed, float freq, const MTile& t, bool need) {
  return m_fractal<false, OCT>(freq, 2.0f, 0.5f, [&](uint32_t k, float f) {
    return m_value_cubic(c.lds, c.bounds, seed + k, f, t.px, t.py, t.pz, need);
  });
}
__device__ __forceinline__ float m_cubic1(const MCtx& c, uint32_t seed, float f, const MTile& t, bool need) {
  return m_value_cubic(c.lds, c.bounds, seed, f, t.px, t.py, t.pz, need);
}
template <int DIST> __device__ __forceinline__ MCell m_cell(const MCtx& c, uint32_t seed, float f, const MTile& t, bool need) {
  return m_cellular<DIST>(c.lds, c.bounds, seed, f, t.px, t.py, t.pz, need);
}
template <int DIST> __device__ __forceinline__ MCell m_cell_at(const MCtx& c, uint32_t seed, float f, float x, float y, float z, bool need) {
  const MBounds none = {{1.0f, 1.0f, 1.0f}, {0.0f, 0.0f, 0.0f}};
  return m_cellular<DIST>(c.lds, none, seed, f, x, y, z, need);
}
__device__ __forceinline__ bool m_any(bool v) { return __ballot(v) != 0; }
// seed of noise object k: octaves use seed + 16 k + octave, so objects never share seeds
__device__ __forceinline__ uint32_t ms(const DMaterial& m, uint32_t k) { return m.seed + 16u * k; }

// The base shape with separately rounded operations (the field kernels fuse them): the
// slope below differences eight probes 0.5 m apart at ~10^3 m from the origin, where the
// probes differ by little more than rounding, so the CPU restatement rounds alike.
// PRIM: the shape is a primitive (none, sphere, box, torus, capsule).  The other shapes'
// code, inlined at the nine evaluations, is most of a kernel that holds it (34,000
// instructions, 97 VGPRs), so the host picks the instantiation.
template <bool PRIM>
__device__ __forceinline__ float m_shape(const DSpec& s, float x, float y, float z) {
  const float* a = s.sp;
  switch (s.shape) {
    case UPF_SHAPE_SPHERE: return sqrtf(x * x + y * y + z * z) - a[0];
    case UPF_SHAPE_BOX: {
      const float qx = fabsf(x) - a[0], qy = fabsf(y) - a[1], qz = fabsf(z) - a[2];
      const float mx = fmaxf(qx, 0.0f), my = fmaxf(qy, 0.0f), mz = fmaxf(qz, 0.0f);
      return sqrtf(mx * mx + my * my + mz * mz) + fminf(fmaxf(qx, fmaxf(qy, qz)), 0.0f) - a[3];
    }
    case UPF_SHAPE_TORUS: {
      const float ring = sqrtf(x * x + z * z) - a[0];
      return sqrtf(ring * ring + y * y) - a[1];
    }
    case UPF_SHAPE_CAPSULE: {
      const float h2 = a[0] * 0.5f;
      const float zc = z - fminf(fmaxf(z, -h2), h2);
      return sqrtf(x * x + y * y + zc * zc) - a[1];
    }
    case UPF_SHAPE_NONE: return 0.0f;
    default:
      if (PRIM) return 0.0f;  // not reached
      if (s.shape >= UPF_SHAPE_H3O) return shape_more(s.shape, s.sp[0], s.sp[1], s.sp[2], s.sp[3], s.w, x, y, z);
      return shape_ext<float>(s.shape, s.sp, x, y, z, 0.0f);
  }
}

// terrainSdfElevation = shape * 10 (sources/modesConfiguration.cpp:230-237), with this
// spec's ratio 1 / elevation_scale
template <bool PRIM>
__device__ __forceinline__ float m_elev_sdf(const DMaterial& m, float x, float y, float z) {
  return m_shape<PRIM>(m.field, x, y, z) / m.field.escale;
}

__device__ __forceinline__ float m_beach(const DMaterial& m, const MTile& t) {  // :34-49
  if (t.biome == kBiomeWater) return 0.0f;
  const float n = m_value1(ms(m, 0), 0.035f, t.elevation, 0.0f, 0.0f);
  return m_range_mask(t.elevation + n * 20.0f, 10.0f, 15.0f);
}

__device__ __forceinline__ void m_precipitation(const MCtx& c, const DMaterial& m, MTile& t) {  // :59-80
  float p = m_cubic_fbm<2>(c, ms(m, 1), 0.001f, t, c.on) * 0.5f + 0.5f;
  p = m_sat(p);
  p = m_smootherstep(p);
  p = m_smootherstep(p);
  p = m_pow(fmaxf(p + 0.2f, 0.0f), 3.0f) * 0.6f;
  p = p * 400.0f;
  p = p + fmaxf(120.0f - fabsf(t.elevation), 0.0f) * 0.2f;
  t.precipitation = fmaxf(p, 0.0f);
}

__device__ __forceinline__ void m_temperature(const MCtx& c, const DMaterial& m, MTile& t) {  // :82-120
  float v = m_simplex_sum<false, 2>(c, ms(m, 2), 0.0003f, 2.0f, 0.4f, t.px, t.py, t.pz) * 0.5f + 0.5f;
  v = m_sat(v);
  v = m_smoothstep(v);
  v = v * 2.0f - 1.0f;
  if (m.poles) {
    float polar = fabsf(m_atan(t.py / sqrtf(t.px * t.px + t.pz * t.pz))) / kPi * 2.0f;
    polar = m_pow(polar, 1.7f);
    polar = polar + m_value_fbm<3>(ms(m, 3), 0.007f, 2.0f, 0.5f, t.px, t.py, t.pz) * 0.1f;
    v = v + (0.6f - polar * 3.2f);
  }
  t.temperature = 15.0f + v * 30.0f - fmaxf(t.elevation, 0.0f) * 0.02f;
}

template <bool PRIM>
__device__ __forceinline__ void m_slope(const DMaterial& m, MTile& t) {  // :122-151
  // anyPerpendicular (sources/math.cpp:65-72)
  float bx = 1.0f, by = 0.0f, bz = 0.0f;
  if (fabsf(t.nx) > 0.9f) { bx = 0.0f; by = 1.0f; }
  float ax = t.ny * bz - t.nz * by, ay = t.nz * bx - t.nx * bz, az = t.nx * by - t.ny * bx;
  const float al = sqrtf(ax * ax + ay * ay + az * az);
  ax = ax / al; ay = ay / al; az = az / al;
  float cx = t.ny * az - t.nz * ay, cy = t.nz * ax - t.nx * az, cz = t.nx * ay - t.ny * ax;  // b = n x a
  const float radius = 0.5f;
  ax = ax * radius; ay = ay * radius; az = az * radius;
  cx = cx * radius; cy = cy * radius; cz = cz * radius;
  const float div = 1.0f / sqrtf(2.0f);
  const float ux = (ax + cx) * div, uy = (ay + cy) * div, uz = (az + cz) * div;
  const float vx = (ax - cx) * div, vy = (ay - cy) * div, vz = (az - cz) * div;
  const float e[8] = {m_elev_sdf<PRIM>(m, t.px + ax, t.py + ay, t.pz + az), m_elev_sdf<PRIM>(m, t.px + cx, t.py + cy, t.pz + cz),
                      m_elev_sdf<PRIM>(m, t.px - ax, t.py - ay, t.pz - az), m_elev_sdf<PRIM>(m, t.px - cx, t.py - cy, t.pz - cz),
                      m_elev_sdf<PRIM>(m, t.px + ux, t.py + uy, t.pz + uz), m_elev_sdf<PRIM>(m, t.px + vx, t.py + vy, t.pz + vz),
                      m_elev_sdf<PRIM>(m, t.px - ux, t.py - uy, t.pz - uz), m_elev_sdf<PRIM>(m, t.px - vx, t.py - vy, t.pz - vz)};
  float e1 = e[0], e2 = e[0];
#pragma unroll
  for (int i = 0; i < 8; i++) { e1 = fminf(e1, e[i]); e2 = fmaxf(e2, e[i]); }
  const float md = (e2 - e1) * 0.1f;
  t.slope = m_atan(md / radius);
}

__device__ __forceinline__ void m_biome(MTile& t) {  // :153-190
  const float T = t.temperature, P = t.precipitation;
  if (t.elevation < 0.0f) t.biome = kBiomeWater;
  else if (T > 20.0f)
    t.biome = P < 40.0f ? kBiomeDesert : (P < 130.0f ? kBiomeSavanna : (P < 230.0f ? kBiomeTropicalSeasonal : kBiomeTropicalRain));
  else if (T > 5.0f)
    t.biome = P < 30.0f ? kBiomeShrubland : (P < 100.0f ? kBiomeGrassland : (P < 200.0f ? kBiomeTemperateSeasonal : kBiomeTemperateRain));
  else if (T > -5.0f) t.biome = P < 30.0f ? kBiomeBare : kBiomeTaiga;
  else t.biome = P < 10.0f ? kBiomeBare : kBiomeTundra;
}

__device__ __forceinline__ void m_type(MTile& t) {  // :192-200
  if (t.elevation < 0.0f) t.type = kTypeWater;
  else if (t.slope > 20.0f / kRadToDeg) t.type = kTypeCliffs;
  else t.type = kTypeFlat;
}

__device__ __forceinline__ void m_bedrock(const MCtx& c, const DMaterial& m, MTile& t) {  // :202-261
  const float dn = m_cubic1(c, ms(m, 5), 0.0031f, t, c.on) * 0.5f + 0.501f;
  const float depth = dn * dn * 2.0f;
  const float freq = m_cubic1(c, ms(m, 6), 0.013f, t, c.on) * 0.15f + 1.0f;
  const float fx = t.px * freq, fy = t.py * freq, fz = t.pz * freq;
  const MCell cell = m_cell_at<kDistHybrid>(c, ms(m, 4), 0.017f, fx, fy, fz, c.on);
  const float cr = m_ret_sub(cell);
  const float cracks = m_sat(m_pow(cr * 0.5f + 0.5f, 0.7f));
  const float value = m_ret_cell(cell);
  const float sat = m_sat(m_cubic_fbm<2>(c, ms(m, 7), 0.0022f, t, c.on) * 0.35f + 0.3f);
  m_hsv_to_rgb(0.07f, sat, m_sat(value * 0.1f + 0.7f) * (cracks * 0.4f + 0.6f), t.r, t.g, t.b);
  t.roughness = m_lerp(0.9f, value * -0.15f + 0.65f, cracks);
  t.height = cracks * depth;
}

__device__ __forceinline__ void m_cliffs(const MCtx& c, const DMaterial& m, MTile& t) {  // :263-293
  const float bf = m_steepness(t.slope, 19.0f, 4.0f);
  if (bf > 0.99999f) return;
  float h, s, v;
  m_rgb_to_hsv(t.r, t.g, t.b, h, s, v);
  h = m_lerp(155.0f / 255.0f, h, m_sharp_edge(bf, 0.005f));
  s = s * (bf * 0.4f + 0.6f);
  v = m_lerp(0.7f, s, bf * 0.8f + 0.2f);
  m_hsv_to_rgb(h, s, v, t.r, t.g, t.b);
  t.roughness = t.roughness * (bf * 0.2f + 0.8f);
  const float cracks = m_sharp_edge(
      m_sat(m_simplex_sum<true, 2>(c, ms(m, 8), 0.047f, 2.0f, 0.5f, t.px, t.py, t.pz) * 2.0f - 1.1f), 0.2f);
  t.height = t.height * m_lerp(1.0f, 0.8f, cracks);
  const float k = m_lerp(1.0f, 0.9f, cracks);
  t.r = t.r * k; t.g = t.g * k; t.b = t.b * k;
  t.roughness = m_lerp(t.roughness, 0.9f, cracks);
}

__device__ __forceinline__ void m_mica(const MCtx& c, const DMaterial& m, MTile& t) {  // :295-336
  if (!m.flowers) return;
  const float bf =
      m_sat((m_ret_mul(m_cell<kDistHybrid>(c, ms(m, 9), 0.02f, t, c.on)) - 0.98f) * 10.0f);
  const bool need = c.on && !(bf < 1e-7f);
  if (!m_any(need)) return;
  const MCell cell = m_cell<kDistManhattan>(c, ms(m, 10), 0.05f, t, need);
  if (!need) return;
  const float cracks = m_sharp_edge(m_sat(m_ret_div(cell) + 0.6f));
  const float r = m_lerp(122.0f / 255.0f, 184.0f / 255.0f, cracks);
  const float g = m_lerp(90.0f / 255.0f, 209.0f / 255.0f, cracks);
  const float b = m_lerp(88.0f / 255.0f, 187.0f / 255.0f, cracks);
  m_blend(t, r, g, b, cracks * 0.3f + 0.4f, 1.0f, t.height * 0.5f, bf);
}

__device__ __forceinline__ void m_dirt(const MCtx& c, const DMaterial& m, MTile& t) {  // :338-402
  float height = m_perlin_fbm<3>(c, ms(m, 11), 0.05f, 2.3f, 0.4f, t.px, t.py, t.pz) * 0.2f + 0.5f;
  const float bf = m_sharp_edge(m_sat(height - t.height + 0.4f)) * m_steepness(t.slope, 20.0f, 5.0f);
  const bool need = c.on && !(bf < 1e-7f);
  if (!m_any(need)) return;
  const float cn = m_cubic_fbm<4>(c, ms(m, 13), 0.02f, t, need);
  if (!need) return;
  float r = 168.0f / 255.0f, g = 94.0f / 255.0f, b = 28.0f / 255.0f;
  {
    const float saturation = m_range_mask(t.precipitation, 0.0f, 50.0f);
    float h, s, v;
    m_rgb_to_hsv(r, g, b, h, s, v);
    s = s * (saturation * 0.7f);
    v = v * 0.8f;
    m_hsv_to_rgb(h, s, v, r, g, b);
  }
  float rough = 0.8f;
  float cracks = m_sharp_edge(
      m_sat(m_simplex_sum<true, 2>(c, ms(m, 12), 0.07f, 2.0f, 0.5f, t.px, t.py, t.pz) * 2.0f - 1.2f), 0.15f);
  const float cm = m_smoothstep(m_sat(cn * 0.5f + 0.5f));
  cracks = cracks * (cm * cm * 0.9f + 0.1f);
  cracks = cracks * (m_range_mask(t.precipitation, 70.0f, 20.0f) * 0.9f + 0.1f);
  height = m_lerp(height, height * 0.5f, cracks);
  r = m_lerp(r, 0.1f, cracks); g = m_lerp(g, 0.1f, cracks); b = m_lerp(b, 0.1f, cracks);
  rough = m_lerp(rough, 0.9f, cracks);
  m_blend(t, r, g, b, rough, 0.0f, height, bf);
}

__device__ __forceinline__ void m_sand(const MCtx& c, const DMaterial& m, MTile& t) {  // :404-465
  const float bf = m_range_mask(t.temperature, 24.0f, 28.0f) * m_steepness(t.slope, 19.0f, 10.0f);
  const bool need = c.on && !(bf < 1e-7f);
  if (!m_any(need)) return;
  const float hue = m_cubic_fbm<2>(c, ms(m, 17), 0.02f, t, need) * 0.1f;
  if (!need) return;
  const float hs = m_simplex_sum<false, 3>(c, ms(m, 14), 0.001f, 2.0f, 0.5f, t.px, t.py, t.pz) * 0.3f + 1.0f;
  const float height =
      (m_simplex_sum<true, 3>(c, ms(m, 15), 0.01f, 2.0f, 0.7f, t.px * hs, t.py * hs, t.pz * hs) * 0.2f) *
          (m_range_mask(t.precipitation, 100.0f, 50.0f) * 0.4f + 0.6f) +
      0.5f;
  const float cs = m_smootherstep(m_smootherstep(
      m_perlin1(c, ms(m, 16), 0.0008f, t.px, t.py, t.pz) * 0.5f + 0.5f));
  float r = 189.0f / 255.0f, g = 174.0f / 255.0f, b = 152.0f / 255.0f;
  m_hue_shift(r, g, b, hue);
  m_mix_color(r, g, b, 187.0f / 255.0f, 104.0f / 255.0f, 50.0f / 255.0f, cs, r, g, b);
  m_deviation(r, g, b, 0.08f, ms(m, 42), t.px, t.py, t.pz);
  {
    float h, s, v;
    m_rgb_to_hsv(r, g, b, h, s, v);
    m_hsv_to_rgb(h * 1.0f, s * 0.7f, v * 0.8f, r, g, b);
  }
  m_blend(t, r, g, b, (hs - 1.0f) * 0.7f + 0.55f + hue, 0.0f, height, bf);
}

__device__ __forceinline__ void m_grass(const MCtx& c, const DMaterial& m, MTile& t) {  // :467-533
  const float bf = m_range_mask(t.temperature, 35.0f, 25.0f) * m_range_mask(t.precipitation, 15.0f, 35.0f) *
                   m_steepness(t.slope, 22.0f, 3.0f) * m_beach(m, t);
  const bool need = c.on && !(bf < 1e-7f);
  if (!m_any(need)) return;
  const MCell patch = m_cell<kDistHybrid>(c, ms(m, 18), 0.1f, t, need);
  const MCell scratch = m_cell<kDistHybrid>(c, ms(m, 20), 0.3f, t, need);
  if (!need) return;
  const float dry = fminf(fmaxf(t.temperature - (t.precipitation + 100.0f) * 30.0f / 400.0f, 0.0f), 5.0f) / 5.0f;
  const float hsb = m_perlin_fbm<2>(c, ms(m, 19), 0.01f, 2.0f, 0.5f, t.px, t.py, t.pz);
  const float hue = hsb * 0.09f - dry * 0.1f;
  float r = 114.0f / 255.0f, g = 187.0f / 255.0f, b = 77.0f / 255.0f;
  m_hue_shift(r, g, b, hue);
  const float pm = m_sharp_edge(m_ret_cell(patch) * 0.5f + 0.2f);
  const float patches =
      m_pow(m_ret_sub(patch) * 0.5f + 0.5f, 0.5f) *
      pm * (1.0f - dry * 0.8f);
  const float k1 = 1.0f - patches * 0.09f;
  r = r * k1; g = g * k1; b = b * k1;
  const float scr =
      m_sat(m_ret_mul(scratch) - 0.2f) *
      (1.0f - dry * 0.5f);
  const float k2 = 1.0f - scr * 0.1f;
  r = r * k2; g = g * k2; b = b * k2;
  const float rough = 0.6f + dry * 0.1f + patches * 0.1f + scr * 0.1f - hsb * 0.1f;
  const float height = m_lerp(t.height, 0.5f, 0.7f) + (0.5f - dry) * 0.2f + patches * 0.05f - scr * 0.02f + hsb * 0.1f + 0.1f;
  m_blend(t, r, g, b, rough, 0.0f, height, bf);
}

__device__ __forceinline__ void m_boulders(const MCtx& c, const DMaterial& m, MTile& t) {  // :535-615
  if (!m.flowers) return;
  const bool need = c.on && !(m_perlin1(c, ms(m, 21), 0.01f, t.px, t.py, t.pz) < 0.15f);
  if (!m_any(need)) return;
  const v4f q = m_voronoi_plane<2>(c.lds, ms(m, 22), 200.0f, t.px, t.py, t.pz, t.nx, t.ny, t.nz, need);
  if (!need) return;
  const float dist = m_dist(q.x, q.y, q.z, t.px, t.py, t.pz);
  const float size = m_smootherstep(m_smootherstep(
                         m_sat(m_perlin1(c, ms(m, 23), 0.09f, t.px, t.py, t.pz) * 0.5f + 0.5f))) *
                         3.0f +
                     3.0f;
  const float bf = m_range_mask(size - dist, 0.0f, 0.5f);
  if (bf < 1e-7f) return;
  const float hue = m_perlin1(c, ms(m, 24), 0.3f, t.px, t.py, t.pz) * 0.12f;
  const float val = m_perlin1(c, ms(m, 25), 0.5f, t.px, t.py, t.pz) * 0.18f;
  float h, s, v;
  m_rgb_to_hsv(154.0f / 255.0f, 154.0f / 255.0f, 154.0f / 255.0f, h, s, v);
  h = m_mod1(h + hue + 1.0f);
  v = m_sat(v + val);
  float r, g, b;
  m_hsv_to_rgb(h, s, v, r, g, b);
  const float rough = m_perlin1(c, ms(m, 26), 0.5f, t.px, t.py, t.pz) * 0.1f + 0.4f;
  const float rel = dist / size;
  m_blend(t, r, g, b, rough, 0.0f, 1.0f - rel * rel * 0.5f, bf);
}

__device__ __forceinline__ void m_water(const MCtx& c, const DMaterial& m, MTile& t) {  // :617-656
  const float sw = m_perlin_fbm<2>(c, ms(m, 27), 0.0015f, 2.0f, 0.5f, t.px, t.py, t.pz) * 0.5f + 0.5f;
  const float hue = m_cubic_fbm<3>(c, ms(m, 28), 0.004f, t, c.on) * 0.09f;
  m_mix_color(40.0f / 255.0f, 63.0f / 255.0f, 168.0f / 255.0f, 39.0f / 255.0f, 154.0f / 255.0f, 186.0f / 255.0f, sw,
              t.r, t.g, t.b);
  m_hue_shift(t.r, t.g, t.b, hue);
  const float a = m_range_mask(t.elevation, -25.0f, 3.0f);
  const float d1 = 1.0f - a * a;
  const float d2 = m_rescale(m_range_mask(t.elevation, 0.0f, -100.0f), 0.0f, 1.0f, 0.7f, 1.0f);
  t.opacity = d1 * d2;
  t.metallic = m_smoothstep(m_range_mask(t.elevation, 3.0f, -30.0f));
}

__device__ __forceinline__ void m_flowers(const MCtx& c, const DMaterial& m, MTile& t) {  // :658-744
  if (!m.flowers) return;
  const bool lily = m.purpose != UPF_PURPOSE_LAND;
  bool need = c.on && (t.biome == kBiomeWater) == lily;
  need = need && !(m_range_mask(fabsf(t.temperature - 18.0f), 12.0f, 7.0f) < 1e-5f);
  need = need && (lily || !(m_range_mask(fabsf(t.precipitation - 200.0f), 100.0f, 70.0f) < 1e-5f));
  if (!m_any(need)) return;
  const v4f q = m_voronoi_plane<1>(c.lds, ms(m, 30), 35.0f, t.px, t.py, t.pz, t.nx, t.ny, t.nz, need);
  const float ex = q.x - t.px, ey = q.y - t.py, ez = q.z - t.pz;
  need = need && !(ex * ex + ey * ey + ez * ez > 16.0f);
  if (!m_any(need)) return;
  const v4f k = m_voronoi_plane<1>(c.lds, ms(m, 29), 200.0f, t.px, t.py, t.pz, t.nx, t.ny, t.nz, need);
  const float fx = q.x - k.x, fy = q.y - k.y, fz = q.z - k.z;
  need = need && !(fx * fx + fy * fy + fz * fz > 400.0f);
  if (!need) return;
  const float dist = m_dist(q.x, q.y, q.z, t.px, t.py, t.pz);
  const float size = m_smootherstep(m_smootherstep(
                         m_sat(m_perlin1(c, ms(m, 31), 0.35f, t.px, t.py, t.pz) * 0.5f + 0.5f))) *
                         2.0f +
                     1.5f;
  const float bf = m_range_mask(size - dist, 0.0f, 0.1f);
  if (bf < 1e-7f) return;
  float r, g, b;
  if (lily) { r = 0.2f; g = 0.14f; b = 0.0f; }
  else {
    const float sel = m_sharp_edge(m_perlin1(c, ms(m, 32), 0.02f, k.x, k.y, k.z) + 0.4f, 0.2f);
    m_mix_color(0.5f, 0.0f, 0.35f, 0.5f, 0.4f, 0.0f, sel, r, g, b);
  }
  m_hue_shift(r, g, b,
              m_perlin1(c, ms(m, 33), 0.005f, t.px, t.py, t.pz) * 0.1f +
                  m_perlin1(c, ms(m, 34), 0.4f, t.px, t.py, t.pz) * 0.1f);
  const float rel = dist / size;
  m_blend(t, r, g, b, 0.8f, lily ? 0.85f : 0.0f, 0.7f + rel * rel * 0.2f, bf);
  t.opacity = m_lerp(t.opacity, 1.0f, bf);
}

__device__ __forceinline__ void m_ice(const MCtx& c, const DMaterial& m, MTile& t) {  // :746-817
  const float off = m_value1(ms(m, 35), 0.035f, t.px, t.py, t.pz) * 1.5f;
  const float bf = m_sharp_edge(m_range_mask(t.temperature + off, 0.0f, -3.0f)) * (1.0f - m_beach(m, t));
  const bool need = c.on && !(bf < 1e-7f);
  if (!m_any(need)) return;
  const float freq = m_value_fbm<3>(ms(m, 36), 0.01f, 2.0f, 0.5f, t.px, t.py, t.pz) * 0.08f + 1.0f;
  const float fx = t.px * freq, fy = t.py * freq, fz = t.pz * freq;
  const MCell c0 = m_cell_at<kDistHybrid>(c, ms(m, 37), 0.05f, fx, fy, fz, need);
  const MCell c1 = m_cell_at<kDistHybrid>(c, ms(m, 37) + 1u, 0.05f * 2.0f, fx, fy, fz, need);
  if (!need) return;
  if (bf > 0.1f && t.type != kTypeCliffs) t.type = kTypeRough;
  // both fBm sums over the same two octaves
  const float cells = m_fractal<false, 2>(0.05f, 2.0f, 0.5f, [&](uint32_t k, float) { return m_ret_cell(k ? c1 : c0); });
  const float subs = m_fractal<false, 2>(0.05f, 2.0f, 0.5f, [&](uint32_t k, float) { return m_ret_sub(k ? c1 : c0); });
  const float thick = m_sharp_edge(m_sat(cells * 0.5f + 0.8f), 0.1f) * 0.6f + 0.4f;
  const float crack = 1.0f - m_pow(subs * 0.5f + 0.5f, 0.3f);
  float r = fmaxf(122.0f / 255.0f - crack * 0.3f, 0.0f);
  float g = fmaxf(162.0f / 255.0f - crack * 0.3f, 0.0f);
  float b = fmaxf(164.0f / 255.0f - crack * 0.3f, 0.0f);
  m_mix_color(t.r, t.g, t.b, r, g, b, thick, r, g, b);
  float rough = 0.15f + crack * 0.6f;
  rough = m_lerp(t.roughness, rough, thick);
  const float height = thick * 0.5f * (1.0f - crack * 0.8f);
  const float op = t.opacity;
  m_blend(t, r, g, b, rough, 0.0f, height, bf);
  t.opacity = m_lerp(op, op * 0.9f + thick * 0.5f, bf);
}

__device__ __forceinline__ void m_snow(const MCtx& c, const DMaterial& m, MTile& t) {  // :819-855
  float bf = m_sharp_edge(
      m_range_mask(t.elevation + m_value1(ms(m, 38), 0.055f, t.px, t.py, t.pz) * 20.0f,
                   220.0f, 240.0f) *
      m_steepness(t.slope, 25.0f, 5.0f));
  const bool need = c.on && !(bf < 1e-7f);  // thick only lowers bf
  if (!m_any(need)) return;
  const float thick = m_cubic_fbm<3>(c, ms(m, 39), 0.05f, t, need) * 0.5f + 0.5f;
  bf = bf * m_sat(thick * 0.5f + 0.7f);
  if (!need || bf < 1e-7f) return;
  const float v = 230.0f / 255.0f;
  m_blend(t, v, v, v, thick * 0.3f + 0.2f, 0.0f, 0.6f + t.height * 0.1f + thick * 0.3f, bf);
}

__device__ __forceinline__ void m_visualization(MTile& t) {  // :857-893
  float r, g, b;
  switch (t.biome) {
    case kBiomeBare: r = g = b = 187.0f; break;
    case kBiomeTundra: r = 175.0f; g = 226.0f; b = 255.0f; break;
    case kBiomeTaiga: r = 193.0f; g = 225.0f; b = 221.0f; break;
    case kBiomeShrubland: r = 200.0f; g = 110.0f; b = 62.0f; break;
    case kBiomeGrassland: r = 239.0f; g = 252.0f; b = 143.0f; break;
    case kBiomeTemperateSeasonal: r = 151.0f; g = 183.0f; b = 102.0f; break;
    case kBiomeTemperateRain: r = 118.0f; g = 169.0f; b = 92.0f; break;
    case kBiomeDesert: r = 221.0f; g = 187.0f; b = 76.0f; break;
    case kBiomeSavanna: r = 253.0f; g = 213.0f; b = 120.0f; break;
    case kBiomeTropicalSeasonal: r = 161.0f; g = 151.0f; b = 0.0f; break;
    case kBiomeTropicalRain: r = 50.0f; g = 122.0f; b = 30.0f; break;
    default: r = 0.0f; g = 0.0f; b = 255.0f; break;  // water
  }
  t.r = r / 255.0f; t.g = g / 255.0f; t.b = b / 255.0f;
  t.roughness = 0.7f;
}

__device__ __forceinline__ void m_finalize(MTile& t) {  // :895-902
  t.r = m_sat(t.r); t.g = m_sat(t.g); t.b = m_sat(t.b);
  t.roughness = m_sat(t.roughness);
  t.metallic = m_sat(t.metallic);
  t.height = m_sat(t.height);
  t.opacity = m_sat(t.opacity);
}

// terrainTile with the configured coloring mode (sources/coloringModes.cpp:905-966).
// The tile arrives with position and unit normal; albedo, roughness, metallic and height
// start at 0, opacity at 1.  Called by all 64 lanes of the wave.
template <bool PRIM>
__device__ __forceinline__ void material_tile(const MCtx& c, const DMaterial& m, MTile& t) {
  t.r = t.g = t.b = 0.0f;
  t.roughness = t.metallic = t.height = 0.0f;
  t.opacity = 1.0f;
  t.slope = t.temperature = t.precipitation = 0.0f;
  t.biome = kBiomeWater + 1;
  t.type = kTypeWater + 1;
  // generateElevation (:51-57)
  t.elevation = m.purpose == UPF_PURPOSE_LAND ? m_elev_sdf<PRIM>(m, t.px, t.py, t.pz)
                                               : elevation_eval<true, true>(m.field, t.px, t.py, t.pz);
  const bool water = m.purpose == UPF_PURPOSE_WATER;
  if (m.coloring == UPF_COLORING_BARREN) {  // :932-952
    m_slope<PRIM>(m, t);
    if (water) {
      t.biome = kBiomeWater;
      t.type = kTypeWater;
      m_water(c, m, t);
    } else {
      t.biome = kBiomeBare;
      t.type = kTypeFlat;
      m_bedrock(c, m, t);
      m_cliffs(c, m, t);
      m_mica(c, m, t);
      m_boulders(c, m, t);
    }
    m_finalize(t);
    return;
  }
  m_precipitation(c, m, t);
  m_temperature(c, m, t);
  m_slope<PRIM>(m, t);
  m_biome(t);
  m_type(t);
  if (m.coloring == UPF_COLORING_DEBUG) {  // :954-966
    m_visualization(t);
    if (water) t.opacity = 0.5f;
    m_finalize(t);
    return;
  }
  if (water) m_water(c, m, t);  // :905-930
  else {
    m_bedrock(c, m, t);
    m_cliffs(c, m, t);
    m_mica(c, m, t);
    m_dirt(c, m, t);
    m_sand(c, m, t);
    m_grass(c, m, t);
    m_boulders(c, m, t);
  }
  m_flowers(c, m, t);
  m_ice(c, m, t);
  if (!water) m_snow(c, m, t);
  m_finalize(t);
}

}  // namespace upf
