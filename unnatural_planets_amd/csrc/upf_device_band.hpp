// upf_device_band.hpp -- bands of grid rows: a wave takes 64 consecutive x nodes of R rows
// of one plane, as upf_device_row.hpp does with two, one octave at a time for all R rows.
//
// The lattice columns, their folds and the reads are those of upf_device_row.hpp, so the
// values are the two-row form's bit for bit.  Both are bound by vector instructions; what a
// wider band saves is what every wave repeats: the rows' octave constants live in the
// registers of the lanes that fold their columns (lane = row + R * column), instead of a
// table in LDS; a round folds 64 / R columns of the octave for every row without looking up
// whose they are; the x part of an octave is computed once for R rows, and a Voronoi layer's
// feature points are hashed once for the rows of one cell, whose x offsets the rows share.
// Every branch on the spec stands outside the loop over the rows (inside it cost a fifth).
// Only layers that every wave evaluates in LDS come here (band_fits on the host): the code
// that would run a layer per lane alone took 7 % of the time, in registers.
// 512^3 torus (six ridged octaves, a mask and a Voronoi layer): 887 -> 525 vector
// instructions per 128 nodes, 1613 -> 863 us with the meshing (R = 4 was slower by a
// fiftieth, R = 16 by a fifteenth: spills).
#pragma once

#include <cmath>

#include "upf_device_row.hpp"

namespace upf {

constexpr int kBandRows = 8;
constexpr int kBandStride = 56;  // columns per row in LDS: rows 16 banks apart
static_assert(kBandRows * kBandStride <= kRowSlice2 && UPF_MAX_OCTAVES * kBandStride <= kRowSlice2, "the columns fit the slice");

constexpr int kWidePoints = 4 * kRowSlice / 3;  // feature points in the slice: x, y, z
constexpr int kWideCells = kWidePoints / 9;     // cells that 64 nodes may reach along x

inline bool reads_layers(const DSpec& s) {
  return s.n_layers > 0 && (s.compose == UPF_COMPOSE_LAND || s.compose == UPF_COMPOSE_NAVIGATION || s.compose == UPF_COMPOSE_ELEVATION_RAW);
}

// A band hashes a cellular octave's points once a row of cells, so rows far apart make them
// anew, for lanes that hold no more nodes.  512 x 64 x 300 nodes 8 m apart along x, with two
// cellular octaves, the rows `pitch` of the finer one's cells apart, row pairs / bands of four
// / of eight: at most 4 cells spanned, pitch 0.5 75 / 58 / 60 us, 1.2 75 / 72 / 75, 3 75 / 77 /
// 82 (with four octaves of gradient noise 84 / 66 / 65); 12 cells (band_cellular_wide), 0.7
// 219 / 183 / -, 0.9 219 / 214 / -, 1.2 219 / 236 / -, and with the gradient noise 0.7 146 /
// 138 / -, 0.9 147 / 154 / -; their adjoint (48 rows of 150 planes) 0.5 140 / 145 and 133 /
// 120, 0.7 140 / 153.
constexpr double kNearCells = 3.9;       // spanned by 64 nodes: the two-row form's reach (cells_in_slice)
constexpr double kNearPitch = 1.25, kWidePitch = 0.8, kWideGradPitch = 0.6;

// Whether every wave of a grid evaluates every layer of the spec in LDS, as columns or cells
// (no simplex, and the octaves' spans over 64 nodes fit).  The bound covers the rounding of
// the nodes' coordinates, so no wave needs more; near it the two-row form decides per wave.
inline bool band_fits(const DSpec& s, const DGrid& g) {
  if (!reads_layers(s)) return true;
  const double step = std::fabs((double)g.s[0]);
  const double reach = std::fabs((double)g.o[0]) + step * g.n[0];
  for (int l = 0; l < s.n_layers; l++) {
    const DLayer& L = s.L[l];
    if (L.noise == UPF_NOISE_SIMPLEX) return false;
    double columns = 0.0;
    const int oct = L.fractal == UPF_FRACTAL_NONE ? 1 : L.octaves;
    for (int k = 0; k < oct; k++) {
      const double f = std::fabs((double)L.freq[k]);
      const double span = f * (63.0 * step + reach * 0x1p-21);  // cells from end to end
      if (L.noise == UPF_NOISE_CELLULAR && !(span <= kWideCells - 3.1 && (span <= kNearCells || f * g.s[1] <= kWidePitch))) return false;
      columns += span + 3.0;
    }
    if (L.noise != UPF_NOISE_CELLULAR && !(columns <= kRowSlice2)) return false;
  }
  return true;
}

// Whether some wave may need band_cellular_wide: a cellular layer past the two-row form's
// reach (cells_in_slice).  The kernels that have it are instantiations of their own: its
// registers cost the others 12 %.
inline bool band_wide(const DSpec& s, const DGrid& g, int slice) {
  const double step = std::fabs((double)g.s[0]);
  const double reach = std::fabs((double)g.o[0]) + step * g.n[0];
  for (int l = 0; l < s.n_layers; l++) {
    const DLayer& L = s.L[l];
    if (L.noise != UPF_NOISE_CELLULAR) continue;
    const int oct = L.fractal == UPF_FRACTAL_NONE ? 1 : L.octaves;
    if (72 * oct > slice) return true;
    for (int k = 0; k < oct; k++)
      if (!(std::fabs((double)L.freq[k]) * (63.0 * step + reach * 0x1p-21) <= kNearCells)) return true;
  }
  return false;
}

// Whether a cellular octave's rows lie too far apart for bands of eight.
inline bool band_far(const DSpec& s, const DGrid& g) {
  if (!reads_layers(s)) return false;
  for (int l = 0; l < s.n_layers; l++) {
    const DLayer& L = s.L[l];
    if (L.noise != UPF_NOISE_CELLULAR) continue;
    for (int k = 0; k < (L.fractal == UPF_FRACTAL_NONE ? 1 : L.octaves); k++)
      if (std::fabs((double)L.freq[k]) * g.s[1] > kNearPitch) return true;
  }
  return false;
}

// Bands that a batch (of eight rows) or a grid's adjoint (of four) needs for its waves to
// fill the machine better than the row forms': 16 to a CU.
constexpr int64_t kBandItems = 4096;

inline int64_t band_items(const DGrid& g, int rows = kBandRows) {
  return (int64_t)((g.n[0] + 63) / 64) * ((g.n[1] + rows - 1) / rows) * g.n[2];
}

// Value v of row r's lane.
__device__ __forceinline__ float band_row(float v, int r) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), r));
}

// A node's value from its octave's columns e[0], e[1].
template <int NOISE>
__device__ __forceinline__ float band_read(const float2* e, float tx, float ux) {
  const float2 e0 = e[0], e1 = e[1];
  if (NOISE == UPF_NOISE_VALUE) return lerpf(e0.x, e1.x, ux);
  return lerpf(fmaf(e0.x, tx, e0.y), fmaf(e1.x, tx - 1.0f, e1.y), ux);
}

// One octave (frequency f, seed sk) of a gradient / value layer at this lane's node of R
// rows; yl: the y of row lane % R.
template <int NOISE, int R>
__device__ __forceinline__ void band_lattice(const RowCtx& c, float f, uint32_t sk, float x, float yl, float z, float* n) {
  float2* slice = reinterpret_cast<float2*>(c.slice);
  const int lane = lane_of(c);
  const float qx = x * f;
  const float fx = floorf(qx);
  int lo, hi;
  lane_range((int)fx, lo, hi);
  const int cols = hi - lo + 2;
  const float qy = yl * f, qz = z * f;
  const float fy = floorf(qy), fz = floorf(qz);
  const float ty = qy - fy, tz = qz - fz;
  const uint32_t y0 = (uint32_t)(int)fy * kPY, z0 = (uint32_t)(int)fz * kPZ;
  const float4 p0 = make_float4(ty, tz, fade(ty), fade(tz));
  const float4 p1 = make_float4(__uint_as_float(sk ^ y0 ^ z0), __uint_as_float(sk ^ (y0 + kPY) ^ z0),
                                __uint_as_float(sk ^ y0 ^ (z0 + kPZ)), __uint_as_float(sk ^ (y0 + kPY) ^ (z0 + kPZ)));
  const float tx = qx - fx;
  const float ux = fade(tx);
  const int o = (int)fx - lo;
  if (cols > kBandStride) {  // one row at a time
#pragma unroll
    for (int r = 0; r < R; r++) {
      const float4 q0 = make_float4(band_row(p0.x, r), p0.y, band_row(p0.z, r), p0.w);
      const float4 q1 = make_float4(band_row(p1.x, r), band_row(p1.y, r), band_row(p1.z, r), band_row(p1.w, r));
      for (int col = lane; col < cols; col += 64) slice[col] = fold_column<NOISE>(c, q0, q1, (uint32_t)(lo + col));
      wave_sync();
      n[r] = band_read<NOISE>(slice + o, tx, ux);
      wave_sync();
    }
    return;
  }
  float2* own = slice + (lane & (R - 1)) * kBandStride;
  for (int b = 0; b < cols; b += 64 / R) {
    const int col = b + lane / R;
    const float2 v = fold_column<NOISE>(c, p0, p1, (uint32_t)(lo + col));
    if (col < cols) own[col] = v;
  }
  wave_sync();
#pragma unroll
  for (int r = 0; r < R; r++)
    n[r] = band_read<NOISE>(slice + r * kBandStride + o, tx, ux);
  wave_sync();
}

// One octave of a cellular layer.  The rows of one lattice cell share its feature points:
// p_x per point, and per row the point's squared y and z distance.
template <int R>
__device__ __forceinline__ void band_cellular(const RowCtx& c, const DLayer& L, float f, uint32_t sk, float x, float yl,
                                              float z, float* n) {
  float* px = reinterpret_cast<float*>(c.slice);
  float* pe = px + 72;
  static_assert(72 * (R + 1) <= 4 * kRowSlice, "points and rows fit the slice");
  const float qx = x * f, qz = z * f;
  const int ix = (int)rintf(qx);
  int lo, hi;
  lane_range(ix, lo, hi);
  const int cyl = (int)rintf(yl * f), cz = __builtin_amdgcn_readfirstlane((int)rintf(qz));
  for (int r0 = 0; r0 < R;) {
    const int cy = __builtin_amdgcn_readlane(cyl, r0);
    const uint32_t rows = (uint32_t)__ballot(cyl == cy) & ((1u << R) - 1u);  // lane r holds row r
    {
      const CellLane cl = cell_lane(c.lane);
      const int kx = lo - 1 + cl.lx, ky = cy - 1 + cl.dy, kz = cz - 1 + cl.dz;
      const uint32_t h = (sk ^ ((uint32_t)kx * kPX) ^ ((uint32_t)ky * kPY) ^ ((uint32_t)kz * kPZ)) * kHM;
      const uint32_t m = h ^ (h >> 15);
      const float py = fmaf((float)((m >> 10) & 1023u), L.js, (float)ky - L.j0);
      const float ez = fmaf((float)((m >> 20) & 1023u), L.js, (float)kz - L.j0) - qz;
      if (cl.c9 < 9) {
        const int at = cl.lx + 8 * cl.c9;
        px[at] = fmaf((float)(m & 1023u), L.js, (float)kx - L.j0);
#pragma unroll
        for (int r = 0; r < R; r++) {
          const float ey = py - band_row(yl, r) * f;
          if ((rows >> r) & 1u) pe[72 * r + at] = fmaf(ez, ez, ey * ey);
        }
      }
    }
    wave_sync();
    const int o = ix - lo;
    float d[27];
#pragma unroll
    for (int q = 0; q < 27; q++) d[q] = px[o + q % 3 + 8 * (q / 3)] - qx;
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (!((rows >> r) & 1u)) continue;
      const float* e = pe + 72 * r + o;
      float best = __builtin_inff();
#pragma unroll
      for (int q = 0; q < 27; q++) best = fminf(best, fmaf(d[q], d[q], e[q % 3 + 8 * (q / 3)]));
      n[r] = sqrt_hw(best);
    }
    wave_sync();
    r0 += __popc(rows);
  }
}

// The feature points (x, y, z - q_z) of the cells that a wave's nodes reach in one row of
// cells cy, as entry lx + stride * (dy + 3 dz) of three arrays: as many cells as fit.
__device__ __forceinline__ void wide_points(const RowCtx& c, const DLayer& L, uint32_t sk, int lo, int n, int cy, int cz,
                                            float qz) {
  float* px = reinterpret_cast<float*>(c.slice);
  const CellLane cl = cell_lane(c.lane);
  const int ky = cy - 1 + cl.dy, kz = cz - 1 + cl.dz;
  for (int b = cl.lx; b < n; b += 7) {
    const int kx = lo - 1 + b;
    const uint32_t h = (sk ^ ((uint32_t)kx * kPX) ^ ((uint32_t)ky * kPY) ^ ((uint32_t)kz * kPZ)) * kHM;
    const uint32_t m = h ^ (h >> 15);
    if (cl.c9 < 9) {
      const int at = b + n * cl.c9;
      px[at] = fmaf((float)(m & 1023u), L.js, (float)kx - L.j0);
      px[kWidePoints + at] = fmaf((float)((m >> 10) & 1023u), L.js, (float)ky - L.j0);
      px[2 * kWidePoints + at] = fmaf((float)((m >> 20) & 1023u), L.js, (float)kz - L.j0) - qz;
    }
  }
}

// One octave of a cellular layer whose lanes span more cells than the two-row form takes:
// the distances in the order of the per-lane form, which that form then runs, the points
// hashed once a wave.  Torus with six octaves and a cellular layer at 6 per unit, 240^3: 269
// us with the layer per lane, 143 here.
template <int R>
__device__ __forceinline__ void band_cellular_wide(const RowCtx& c, const DLayer& L, float f, uint32_t sk, float x, float yl,
                                                   float z, float* n) {
  const float* px = reinterpret_cast<const float*>(c.slice);
  const float qx = x * f, qz = z * f;
  const int ix = (int)rintf(qx);
  int lo, hi;
  lane_range(ix, lo, hi);
  const int cells = hi - lo + 3;
  const int cyl = (int)rintf(yl * f), cz = __builtin_amdgcn_readfirstlane((int)rintf(qz));
  for (int r0 = 0; r0 < R;) {
    const int cy = __builtin_amdgcn_readlane(cyl, r0);
    const uint32_t rows = (uint32_t)__ballot(cyl == cy) & ((1u << R) - 1u);  // lane r holds row r
    wide_points(c, L, sk, lo, cells, cy, cz, qz);
    wave_sync();
    float best[R];
#pragma unroll
    for (int r = 0; r < R; r++) best[r] = __builtin_inff();
    for (int c9 = 0; c9 < 9; c9++) {
      const float* p = px + (ix - lo) + cells * c9;
#pragma unroll
      for (int q = 0; q < 3; q++) {
        const float dx = p[q] - qx, py = p[kWidePoints + q], dz = p[2 * kWidePoints + q];
        const float dxx = dx * dx;
#pragma unroll
        for (int r = 0; r < R; r++) {
          const float dy = py - band_row(yl, r) * f;
          best[r] = fminf(best[r], fmaf(dz, dz, fmaf(dy, dy, dxx)));
        }
      }
    }
#pragma unroll
    for (int r = 0; r < R; r++)
      if ((rows >> r) & 1u) n[r] = sqrt_hw(best[r]);
    wave_sync();
    r0 += __popc(rows);
  }
}

// Whether the two-row form evaluates a cellular layer in LDS: at most 5 cells spanned, all
// octaves in the slice.
__device__ __forceinline__ bool cells_in_slice(const DLayer& L, int oct, float x, int slice) {
  bool fits = 72 * oct <= slice;
  for (int k = 0; k < oct; k++) {
    int lo, hi;
    lane_range((int)rintf(x * L.freq[k]), lo, hi);
    fits = fits && hi - lo <= 4;
  }
  return __builtin_amdgcn_readfirstlane(fits);
}

// One layer at this lane's node of R rows.
template <int R, bool WIDE>
__device__ __forceinline__ void band_layer(const RowCtx& c, const DLayer& L, float x, float yl, float z, float* out) {
  const int oct = L.fractal == UPF_FRACTAL_NONE ? 1 : L.octaves;
  const bool wide = WIDE && L.noise == UPF_NOISE_CELLULAR && !cells_in_slice(L, oct, x, kRowSlice2);
#pragma unroll
  for (int r = 0; r < R; r++) out[r] = 0.0f;
  for (int k = 0; k < oct; k++) {
    const float f = L.freq[k], amp = L.amp[k];
    const uint32_t sk = L.seed + (uint32_t)k;
    float n[R];
    if (L.noise == UPF_NOISE_GRADIENT) {
      band_lattice<UPF_NOISE_GRADIENT, R>(c, f, sk, x, yl, z, n);
    } else if (L.noise == UPF_NOISE_VALUE) {
      band_lattice<UPF_NOISE_VALUE, R>(c, f, sk, x, yl, z, n);
    } else if (wide) {
      band_cellular_wide<R>(c, L, f, sk, x, yl, z, n);
    } else {
      band_cellular<R>(c, L, f, sk, x, yl, z, n);
    }
    if (L.fractal == UPF_FRACTAL_RIDGED) {
#pragma unroll
      for (int r = 0; r < R; r++) n[r] = fmaf(-2.0f, fabsf(n[r]), 1.0f);
    }
    if (L.fractal == UPF_FRACTAL_NONE) {
#pragma unroll
      for (int r = 0; r < R; r++) out[r] = n[r];
    } else {
#pragma unroll
      for (int r = 0; r < R; r++) out[r] = fmaf(amp, n[r], out[r]);
    }
  }
}

// f at this lane's node of R rows (row_field's values).
template <int R, bool COMPOSED, bool WIDE>
__device__ __forceinline__ void band_field(const RowCtx& c, const DSpec& s, float x, float yl, float z, float* out) {
  const bool need_elev = s.compose == UPF_COMPOSE_LAND || s.compose == UPF_COMPOSE_NAVIGATION ||
                         s.compose == UPF_COMPOSE_ELEVATION_RAW;
  float acc[R], m[R];
#pragma unroll
  for (int r = 0; r < R; r++) acc[r] = m[r] = 0.0f;
  for (int l = 0; need_elev && l < s.n_layers; l++) {
    const DLayer& L = s.L[l];
    float v[R];
    band_layer<R, WIDE>(c, L, x, yl, z, v);
#pragma unroll
    for (int r = 0; r < R; r++) v[r] = L.weight * v[r];
    if (L.blend == UPF_BLEND_ADD) {
#pragma unroll
      for (int r = 0; r < R; r++) acc[r] = acc[r] + v[r];
    } else if (L.blend == UPF_BLEND_MASK) {
#pragma unroll
      for (int r = 0; r < R; r++) m[r] = __builtin_amdgcn_fmed3f(v[r] + 0.5f, 0.0f, 1.0f);
    } else {
#pragma unroll
      for (int r = 0; r < R; r++) acc[r] = fmaf(m[r], v[r] - acc[r], acc[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < R; r++) {
    const float shape = s.compose == UPF_COMPOSE_ELEVATION_RAW ? 0.0f : shape_eval<false, COMPOSED>(s, x, band_row(yl, r), z);
    switch (s.compose) {
      case UPF_COMPOSE_LAND: out[r] = shape - s.escale * acc[r]; break;
      case UPF_COMPOSE_WATER: out[r] = shape; break;
      case UPF_COMPOSE_NAVIGATION: out[r] = shape - s.escale * fmaxf(acc[r], 0.0f); break;
      case UPF_COMPOSE_ELEVATION: out[r] = shape / s.escale; break;
      default: out[r] = acc[r]; break;
    }
  }
}

}  // namespace upf
