// upf_device_band_grad.hpp -- the fused forward + adjoint of upf_device_row_grad.hpp over
// bands of R grid rows, as upf_device_band.hpp is the forward field's: one octave at a time,
// the rows' octave constants in the lanes that fold their columns, the x part of an octave
// computed once for R rows, a Voronoi layer's points hashed once for the rows of one cell,
// and one wave sum per parameter and band instead of one per row.
//
// For layer stacks without a mask, which need no layer twice and whose layers' coefficients
// are the same at every node; f and df/dp are the row kernel's bit for bit.  A cellular
// layer's nearest point is kept as its index: its coordinates are read once at the end (five
// selects a point before).  256^3, torus with 4 octaves and a cellular layer, all gradients:
// 460 us in rows, 243 in bands; 96^3 61 / 52, 160^3 172 / 96.  (Eight rows a band do not fit
// the registers: 5.5 ms.)
#pragma once

#include "upf_device_band.hpp"
#include "upf_device_row_grad.hpp"

namespace upf {

constexpr int kBandGradRows = 4;
constexpr int kBandGradStride = 42;  // columns per row and plane in LDS
constexpr int kBandGradPlane = kBandGradRows * kBandGradStride;
static_assert(3 * kBandGradPlane <= kRowSlice2, "three planes of columns fit the slice");

// Whether every wave of a grid evaluates the spec's gradient in bands (as band_fits), with
// the row kernel's choice of layers in LDS.
inline bool band_grad_fits(const DSpec& s, const DGrid& g) {
  if (g.n[1] <= kBandGradRows / 2 || !s.all_add || spec_composed(s) || s.compose == UPF_COMPOSE_NAVIGATION) return false;
  if (s.compose != UPF_COMPOSE_LAND && s.compose != UPF_COMPOSE_ELEVATION_RAW) return true;  // no layer is read
  const double step = std::fabs((double)g.s[0]);
  const double reach = std::fabs((double)g.o[0]) + step * g.n[0];
  for (int l = 0; l < s.n_layers; l++) {
    const DLayer& L = s.L[l];
    if (L.noise == UPF_NOISE_SIMPLEX) return false;
    const bool cell = L.noise == UPF_NOISE_CELLULAR;
    const int oct = L.fractal == UPF_FRACTAL_NONE ? 1 : L.octaves;
    double columns = 0.0;
    for (int k = 0; k < oct; k++) {
      const double f = std::fabs((double)L.freq[k]);
      const double span = f * (63.0 * step + reach * 0x1p-21);
      if (!(span <= (cell ? kWideCells - 3.1 : kBandGradStride - 2.1))) return false;
      if (cell && span > kNearCells && f * g.s[1] > kWideGradPitch) return false;
      columns += span + 3.0;
    }
    if (!cell && !(3.0 * columns <= kRowSlice2)) return false;
  }
  return true;
}

inline int64_t band_grad_items(const DGrid& g) {
  return (int64_t)((g.n[0] + 63) / 64) * ((g.n[1] + kBandGradRows - 1) / kBandGradRows) * g.n[2];
}

// One octave of a gradient / value layer: n and dn/dq of this lane's node of R rows.
template <int NOISE, int R>
__device__ __forceinline__ void band_lattice_d(const RowCtx& c, float f, uint32_t sk, float x, float yl, float z, float* n,
                                               float* nx, float* ny, float* nz) {
  float2* slice = reinterpret_cast<float2*>(c.slice);
  const int lane = lane_of(c);
  const float qx = x * f;
  const float fx = floorf(qx);
  int lo, hi;
  lane_range((int)fx, lo, hi);
  const int cols = hi - lo + 2;
  {
    const float qy = yl * f, qz = z * f;
    const float fy = floorf(qy), fz = floorf(qz);
    const float ty = qy - fy, tz = qz - fz;
    const uint32_t y0 = (uint32_t)(int)fy * kPY, z0 = (uint32_t)(int)fz * kPZ;
    const float4 p0 = make_float4(ty, tz, fade(ty), fade(tz));
    const float4 p1 = make_float4(__uint_as_float(sk ^ y0 ^ z0), __uint_as_float(sk ^ (y0 + kPY) ^ z0),
                                  __uint_as_float(sk ^ y0 ^ (z0 + kPZ)), __uint_as_float(sk ^ (y0 + kPY) ^ (z0 + kPZ)));
    const float duy = dfade(ty), duz = dfade(tz);
    float2* own = slice + (lane & (R - 1)) * kBandGradStride;
    for (int b = 0; b < cols; b += 64 / R) {
      const int col = b + lane / R;
      float2 v, vy, vz;
      fold_column_d<NOISE>(c, p0, p1, duy, duz, (uint32_t)(lo + col), v, vy, vz);
      if (col < cols) {
        own[col] = v;
        own[kBandGradPlane + col] = vy;
        own[2 * kBandGradPlane + col] = vz;
      }
    }
  }
  const float tx = qx - fx, ux = fade(tx), dux = dfade(tx);
  const float2* e = slice + ((int)fx - lo);
  wave_sync();
#pragma unroll
  for (int r = 0; r < R; r++)
    n[r] = col_value_d<NOISE>(tx, ux, dux, e + r * kBandGradStride, kBandGradPlane, nx[r], ny[r], nz[r]);
  wave_sync();
}

// One octave of a cellular layer.
template <int R>
__device__ __forceinline__ void band_cellular_d(const RowCtx& c, const DLayer& L, float f, uint32_t sk, float x, float yl,
                                                float z, float* n, float* nx, float* ny, float* nz) {
  float* px = reinterpret_cast<float*>(c.slice);
  float *py = px + 72, *pz = px + 144, *pe = px + 216;  // x, y, q_z - z of the points; and per row
  static_assert(216 + 72 * R <= 4 * kRowSlice, "points and rows fit the slice");
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
      const float ypt = fmaf((float)((m >> 10) & 1023u), L.js, (float)ky - L.j0);
      const float ez = fmaf((float)((m >> 20) & 1023u), L.js, (float)kz - L.j0) - qz;
      if (cl.c9 < 9) {
        const int at = cl.lx + 8 * cl.c9;
        px[at] = fmaf((float)(m & 1023u), L.js, (float)kx - L.j0);
        py[at] = ypt;
        pz[at] = -ez;
#pragma unroll
        for (int r = 0; r < R; r++) {
          const float ey = ypt - band_row(yl, r) * f;
          if ((rows >> r) & 1u) pe[72 * r + at] = fmaf(ez, ez, ey * ey);
        }
      }
    }
    wave_sync();
    const int o = ix - lo;
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (!((rows >> r) & 1u)) continue;
      const float* e = pe + 72 * r + o;
      float best = __builtin_inff();
      int at = -1;
#pragma unroll
      for (int q = 0; q < 27; q++) {
        const float d = px[o + q % 3 + 8 * (q / 3)] - qx;
        const float d2 = fmaf(d, d, e[q % 3 + 8 * (q / 3)]);
        at = d2 < best ? q % 3 + 8 * (q / 3) : at;
        best = fminf(best, d2);
      }
      const int p = o + max(at, 0);
      const float rr = sqrt_hw(best);
      const float inv = rr > 0.0f ? 1.0f / rr : 0.0f;
      n[r] = rr;
      nx[r] = (qx - (at < 0 ? qx : px[p])) * inv;
      ny[r] = (at < 0 ? 0.0f : -(py[p] - band_row(yl, r) * f)) * inv;
      nz[r] = (at < 0 ? 0.0f : pz[p]) * inv;
    }
    wave_sync();
    r0 += __popc(rows);
  }
}

// The same over more cells, as band_cellular_wide.
template <int R>
__device__ __forceinline__ void band_cellular_wide_d(const RowCtx& c, const DLayer& L, float f, uint32_t sk, float x, float yl,
                                                     float z, float* n, float* nx, float* ny, float* nz) {
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
    int at[R];
#pragma unroll
    for (int r = 0; r < R; r++) { best[r] = __builtin_inff(); at[r] = -1; }
    for (int c9 = 0; c9 < 9; c9++) {
      const int o = ix - lo + cells * c9;
      const float* p = px + o;
#pragma unroll
      for (int q = 0; q < 3; q++) {
        const float dx = p[q] - qx, py = p[kWidePoints + q], dz = p[2 * kWidePoints + q];
        const float dxx = dx * dx;
#pragma unroll
        for (int r = 0; r < R; r++) {
          const float dy = py - band_row(yl, r) * f;
          const float d2 = fmaf(dz, dz, fmaf(dy, dy, dxx));
          at[r] = d2 < best[r] ? o + q : at[r];
          best[r] = fminf(best[r], d2);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (!((rows >> r) & 1u)) continue;
      const int p = max(at[r], 0);
      const float rr = sqrt_hw(best[r]);
      const float inv = rr > 0.0f ? 1.0f / rr : 0.0f;
      n[r] = rr;
      nx[r] = (at[r] < 0 ? 0.0f : qx - px[p]) * inv;
      ny[r] = (at[r] < 0 ? 0.0f : band_row(yl, r) * f - px[kWidePoints + p]) * inv;
      nz[r] = (at[r] < 0 ? 0.0f : -px[2 * kWidePoints + p]) * inv;
    }
    wave_sync();
    r0 += __popc(rows);
  }
}

// f, df/dp and (THETA) the sums of w df/dtheta at this lane's node of R rows.
template <int R, bool THETA, bool WIDE>
__device__ __forceinline__ void band_field_grad(const RowCtx& c, const DSpec& s, float x, float yl, float z,
                                                const float* w, float* out, float (*g)[3], ThetaAcc& acc) {
  const bool raw = s.compose == UPF_COMPOSE_ELEVATION_RAW;
  const bool need_elev = s.compose == UPF_COMPOSE_LAND || raw;
  float shape[R], dps[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  const float dshape = s.compose == UPF_COMPOSE_ELEVATION ? 1.0f / s.escale : 1.0f;
#pragma unroll
  for (int r = 0; r < R; r++) {
    float gs[3] = {0.0f, 0.0f, 0.0f}, dp[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    shape[r] = raw ? 0.0f : shape_eval_d<false, false>(s, x, band_row(yl, r), z, gs, dp);
#pragma unroll
    for (int a = 0; a < 3; a++) g[r][a] = dshape * gs[a];
#pragma unroll
    for (int i = 0; i < 4; i++) dps[i] = fmaf(w[r] * dshape, dp[i], dps[i]);
  }
  if (THETA && !raw) {
    const int np = shape_param_count(s.shape);
    for (int i = 0; i < 4; i++)
      if (i < np) acc.add(kThShape + i, i == 0 ? dps[0] : (i == 1 ? dps[1] : (i == 2 ? dps[2] : dps[3])));
  }
  float elev[R];
#pragma unroll
  for (int r = 0; r < R; r++) elev[r] = 0.0f;
  const float fe = raw ? 1.0f : -s.escale;
  for (int l = 0; need_elev && l < s.n_layers; l++) {
    const DLayer& L = s.L[l];
    const int oct = L.fractal == UPF_FRACTAL_NONE ? 1 : L.octaves;
    const bool wide = WIDE && L.noise == UPF_NOISE_CELLULAR && !cells_in_slice(L, oct, x, kRowSlice);
    const float coeff = fe * L.weight;
    float v[R];
#pragma unroll
    for (int r = 0; r < R; r++) v[r] = 0.0f;
    for (int k = 0; k < oct; k++) {
      const float f = L.freq[k], amp = L.amp[k];
      const uint32_t sk = L.seed + (uint32_t)k;
      float n[R], nx[R], ny[R], nz[R], dterm[R];
      if (L.noise == UPF_NOISE_GRADIENT) band_lattice_d<UPF_NOISE_GRADIENT, R>(c, f, sk, x, yl, z, n, nx, ny, nz);
      else if (L.noise == UPF_NOISE_VALUE) band_lattice_d<UPF_NOISE_VALUE, R>(c, f, sk, x, yl, z, n, nx, ny, nz);
      else if (wide) band_cellular_wide_d<R>(c, L, f, sk, x, yl, z, n, nx, ny, nz);
      else band_cellular_d<R>(c, L, f, sk, x, yl, z, n, nx, ny, nz);
      if (L.fractal == UPF_FRACTAL_RIDGED) {
#pragma unroll
        for (int r = 0; r < R; r++) {
          dterm[r] = (n[r] < 0.0f ? 2.0f : -2.0f) * amp;
          n[r] = fmaf(-2.0f, fabsf(n[r]), 1.0f);
        }
      } else {
#pragma unroll
        for (int r = 0; r < R; r++) dterm[r] = L.fractal == UPF_FRACTAL_NONE ? 1.0f : amp;
      }
      if (L.fractal == UPF_FRACTAL_NONE) {
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = n[r];
      } else {
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = fmaf(amp, n[r], v[r]);
      }
      float tf = 0.0f, ta = 0.0f;
#pragma unroll
      for (int r = 0; r < R; r++) {
        const float sf = coeff * dterm[r] * f;
        g[r][0] = fmaf(sf, nx[r], g[r][0]);
        g[r][1] = fmaf(sf, ny[r], g[r][1]);
        g[r][2] = fmaf(sf, nz[r], g[r][2]);
        if (THETA) {
          const float qdot = fmaf(nz[r], z, fmaf(ny[r], band_row(yl, r), nx[r] * x));
          const float ct = w[r] * coeff;
          tf = fmaf(ct * dterm[r], qdot, tf);
          ta = fmaf(ct, n[r], ta);
        }
      }
      if (THETA) {
        acc.add(kThFreq + l * UPF_MAX_OCTAVES + k, tf);
        if (L.fractal != UPF_FRACTAL_NONE) acc.add(kThAmp + l * UPF_MAX_OCTAVES + k, ta);
      }
    }
    float tw = 0.0f;
#pragma unroll
    for (int r = 0; r < R; r++) {
      elev[r] = fmaf(L.weight, v[r], elev[r]);
      tw = fmaf(w[r] * fe, v[r], tw);
    }
    if (THETA) acc.add(kThWeight + l, tw);
  }
#pragma unroll
  for (int r = 0; r < R; r++) {
    switch (s.compose) {
      case UPF_COMPOSE_LAND: out[r] = shape[r] - s.escale * elev[r]; break;
      case UPF_COMPOSE_ELEVATION: out[r] = shape[r] / s.escale; break;
      case UPF_COMPOSE_ELEVATION_RAW: out[r] = elev[r]; break;
      default: out[r] = shape[r]; break;
    }
  }
}

}  // namespace upf
