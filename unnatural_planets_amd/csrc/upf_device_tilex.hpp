// upf_device_tilex.hpp -- grid tiles in the exact form: the elevation modes and the further
// shapes over 16 x 4 nodes of R consecutive planes per wave (lane = x + 16 y), every
// operation rounded as the per-lane functions of upf_device.hpp (X = true) round it, so
// that the results are theirs bit for bit.
//
// Per octave the lattice points that a tile's nodes read are few: the lanes hash the box
// of them once into the wave's LDS, and every lane does its own trilinear sum in the
// per-lane order, x first.
//   value:    the lattice values; the x and y sums are shared by the planes of one lattice
//             cell, which leaves a plane one interpolation;
//   gradient: the gradient vectors; two components of a vector are not 0 and they are +-1,
//             so g_z tz + (g_y ty + g_x tx) in fused operations is gdot's one rounded sum,
//             and its x and y part is shared by the planes of one cell;
//   impact Voronoi: the points of the cells around the tile, one cell per lane;
//   simplex:  per lane (its lattice is skewed), the gradients from LDS.
// The planes' z parts are computed one per lane and read as scalars.  An octave whose box
// does not fit the LDS runs per lane.
//
// A tile is compact because the modes skip work that a whole wave does not need: of the
// lakes planet's waves at 500^3, 62% need the ridges at 64 x 2 nodes and 41% at 16 x 4 x 2
// (32% of the nodes do).
#pragma once

#include "upf_device_row.hpp"

namespace upf {

// Quotient a / b of small non-negative integers (a < 4096, 1 <= b <= 512; here a task or
// lane index and a region size) with the divisor given as rb = 1 / b in float32:
// (a + 1/2) / b lies at least 1 / (2 b) >= 2^-10 away from an integer, and the roundings
// of rb and of the product move it by less than 4096 * 2^-23 = 2^-11, so truncation
// gives the exact quotient (an integer division by a variable is a long correction
// sequence).
__device__ __forceinline__ int small_div(int a, float rb) { return (int)(((float)a + 0.5f) * rb); }

constexpr int kTX = 16, kTY = 4;   // nodes of a wave's tile in a plane
constexpr int kTLds = 256;         // float4 entries of LDS per wave
static_assert(kTX * kTY == 64, "a lane per node");

struct TileCtx {
  float4* lds;         // this wave's kTLds entries
  const float4* gtab;  // 16 gradient vectors in LDS
  int lane;
};

// The box of lattice cells of a tile: lowest point and points per axis (one more than
// cells); fits when its points are at most `cap`.
struct TileBox {
  int x, y, z, nx, ny, nz;
  bool fits;
};
__device__ __forceinline__ TileBox tile_box(int ix, int iy, int z0, int z1, int more, int cap) {
  const int x0 = __builtin_amdgcn_readfirstlane(ix), x1 = __builtin_amdgcn_readlane(ix, kTX - 1);
  const int y0 = __builtin_amdgcn_readfirstlane(iy), y1 = __builtin_amdgcn_readlane(iy, 64 - kTX);
  TileBox b;
  b.x = min(x0, x1); b.y = min(y0, y1); b.z = min(z0, z1);
  const uint32_t ex = (uint32_t)max(x0, x1) - (uint32_t)b.x, ey = (uint32_t)max(y0, y1) - (uint32_t)b.y,
                 ez = (uint32_t)max(z0, z1) - (uint32_t)b.z;
  b.nx = (int)ex + more; b.ny = (int)ey + more; b.nz = (int)ez + more;
  b.fits = ex < 1024u && ey < 1024u && ez < 1024u && b.nx * b.ny <= cap && b.nx * b.ny * b.nz <= cap;
  return b;
}
// make(e, i, j, k) for the box's points e = i + nx (j + ny k), one per lane
template <class Make>
__device__ __forceinline__ void tile_fill(int lane, const TileBox& b, Make make) {
  // 1 ulp reciprocals: small_div's margin for quotients of up to 1,024 is 2^13 ulps
  const float rx = __builtin_amdgcn_rcpf((float)b.nx), ry = __builtin_amdgcn_rcpf((float)b.ny);
  const int n = b.nx * b.ny * b.nz;
  wave_sync();  // earlier readers are done
  for (int e = lane; e < n; e += 64) {
    const int q = small_div(e, rx), k = small_div(q, ry);
    make(e, e - q * b.nx, q - k * b.ny, k);
  }
  wave_sync();
}

// What runs per lane, out of line: rarely needed, and inlined it would be most of the
// kernel's code.
__device__ __noinline__ float lane_gradient(uint32_t seed, float x, float y, float z) { return noise_gradient<true>(seed, x, y, z); }
__device__ __noinline__ float lane_value(uint32_t seed, float x, float y, float z) { return noise_value<true>(seed, x, y, z); }
__device__ __noinline__ float lane_cellular(uint32_t seed, float x, float y, float z, float js, float j0) {
  return noise_cellular<true>(seed, x, y, z, js, j0);
}
struct Point3 {
  float x, y, z;
};
__device__ __noinline__ Point3 lane_voronoi(uint32_t seed, int ppc, float cell, float x, float y, float z) {
  float c[3];
  voronoi_nearest(seed, ppc, cell, x, y, z, c);
  return {c[0], c[1], c[2]};
}

// acc after an octave of amplitude amp, in the exact form
__device__ __forceinline__ float fractal_x(int fractal, float amp, float n, float acc) {
  return fractal == UPF_FRACTAL_NONE ? n
         : (fractal == UPF_FRACTAL_RIDGED ? mad_x<true>(amp, mad_x<true>(-2.0f, fabsf(n), 1.0f), acc)
                                          : mad_x<true>(amp, n, acc));
}

// One gradient or value layer at this lane's R nodes (x, y, z[r]).
template <int NOISE, int R>
__device__ __forceinline__ void tile_lattice(const TileCtx& c, const DLayer& L, float x, float y, const float* z,
                                             float* out) {
  constexpr bool GRAD = NOISE == UPF_NOISE_GRADIENT;
  static_assert((R & (R - 1)) == 0 && R * UPF_MAX_OCTAVES <= 64, "a lane per plane and octave");
  constexpr int kCap = GRAD ? kTLds : 4 * kTLds;
  const int oct = L.fractal == UPF_FRACTAL_NONE ? 1 : L.octaves;
  // the z part of plane r and octave k, in lane r + R k
  float zl = z[0], fl = L.freq[0];
#pragma unroll
  for (int r = 1; r < R; r++)
    if ((c.lane & (R - 1)) == r) zl = z[r];
#pragma unroll
  for (int k = 1; k < UPF_MAX_OCTAVES; k++)
    if (k < oct && c.lane / R == k) fl = L.freq[k];
  const float qz = zl * fl, fz = floorf(qz), tzl = qz - fz, uzl = fade<true>(tzl);
  const int izl = (int)fz;
  const auto plane = [&](float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
#pragma unroll
  for (int r = 0; r < R; r++) out[r] = 0.0f;
  for (int k = 0; k < oct; k++) {
    const float f = L.freq[k], amp = L.amp[k];
    const uint32_t seed = L.seed + (uint32_t)k;
    const float qx = x * f, qy = y * f;
    const float fx = floorf(qx), fy = floorf(qy);
    const int ix = (int)fx, iy = (int)fy;
    const TileBox b = tile_box(ix, iy, __builtin_amdgcn_readlane(izl, R * k), __builtin_amdgcn_readlane(izl, R * k + R - 1),
                               2, kCap);
    if (!b.fits) {
#pragma unroll
      for (int r = 0; r < R; r++) {
        const float n = GRAD ? lane_gradient(seed, qx, qy, z[r] * f) : lane_value(seed, qx, qy, z[r] * f);
        out[r] = fractal_x(L.fractal, amp, n, out[r]);
      }
      continue;
    }
    const uint32_t hx = (uint32_t)b.x * kPX, hy = (uint32_t)b.y * kPY, hz = (uint32_t)b.z * kPZ;
    tile_fill(c.lane, b, [&](int e, int i, int j, int kk) {
      const uint32_t h = (seed ^ (hx + (uint32_t)i * kPX) ^ (hy + (uint32_t)j * kPY) ^ (hz + (uint32_t)kk * kPZ)) * kHM;
      if (GRAD) c.lds[e] = c.gtab[h >> 28];
      else reinterpret_cast<float*>(c.lds)[e] = lattice_value(h);
    });
    const float tx = qx - fx, ty = qy - fy;
    const float ux = fade<true>(tx), uy = fade<true>(ty);
    const float sx = tx - 1.0f, sy = ty - 1.0f;
    const int o = (ix - b.x) + b.nx * (iy - b.y), nxy = b.nx * b.ny;
    float za = 0.0f, zb = 0.0f;  // value: the x and y sums below and above
    float p[8], gz[8];           // gradient: the corners' x and y parts and z components
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int iz = __builtin_amdgcn_readlane(izl, R * k + r);
      const float uz = plane(uzl, R * k + r);
      const bool fresh = r == 0 || iz != __builtin_amdgcn_readlane(izl, R * k + (r ? r - 1 : 0));
      float n;
      if (GRAD) {
        if (fresh) {
          const float4* g = c.lds + o + nxy * (iz - b.z);
#pragma unroll
          for (int q = 0; q < 8; q++) {
            const float4 v = g[(q & 1) + ((q & 2) ? b.nx : 0) + ((q & 4) ? nxy : 0)];
            p[q] = fmaf(v.y, (q & 2) ? sy : ty, v.x * ((q & 1) ? sx : tx));
            gz[q] = v.z;
          }
        }
        const float tz = plane(tzl, R * k + r), sz = tz - 1.0f;
        float d[8];
#pragma unroll
        for (int q = 0; q < 8; q++) d[q] = fmaf(gz[q], (q & 4) ? sz : tz, p[q]);
        const float x00 = lerpf<true>(d[0], d[1], ux), x10 = lerpf<true>(d[2], d[3], ux);
        const float x01 = lerpf<true>(d[4], d[5], ux), x11 = lerpf<true>(d[6], d[7], ux);
        n = lerpf<true>(lerpf<true>(x00, x10, uy), lerpf<true>(x01, x11, uy), uz);
      } else {
        if (fresh) {
          const float* v = reinterpret_cast<const float*>(c.lds) + o + nxy * (iz - b.z);
          const float x00 = lerpf<true>(v[0], v[1], ux), x10 = lerpf<true>(v[b.nx], v[b.nx + 1], ux);
          v += nxy;
          const float x01 = lerpf<true>(v[0], v[1], ux), x11 = lerpf<true>(v[b.nx], v[b.nx + 1], ux);
          za = lerpf<true>(x00, x10, uy);
          zb = lerpf<true>(x01, x11, uy);
        }
        n = lerpf<true>(za, zb, uz);
      }
      out[r] = fractal_x(L.fractal, amp, n, out[r]);
    }
  }
}

// noise_simplex with the gradients in LDS; a corner out of reach adds 0.
__device__ __forceinline__ float tile_simplex(const float4* gtab, uint32_t seed, float x, float y, float z) {
  SimplexCell s;
  simplex_cell(x, y, z, s);
  float n = 0.0f;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const float dx = s.d[q][0], dy = s.d[q][1], dz = s.d[q][2];
    const float t = 0.5f - (dx * dx + dy * dy + dz * dz);
    const float t2 = t * t;
    const float v = n + t2 * t2 * dot_g(gtab[simplex_hash(seed, s, q) >> 28], dx, dy, dz);
    n = t > 0.0f ? v : n;
  }
  return 72.0f * n;
}

// One layer at this lane's R nodes; at_lane: sampled at (px[r], py[r], pz[r]) instead (the
// legacy mode's and the craters' second layer), per lane.
template <int R>
__device__ __forceinline__ void tile_layer(const TileCtx& c, const DLayer& L, float x, float y, const float* z,
                                           bool at_lane, const Point3* at, float* out) {
  if (!at_lane && L.noise == UPF_NOISE_GRADIENT) {
    tile_lattice<UPF_NOISE_GRADIENT, R>(c, L, x, y, z, out);
    return;
  }
  if (!at_lane && L.noise == UPF_NOISE_VALUE) {
    tile_lattice<UPF_NOISE_VALUE, R>(c, L, x, y, z, out);
    return;
  }
  const int oct = L.fractal == UPF_FRACTAL_NONE ? 1 : L.octaves;
#pragma unroll
  for (int r = 0; r < R; r++) out[r] = 0.0f;
  for (int k = 0; k < oct; k++) {
    const float f = L.freq[k], amp = L.amp[k];
    const uint32_t seed = L.seed + (uint32_t)k;
#pragma unroll
    for (int r = 0; r < R; r++) {
      const float qx = (at_lane ? at[r].x : x) * f, qy = (at_lane ? at[r].y : y) * f, qz = (at_lane ? at[r].z : z[r]) * f;
      float n;
      if (L.noise == UPF_NOISE_SIMPLEX) n = tile_simplex(c.gtab, seed, qx, qy, qz);
      else if (L.noise == UPF_NOISE_VALUE) n = lane_value(seed, qx, qy, qz);
      else if (L.noise == UPF_NOISE_GRADIENT) n = lane_gradient(seed, qx, qy, qz);
      else n = lane_cellular(seed, qx, qy, qz, L.js, L.j0);
      out[r] = fractal_x(L.fractal, amp, n, out[r]);
    }
  }
}

// voronoi_nearest at this lane's R nodes: the points of the cells that the tile's lanes
// look at are made once, one cell per lane.
template <int R>
__device__ __forceinline__ void tile_voronoi(const TileCtx& c, uint32_t seed, int ppc, float cell, float px, float py,
                                             const float* pz, ModeState<float>* st) {
  const float freq = 1.0f / cell;
  const int32_t cx = cell_index(px * freq), cy = cell_index(py * freq);
  int32_t cz[R];
#pragma unroll
  for (int r = 0; r < R; r++) cz[r] = __builtin_amdgcn_readfirstlane(cell_index(pz[r] * freq));
  const TileBox b = tile_box(cx, cy, cz[0], cz[R - 1], 3, ppc > 0 ? kTLds / ppc : 0);
  if (!b.fits) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      const Point3 q = lane_voronoi(seed, ppc, cell, px, py, pz[r]);
      st[r].c[0] = q.x; st[r].c[1] = q.y; st[r].c[2] = q.z;
    }
    return;
  }
  const uint32_t h0 = fmix32(seed), h1 = fmix32(h0), h2 = fmix32(h1);
  tile_fill(c.lane, b, [&](int e, int i, int j, int k) {
    const int32_t kx = b.x - 1 + i, ky = b.y - 1 + j, kz = b.z - 1 + k;
    uint32_t s0 = (uint32_t)kx, s1 = (uint32_t)ky, s2 = (uint32_t)kz;
    for (int q = 0; q <= ppc; q++) {
      const uint32_t t0 = h0 + s0 + s1 + fmix32(s0);
      const uint32_t t1 = h1 + s1 + s2 + fmix32(s1);
      const uint32_t t2 = h2 + s2 + s0 + fmix32(s2);
      s0 = t0; s1 = t1; s2 = t2;
      if (q == 0) continue;
      c.lds[e * ppc + q - 1] = make_float4(((float)((int32_t)s0 % 65536) / 65535.0f + (float)kx) * cell,
                                           ((float)((int32_t)s1 % 65536) / 65535.0f + (float)ky) * cell,
                                           ((float)((int32_t)s2 % 65536) / 65535.0f + (float)kz) * cell, 0.0f);
    }
  });
#pragma unroll
  for (int r = 0; r < R; r++) {
    float best = __builtin_inff();
    st[r].c[0] = st[r].c[1] = st[r].c[2] = 0.0f;
    for (int dz = 0; dz < 3; dz++)
      for (int dy = 0; dy < 3; dy++) {
        const float4* q = c.lds + (size_t)(((cx - b.x) + b.nx * ((cy - b.y) + dy + b.ny * (cz[r] - b.z + dz))) * ppc);
        for (int i = 0; i < 3 * ppc; i++) {
          const float4 p = q[i];
          const float ex = p.x - px, ey = p.y - py, ez = p.z - pz[r];
          const float d2 = ex * ex + ey * ey + ez * ez;
          if (d2 < best) { best = d2; st[r].c[0] = p.x; st[r].c[1] = p.y; st[r].c[2] = p.z; }
        }
      }
  }
}

// elevation_eval<true, true> at this lane's R nodes, for the lakes and islands modes: the
// mountains' ridges and terraces come multiplied by masks of the second layer; where a
// mask is 0 for every node of the wave its layer is not evaluated (any finite value times
// 0 is the same 0), nor is any layer after the first where every node is flat.
template <int R>
__device__ __forceinline__ void tile_hills(const TileCtx& c, const DSpec& s, float x, float y, const float* z, float* out) {
  const int mode = s.mode;
  ModeState<float> st[R];
#pragma unroll
  for (int r = 0; r < R; r++) st[r].v1 = st[r].v2 = st[r].v3 = 0.0f;
  for (int l = 0; l < 4; l++) {
    if (l > 0) {
      bool need = false;
#pragma unroll
      for (int r = 0; r < R; r++) {
        const float mask = l == 1 ? 1.0f : (l == 2 ? mode_ridge_mask(st[r], 0.0f) : mode_terrace_mask(st[r], 0.0f));
        need = need || (!st[r].flat && mask * st[r].cover != 0.0f);
      }
      if (__ballot(need) == 0) continue;
    }
    float v[R];
    tile_layer<R>(c, s.L[l], x, y, z, false, nullptr, v);
#pragma unroll
    for (int r = 0; r < R; r++) (void)mode_after(mode, l, v[r], 0.0f, st[r]);
  }
#pragma unroll
  for (int r = 0; r < R; r++) out[r] = mode_finish(mode, st[r], x, y, z[r], 0.0f);
}

// elevation_eval<true, true> at this lane's R nodes, for the other modes and the layer
// stack.
template <int R>
__device__ __forceinline__ void tile_elevation(const TileCtx& c, const DSpec& s, float x, float y, const float* z,
                                               float* out) {
  const int mode = s.mode;
  const bool stack = mode == UPF_ELEV_LAYERS;
  ModeState<float> st[R];  // v0 and v1 hold the sum and the mask of the layer stack
#pragma unroll
  for (int r = 0; r < R; r++) st[r].v0 = st[r].v1 = 0.0f;
  if (mode == UPF_ELEV_CRATERS) tile_voronoi<R>(c, s.L[0].seed, s.L[0].octaves, s.L[0].freq[0], x, y, z, st);
  for (int l = mode == UPF_ELEV_CRATERS ? 1 : 0; l < s.n_layers; l++) {  // the craters' first: the Voronoi's parameters
    const DLayer& L = s.L[l];
    const bool at_lane = (mode == UPF_ELEV_LEGACY || mode == UPF_ELEV_CRATERS) && l == 1;
    Point3 at[R];
    float v[R];
#pragma unroll
    for (int r = 0; r < R; r++) mode_position(mode, l, st[r], x, y, z[r], 0.0f, at[r].x, at[r].y, at[r].z);
    tile_layer<R>(c, L, x, y, z, at_lane, at, v);
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (!stack) {
        if (l == 0) st[r].v0 = v[r];
        else st[r].v1 = v[r];
        continue;
      }
      const float w = L.weight * v[r];
      if (L.blend == UPF_BLEND_ADD) st[r].v0 = st[r].v0 + w;
      else if (L.blend == UPF_BLEND_MASK) st[r].v1 = __builtin_amdgcn_fmed3f(w + 0.5f, 0.0f, 1.0f);
      else st[r].v0 = mad_x<true>(st[r].v1, w - st[r].v0, st[r].v0);
    }
  }
#pragma unroll
  for (int r = 0; r < R; r++) out[r] = stack ? st[r].v0 : mode_finish(mode, st[r], x, y, z[r], 0.0f);
}

// field_eval<true> at this lane's R nodes.  PRIM: the shape is a primitive (the other
// shapes' code would set the kernel's registers).  HILLS: the lakes or islands mode.
template <int R, bool PRIM, bool HILLS>
__device__ __forceinline__ void tile_field(const TileCtx& c, const DSpec& s, float x, float y, const float* z,
                                           float* out) {
  const bool need_elev = s.compose == UPF_COMPOSE_LAND || s.compose == UPF_COMPOSE_NAVIGATION ||
                         s.compose == UPF_COMPOSE_ELEVATION_RAW;
  float elev[R];
#pragma unroll
  for (int r = 0; r < R; r++) elev[r] = 0.0f;
  if (need_elev && HILLS) tile_hills<R>(c, s, x, y, z, elev);
  if (need_elev && !HILLS) tile_elevation<R>(c, s, x, y, z, elev);
#pragma unroll
  for (int r = 0; r < R; r++) {
    const float shape = s.compose == UPF_COMPOSE_ELEVATION_RAW ? 0.0f : shape_eval<!PRIM, !PRIM, true>(s, x, y, z[r]);
    switch (s.compose) {
      case UPF_COMPOSE_LAND: out[r] = shape - s.escale * elev[r]; break;
      case UPF_COMPOSE_WATER: out[r] = shape; break;
      case UPF_COMPOSE_NAVIGATION: out[r] = shape - s.escale * fmaxf(elev[r], 0.0f); break;
      case UPF_COMPOSE_ELEVATION: out[r] = shape / s.escale; break;
      default: out[r] = elev[r]; break;
    }
  }
}

}  // namespace upf
