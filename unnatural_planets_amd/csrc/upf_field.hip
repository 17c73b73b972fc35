// upf_field.hip -- field evaluation kernels (forward and fused forward+adjoint) and
// their C-ABI entry points.
//
// Replaces the per-node callback the reference hands to cage's marching cubes,
// cubes->updateByPosition(Delegate<Real(const Vec3&)>(terrainSdfLand))
// (sources/meshGeneration.cpp:38), and the point-wise terrainSdf* calls
// (sources/coloringModes.cpp:51-57,122-151).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "upf_device_grad.hpp"
#include "upf_device_row.hpp"
#include "upf_device_row_grad.hpp"
#include "upf_device_tilex.hpp"
#include "upf_device_band.hpp"
#include "upf_device_band_grad.hpp"
#include "upf_internal.hpp"

namespace upf {

// One thread per node.  A workgroup covers 64 consecutive x nodes of 4 rows, so each
// wave writes 256 contiguous bytes.
constexpr int kGridBX = 64;
constexpr int kGridBY = 4;

// Optional fused output: the marching-cubes sign mask of the wave's 64-node group,
// bit = (node inside the row and f < iso), at S[(k * ny + j) * gpr + xb].
__device__ __forceinline__ void write_signs(uint64_t* __restrict__ S, const DGrid& g, int xb, int j, int k,
                                            bool valid, float v, float iso) {
  const uint64_t m = __ballot(valid && v < iso);
  if ((threadIdx.x & 63) == 0) S[((int64_t)k * g.n[1] + j) * ((g.n[0] + 63) / 64) + xb] = m;
}

// The EXT instantiation (elevation modes, further shapes) takes 108 VGPRs unconstrained
// (four waves per SIMD); at six waves (72 VGPRs, nothing spilled) the 512^3 lakes field
// went from 5.44 to 4.78 ms.
template <bool EXT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(EXT ? 6 : 8))) void k_eval_grid(const DSpec s, const DGrid g, float* __restrict__ out,
                                                   uint64_t* __restrict__ S, float iso) {
  const int i = blockIdx.x * kGridBX + threadIdx.x;
  const int j = blockIdx.y * kGridBY + threadIdx.y;
  const int k = blockIdx.z;
  if (j >= g.n[1]) return;  // whole waves
  const bool valid = i < g.n[0];
  const int ic = min(i, g.n[0] - 1);
  const float x = node_coord(g.o[0], g.s[0], ic);
  const float y = node_coord(g.o[1], g.s[1], j);
  const float z = node_coord(g.o[2], g.s[2], k);
  const float v = field_eval<EXT>(s, x, y, z);
  if (valid) out[((size_t)k * g.n[1] + j) * g.n[0] + i] = v;
  if (S) write_signs(S, g, blockIdx.x, j, k, valid, v, iso);
}

// Wave-cooperative rows (upf_device_row.hpp): each wave evaluates 64 x nodes of
// kRowsPerWave rows j .. j + kRowsPerWave - 1 of one plane (they share the lattice column
// spans and the x part of the interpolation); lanes past the end of the row stand in for
// the last node so that all 64 lanes take part in the shared lattice work, rows past the
// end of the plane repeat its last row, and only real nodes are stored.  A workgroup
// covers 64 x nodes of kRowWaves row groups.
// Two rows, the octaves unrolled (four rows spill).  Grids with rows to spare run in bands of
// eight, k_eval_grid_band: this form is for small ones, and decides per wave whether a layer
// fits LDS.
constexpr int kRowsPerWave = 2;
constexpr int kRowWaves = 4;
static_assert(kRowsPerWave <= kRowMaxRows, "the per-octave table holds kRowMaxRows rows");

// Seven waves per SIMD (at most 72 VGPRs): the kernel keeps the VALU busy ~93% of the
// time at five waves and the extra waves fill the issue slots the others leave.  On the
// 512^3 torus workload: five waves 1.80 ms, six 1.56 ms, seven 1.45 ms once the
// lane-derived values are recomputed at their use (lane_of; before, seven waves spilled
// 11 VGPRs to scratch, 2.5 GB of writes per launch), eight 1.69 ms (29 VGPRs spilled).
// The wave's LDS bases come from a scalar wave index and the node index is recomputed
// after the layers, so nothing is spilled.
template <bool COMPOSED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(7))) void k_eval_grid_row(
    const DSpec s, const DGrid g, float* __restrict__ out, uint64_t* __restrict__ S, float iso) {
  constexpr int R = kRowsPerWave;
  __shared__ float4 s_slice[kRowWaves][kRowSlice];
  __shared__ float4 s_gtab[16];
  __shared__ float4 s_oct[kRowWaves][kRowOctTab];
  if (threadIdx.y == 0 && threadIdx.x < 16) s_gtab[threadIdx.x] = gradient_entry(threadIdx.x);
  __syncthreads();
  const int lane = threadIdx.x;
  const int j = __builtin_amdgcn_readfirstlane((blockIdx.y * kRowWaves + threadIdx.y) * R);
  const int k = blockIdx.z;
  if (j >= g.n[1]) return;
  const int rows = min(R, g.n[1] - j);  // real rows of this wave
  const int ic = min((int)blockIdx.x * kGridBX + lane, g.n[0] - 1);
  const float x = node_coord(g.o[0], g.s[0], ic);
  float y[R];
#pragma unroll
  for (int r = 0; r < R; r++) y[r] = node_coord(g.o[1], g.s[1], j + min(r, rows - 1));
  const float z = node_coord(g.o[2], g.s[2], k);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.y);  // LDS bases in scalar registers
  const RowCtx c = make_row_ctx(s_slice[wv], s_gtab, s_oct[wv], lane);
  float v[R];
  row_field<R, COMPOSED>(c, s, x, y, z, v);
  const int i = (int)blockIdx.x * kGridBX + lane_of(c);  // recomputed: not live across the layers
  const bool valid = i < g.n[0];
  const size_t row0 = ((size_t)k * g.n[1] + j) * g.n[0];
#pragma unroll
  for (int r = 0; r < R; r++)
    if (r < rows && valid) out[row0 + (size_t)r * g.n[0] + i] = v[r];
  if (S) {
#pragma unroll
    for (int r = 0; r < R; r++)
      if (r < rows) write_signs(S, g, blockIdx.x, j + r, k, valid, v[r], iso);
  }
}

// Bands of R rows (upf_device_band.hpp), the same values as k_eval_grid_row.  512^3
// torus at 7 waves a SIMD 863 us, at 6 909, at 8 (64 registers, spills) 928.
template <int R, bool COMPOSED, bool WIDE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(7))) void k_eval_grid_band(
    const DSpec s, const DGrid g, float* __restrict__ out, uint64_t* __restrict__ S, float iso) {
  __shared__ float4 s_slice[kRowWaves][kRowSlice];
  __shared__ float4 s_gtab[16];
  if (threadIdx.y == 0 && threadIdx.x < 16) s_gtab[threadIdx.x] = gradient_entry(threadIdx.x);
  __syncthreads();
  const int lane = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int j = (blockIdx.y * kRowWaves + wv) * R;
  const int k = blockIdx.z;
  if (j >= g.n[1]) return;
  const int rows = min(R, g.n[1] - j);  // real rows of this wave
  const int ic = min((int)blockIdx.x * kGridBX + lane, g.n[0] - 1);
  const float x = node_coord(g.o[0], g.s[0], ic);
  const float yl = node_coord(g.o[1], g.s[1], j + min(lane & (R - 1), rows - 1));
  const float z = node_coord(g.o[2], g.s[2], k);
  const RowCtx c = make_row_ctx(s_slice[wv], s_gtab, nullptr, lane);
  float v[R];
  band_field<R, COMPOSED, WIDE>(c, s, x, yl, z, v);
  const int i = (int)blockIdx.x * kGridBX + lane_of(c);  // recomputed: not live across the layers
  const bool valid = i < g.n[0];
  const size_t row0 = ((size_t)k * g.n[1] + j) * g.n[0];
#pragma unroll
  for (int r = 0; r < R; r++)
    if (r < rows && valid) out[row0 + (size_t)r * g.n[0] + i] = v[r];
  if (S) {
#pragma unroll
    for (int r = 0; r < R; r++)
      if (r < rows) write_signs(S, g, blockIdx.x, j + r, k, valid, v[r], iso);
  }
}

// The elevation modes and the further shapes, in the exact form (upf_device_tilex.hpp): a
// workgroup covers 64 x nodes of kTY rows and kTZ planes, its four waves 16 nodes each.
// A wave's 16 bits of each row's sign word are stored by themselves.
//
// VALU-bound.  500^3 lakes field, VALU instructions per 64 nodes and time of the land mesh
// call: per lane 2,198, 5.75 ms; 64 x 2 nodes a wave with x columns 1,150, 3.77 ms; tiles of
// 16 x 4 x 2 1,000, 3.23 ms; of 16 x 4 x 4 867, 2.95 ms at six waves per SIMD and 2.87 ms at
// seven (72 VGPRs from 80; the few spilled are around the rare per-lane calls).
template <int R, bool PRIM, bool HILLS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(PRIM ? 7 : 4))) void k_eval_grid_tilex(const DSpec s, const DGrid g, float* __restrict__ out,
                                                         uint16_t* __restrict__ S, float iso) {
  __shared__ float4 s_lds[4][kTLds];
  __shared__ float4 s_gtab[16];
  if (threadIdx.x < 16) s_gtab[threadIdx.x] = gradient_entry(threadIdx.x);
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i0 = blockIdx.x * 64 + wv * kTX, k0 = blockIdx.z * R;
  const int i = i0 + (lane & (kTX - 1)), j = blockIdx.y * kTY + lane / kTX;
  float v[R] = {};
  if (i0 < g.n[0]) {  // lanes past the end of a row or plane stand in for the last node
    const float x = node_coord(g.o[0], g.s[0], min(i, g.n[0] - 1));
    const float y = node_coord(g.o[1], g.s[1], min(j, g.n[1] - 1));
    float z[R];
#pragma unroll
    for (int r = 0; r < R; r++) z[r] = node_coord(g.o[2], g.s[2], min(k0 + r, g.n[2] - 1));
    const TileCtx c = {s_lds[wv], s_gtab, lane};
    tile_field<R, PRIM, HILLS>(c, s, x, y, z, v);
  }
  const bool valid = i < g.n[0] && j < g.n[1];
  const int gpr = (g.n[0] + 63) / 64;
#pragma unroll
  for (int r = 0; r < R; r++) {
    if (k0 + r >= g.n[2]) break;
    const int64_t row = (int64_t)(k0 + r) * g.n[1] + j;
    if (valid) out[row * g.n[0] + i] = v[r];
    if (S) {
      const uint64_t m = __ballot(valid && v[r] < iso);
      if ((lane & (kTX - 1)) == 0 && j < g.n[1])
        S[(row * gpr + blockIdx.x) * 4 + wv] = (uint16_t)(m >> lane);
    }
  }
}

template <bool EXT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(EXT ? 6 : 8))) void k_eval_points(const DSpec s, const float* __restrict__ xyz, int64_t n,
                                                     float* __restrict__ f) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  f[i] = field_eval<EXT>(s, xyz[3 * i], xyz[3 * i + 1], xyz[3 * i + 2]);
}

// Fused forward + adjoint over a grid-stride loop; every lane of a block runs the same
// number of iterations so the wave reductions inside ThetaAcc see all 64 lanes.
template <bool THETA, bool GRID, bool EXT>
__global__ __launch_bounds__(256) void k_adjoint(const DSpec s, const DGrid g, const float* __restrict__ xyz,
                                                 int64_t n, const float* __restrict__ dLdf, float* __restrict__ fout,
                                                 float* __restrict__ dfdx, float* __restrict__ dLdtheta) {
  __shared__ float th[4][UPF_THETA_COUNT];
  const int wave = threadIdx.x >> 6;
  if (THETA) {
    for (int t = threadIdx.x; t < 4 * UPF_THETA_COUNT; t += 256) (&th[0][0])[t] = 0.0f;
    __syncthreads();
  }
  ThetaAcc acc{th[wave]};
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t base = (int64_t)blockIdx.x * 256; base < n; base += stride) {
    const int64_t idx = base + threadIdx.x;
    const bool valid = idx < n;
    const int64_t i = valid ? idx : n - 1;
    float x, y, z;
    if (GRID) {
      const int64_t nxy = (int64_t)g.n[0] * g.n[1];
      const int kk = (int)(i / nxy);
      const int64_t r = i - (int64_t)kk * nxy;
      const int jj = (int)(r / g.n[0]);
      const int ii = (int)(r - (int64_t)jj * g.n[0]);
      x = node_coord(g.o[0], g.s[0], ii);
      y = node_coord(g.o[1], g.s[1], jj);
      z = node_coord(g.o[2], g.s[2], kk);
    } else {
      x = xyz[3 * i]; y = xyz[3 * i + 1]; z = xyz[3 * i + 2];
    }
    const float w = (THETA && valid) ? dLdf[i] : 0.0f;
    float gr[3];
    const float f = field_grad<THETA, EXT>(s, x, y, z, w, gr, acc);
    if (valid) {
      if (fout) fout[i] = f;
      if (dfdx) { dfdx[3 * i] = gr[0]; dfdx[3 * i + 1] = gr[1]; dfdx[3 * i + 2] = gr[2]; }
    }
  }
  if (THETA) {
    __syncthreads();
    for (int t = threadIdx.x; t < UPF_THETA_COUNT; t += 256) {
      const float v = th[0][t] + th[1][t] + th[2][t] + th[3][t];
      if (v != 0.0f) atomicAdd(dLdtheta + t, v);
    }
  }
}

// Fused forward + adjoint over a grid with wave-cooperative rows: persistent waves
// stride over 64-node row segments (so a block's θ partials are flushed once at the
// end); lanes past the end of a row stand in for its last node with dLdf = 0.  Six
// waves per SIMD (at most 80 VGPRs): on the 512^3 torus workload with dL/dtheta, 9.94 ms
// unconstrained (109 VGPRs), 8.48 ms at five waves, 7.80 ms at six once the lane-derived
// values are recomputed at their use (lane_of; the spills left are in the prologue of
// these persistent waves).
template <bool THETA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6))) void k_adjoint_rows(const DSpec s, const DGrid g, int64_t items,
                                                      const float* __restrict__ dLdf, float* __restrict__ fout,
                                                      float* __restrict__ dfdx, float* __restrict__ dLdtheta) {
  __shared__ float4 s_slice[4][kRowSlice];
  __shared__ float4 s_gtab[16];
  __shared__ float4 s_oct[4][kRowOctTab];
  __shared__ float th[4][UPF_THETA_COUNT];
  if (threadIdx.x < 16) s_gtab[threadIdx.x] = gradient_entry(threadIdx.x);
  if (THETA)
    for (int t = threadIdx.x; t < 4 * UPF_THETA_COUNT; t += 256) (&th[0][0])[t] = 0.0f;
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const RowCtx c = make_row_ctx(s_slice[wave], s_gtab, s_oct[wave], lane);
  ThetaAcc acc{th[wave]};
  const int gpr = (g.n[0] + 63) / 64;
  const int64_t stride = (int64_t)gridDim.x * 4;
  // item r = (k * ny + j) * gpr + xb, decomposed once; each step adds the stride's own
  // digits (sk, sj, sx) with carries instead of dividing r again
  int64_t r = (int64_t)blockIdx.x * 4 + wave;
  int xb = (int)(r % gpr), j = (int)((r / gpr) % g.n[1]), k = (int)(r / gpr / g.n[1]);
  const int sx = (int)(stride % gpr), sj = (int)((stride / gpr) % g.n[1]), sk = (int)(stride / gpr / g.n[1]);
  for (; r < items; r += stride) {
    // the row's first node (uniform) and this lane's 32-bit offset in it
    const int64_t row0 = ((int64_t)k * g.n[1] + j) * g.n[0];
    const int i = xb * 64 + lane;
    const bool valid = i < g.n[0];
    const int ic = min(i, g.n[0] - 1);
    const float x = node_coord(g.o[0], g.s[0], ic);
    const float y = node_coord(g.o[1], g.s[1], j);
    const float z = node_coord(g.o[2], g.s[2], k);
    const float w = (THETA && valid) ? dLdf[row0 + ic] : 0.0f;
    float gr[3];
    const float f = row_field_grad<THETA>(c, s, x, y, z, w, gr, acc);
    if (valid) {
      const int64_t node = row0 + ic;
      if (fout) fout[node] = f;
      if (dfdx) { dfdx[3 * node] = gr[0]; dfdx[3 * node + 1] = gr[1]; dfdx[3 * node + 2] = gr[2]; }
    }
    xb += sx;
    const int cx = xb >= gpr;
    xb -= cx ? gpr : 0;
    j += sj + cx;
    const int cj = j >= g.n[1];
    j -= cj ? g.n[1] : 0;
    k += sk + cj;
  }
  if (THETA) {
    __syncthreads();
    for (int t = threadIdx.x; t < UPF_THETA_COUNT; t += 256) {
      const float v = th[0][t] + th[1][t] + th[2][t] + th[3][t];
      if (v != 0.0f) atomicAdd(dLdtheta + t, v);
    }
  }
}

// The same over bands of kBandGradRows rows (upf_device_band_grad.hpp), for the specs that
// band_grad_fits accepts.  Sixteen waves a workgroup, one workgroup a CU: the sums meet
// dLdtheta in 256 float additions at most, whose rounding is most of a sum's error (256^3,
// relative: 5.0e-7 of the row kernel's 1,536 workgroups, 7.0e-7 of 1,280 with four waves at
// five a SIMD, 1.8e-7 so; that form ran 230 us against 243).
constexpr int kBandGradWaves = 16;

template <bool THETA, bool WIDE>
__global__ __launch_bounds__(64 * kBandGradWaves) __attribute__((amdgpu_waves_per_eu(4))) void k_adjoint_bands(const DSpec s, const DGrid g, int64_t items,
                                                      const float* __restrict__ dLdf, float* __restrict__ fout,
                                                      float* __restrict__ dfdx, float* __restrict__ dLdtheta) {
  constexpr int R = kBandGradRows;
  __shared__ float4 s_slice[kBandGradWaves][kRowSlice];
  __shared__ float4 s_gtab[16];
  __shared__ float th[kBandGradWaves][UPF_THETA_COUNT];
  if (threadIdx.x < 16) s_gtab[threadIdx.x] = gradient_entry(threadIdx.x);
  if (THETA)
    for (int t = threadIdx.x; t < kBandGradWaves * UPF_THETA_COUNT; t += 64 * kBandGradWaves) (&th[0][0])[t] = 0.0f;
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const RowCtx c = make_row_ctx(s_slice[wave], s_gtab, nullptr, threadIdx.x & 63);
  ThetaAcc acc{th[wave]};
  const int gpr = (g.n[0] + 63) / 64, bands = (g.n[1] + R - 1) / R;
  const int64_t stride = (int64_t)gridDim.x * kBandGradWaves;
  int64_t it = (int64_t)blockIdx.x * kBandGradWaves + wave;  // (k * bands + band) * gpr + xb, as k_adjoint_rows
  int xb = (int)(it % gpr), band = (int)((it / gpr) % bands), k = (int)(it / gpr / bands);
  const int sx = (int)(stride % gpr), sj = (int)((stride / gpr) % bands), sk = (int)(stride / gpr / bands);
  for (; it < items; it += stride) {
    const int lane = lane_of(c);
    const int j = band * R, rows = min(R, g.n[1] - j);
    const int64_t row0 = ((int64_t)k * g.n[1] + j) * g.n[0];
    const int i = xb * 64 + lane;
    const bool valid = i < g.n[0];
    const int ic = min(i, g.n[0] - 1);
    const float x = node_coord(g.o[0], g.s[0], ic);
    const float yl = node_coord(g.o[1], g.s[1], j + min(lane & (R - 1), rows - 1));
    const float z = node_coord(g.o[2], g.s[2], k);
    float w[R], f[R], gr[R][3];
#pragma unroll
    for (int r = 0; r < R; r++) w[r] = THETA && valid && r < rows ? dLdf[row0 + (int64_t)r * g.n[0] + ic] : 0.0f;
    band_field_grad<R, THETA, WIDE>(c, s, x, yl, z, w, f, gr, acc);
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int64_t node = row0 + (int64_t)r * g.n[0] + xb * 64 + lane_of(c);
      if (r < rows && xb * 64 + lane_of(c) < g.n[0]) {
        if (fout) fout[node] = f[r];
        if (dfdx) { dfdx[3 * node] = gr[r][0]; dfdx[3 * node + 1] = gr[r][1]; dfdx[3 * node + 2] = gr[r][2]; }
      }
    }
    xb += sx;
    const int cx = xb >= gpr;
    xb -= cx ? gpr : 0;
    band += sj + cx;
    const int cj = band >= bands;
    band -= cj ? bands : 0;
    k += sk + cj;
  }
  if (THETA) {
    __syncthreads();
    for (int t = threadIdx.x; t < UPF_THETA_COUNT; t += 64 * kBandGradWaves) {
      float v = 0.0f;
      for (int q = 0; q < kBandGradWaves; q++) v = v + th[q][t];
      if (v != 0.0f) atomicAdd(dLdtheta + t, v);
    }
  }
}

namespace {
int adjoint_blocks(int64_t n) {
  // enough workgroups to fill 256 CUs several times; capped so the per-block θ
  // flush stays a few hundred thousand atomics at most
  const int64_t want = (n + 255) / 256;
  return (int)(want < 4096 ? (want > 0 ? want : 1) : 4096);
}
}  // namespace

void lanes_launch(const DSpec& s, const DGrid& g, float* d_field, uint64_t* S, float iso, hipStream_t stream) {
  const dim3 blocks((g.n[0] + kGridBX - 1) / kGridBX, (g.n[1] + kGridBY - 1) / kGridBY, g.n[2]);
  const auto kernel = spec_ext(s) ? k_eval_grid<true> : k_eval_grid<false>;
  hipLaunchKernelGGL(kernel, blocks, dim3(kGridBX, kGridBY, 1), 0, stream, s, g, d_field, S, iso);
}

template <int R>
void tilex_launch(const DSpec& s, const DGrid& g, float* d_field, uint64_t* S, float iso, hipStream_t stream) {
  const dim3 blocks((g.n[0] + 63) / 64, (g.n[1] + kTY - 1) / kTY, (g.n[2] + R - 1) / R);
  const bool prim = s.shape < UPF_SHAPE_H3O && !spec_composed(s);
  const bool hills = s.mode == UPF_ELEV_LAKES || s.mode == UPF_ELEV_ISLANDS;
  const auto kernel = prim ? (hills ? k_eval_grid_tilex<R, true, true> : k_eval_grid_tilex<R, true, false>)
                           : (hills ? k_eval_grid_tilex<R, false, true> : k_eval_grid_tilex<R, false, false>);
  hipLaunchKernelGGL(kernel, blocks, dim3(256), 0, stream, s, g, d_field, reinterpret_cast<uint16_t*>(S), iso);
}

// The exact form's kernel.  From 2^21 nodes on (128^3) four planes a wave share its lattice work
// (400^3: lakes 2,805 us per lane, 1,185 in tiles; craters 11,142 and 1,523; legacy 1,483 and
// 1,043).  Below, four planes leave too few waves (48^3 lakes: 14.8 us per lane, 28 with four
// planes, 15.2 with one): one plane a wave, but per lane for the legacy mode and the layer
// stack, most of whose layers the tiles evaluate per lane anyway (110^3 legacy: 39.4 us per
// lane, 43.7 in one-plane tiles).
// What four planes save depends on the layers, and it has to pay for the nodes that a tile's
// 4 rows and 4 planes stand for beyond the grid (`py` and `pz` times the grid's).  Microseconds
// per lane / one plane / four, for 2048 x 2048 nodes of 2 planes, then for 2048 x 2 x 2048:
//   masked (lakes, islands) or shared (craters) work: lakes 327 / 227 / 322, 363 / 468 / 327
//     (3 planes 488 / 336 / 322); craters 1,308 / 232 / 371
//   gradient and value layers alone: 5 octaves on the gear 183 / 160 / 210, 207 / 315 / 212 (5
//     planes 450 / 393 / 412)
//   these among others: legacy 157 / 184 / 252, 180 / 364 / 253 (5 planes 382 / 452 / 492, 5 rows
//     423 / 722 / 494); 11 octaves of all kinds 484 / 535 / 906, 636 / 1,061 / 909 (9
//     rows at 1024 567 / 797 / 687; 700 x 5 x 700 167 / - / 234, but 1024 x 5 x 1024 482 / 534 /
//     461)
//   none: simple 181 / 165 / 308, 209 / 325 / 310 (5 planes 444 / 404 / 607, 5 rows 477 / 645 /
//     607); cells on the gear 372 / 365 / 714, 452 / 722 / 717 (at 1024 9 rows 441 / 546 /
//     541); these from 2^16 tiles of a plane on, 2^22 nodes (mandelbulb 128^3 332 / 293 / 387,
//     256^3 2,013 / 1,908 / 2,126; simple 128^3 50 / 45 / 49, 200^3 225 / 201 / 195; 2 x 1024 x
//     1024 1,463 / 580 / 512).
constexpr int64_t kTileNodes = (int64_t)1 << 21, kLaneTiles = (int64_t)1 << 16;

// Octaves of the layers read whose lattices a tile's planes share, and the others.
void tile_octaves(const DSpec& s, int* shared, int* other) {
  *shared = *other = 0;
  for (int l = 0; reads_layers(s) && l < s.n_layers; l++) {
    const DLayer& L = s.L[l];
    const bool lattice = (L.noise == UPF_NOISE_GRADIENT || L.noise == UPF_NOISE_VALUE) && !(s.mode == UPF_ELEV_LEGACY && l == 1);
    (lattice ? *shared : *other) += L.fractal == UPF_FRACTAL_NONE ? 1 : L.octaves;
  }
}

// Whether every layer is certain to be finite, and its powers: the tiles of the lakes and
// islands modes leave out layers whose mask is 0, which an infinite one would turn into NaN.
bool layers_finite(const DSpec& s, const DGrid& g) {
  double reach = 0.0;
  for (int a = 0; a < 3; a++) reach = std::max(reach, std::fabs((double)g.o[a]) + (double)g.s[a] * g.n[a]);
  for (int l = 0; l < s.n_layers; l++) {
    const DLayer& L = s.L[l];
    const double noise = L.noise == UPF_NOISE_CELLULAR ? 1.0 + std::fabs((double)L.jitter) : 1.0;
    double amps = 1.0;
    for (int k = 0; k < (L.fractal == UPF_FRACTAL_NONE ? 1 : L.octaves); k++) {
      if (std::fabs((double)L.freq[k]) * reach > 0x1p30) return false;
      amps += std::fabs((double)L.amp[k]);
    }
    if (noise * amps > 0x1p40) return false;
  }
  return true;
}

void exact_launch(const DSpec& s, const DGrid& g, float* d_field, uint64_t* S, float iso, hipStream_t stream) {
  const bool hills = reads_layers(s) && (s.mode == UPF_ELEV_LAKES || s.mode == UPF_ELEV_ISLANDS);
  if (hills && !layers_finite(s, g)) {
    lanes_launch(s, g, d_field, S, iso, stream);
    return;
  }
  const bool craters = reads_layers(s) && s.mode == UPF_ELEV_CRATERS, stack = s.mode == UPF_ELEV_LAYERS;
  int shared, other;
  tile_octaves(s, &shared, &other);
  const auto padded = [](int n) { return (double)((n + 3) / 4 * 4) / n; };
  const double py = padded(g.n[1]), pz = padded(g.n[2]);
  const bool lattices = shared && !other;
  const bool rows_fit = hills || craters || py <= (stack ? (lattices ? 1.7 : 1.15) : 1.5);
  const bool planes_fit = pz <= (hills || craters || lattices ? 1.7 : 1.15);
  const int64_t nodes = (int64_t)g.n[0] * g.n[1] * g.n[2];
  const int64_t tiles = (int64_t)((g.n[0] + kTX - 1) / kTX) * ((g.n[1] + kTY - 1) / kTY) * g.n[2];  // of a plane each
  if (rows_fit && planes_fit && nodes >= kTileNodes && (hills || craters || shared || tiles >= kLaneTiles)) {
    tilex_launch<4>(s, g, d_field, S, iso, stream);
  } else if (!craters && (g.n[1] == 2 || (nodes >= kTileNodes && !rows_fit) ||
                          ((stack || s.mode == UPF_ELEV_LEGACY) && (shared || nodes < kTileNodes)))) {
    lanes_launch(s, g, d_field, S, iso, stream);
  } else {
    tilex_launch<1>(s, g, d_field, S, iso, stream);
  }
}

// The rows of a band by the number of bands: eight from 8,192 on (a little more than the
// machine's 7,168 waves of seven a SIMD), four below, two rows (k_eval_grid_row) where even
// those are few.  5 octaves on a torus, eight / four: 128^3 (4,096 bands of eight) 16.2 / 15.7
// us, 144^3 22.3 / 22.1, 160^3 (9,600) 24.7 / 25.0, 256^3 55 / 63; four / two: 64^3 (1,024 of
// four) 10.3 / 10.0, 72^3 10.6 / 11.8, 127^3 14.8 / 19.7.  Layers of band_cellular_wide in bands
// of four only, which hold its distances without spilling (4 octaves of cells at 400^3 1,592 /
// 1,211 us, a torus with one such layer at 310^3 225 / 231).
// And by the rows of a plane, whose last band stands for rows that are not there and whose
// workgroup, of four bands, for bands that are not: 512 x 60,000 nodes in planes of 3 to
// 13 rows, the same octaves, eight / four / two: 4 rows - / 238 / 251, 5 rows 258 / 228 / 233, 9
// rows 177 / 155 / 305, 12 rows 135 / 119 / 232, 13 rows 125 / 132 / 213 (64 x 5 x 20000 nodes
// with more than 64 columns an octave 137 / 116 / 108); the shape alone: 3 rows - / 85 / 81, 6
// rows 72 / 52 / 49, 7 rows 63 / 45 / 49.
constexpr int64_t kBandGridItems = 8192;
constexpr int kBandGridRows = 13;
constexpr int kHalfBandRows = 4;
constexpr int64_t kHalfBandItems = 2048;

bool half_band_rows(const DSpec& s, const DGrid& g) {
  const int rows = g.n[1];
  if (rows >= kBandGridRows) return true;
  return (rows > 6 || (reads_layers(s) && rows > 2 && rows <= kHalfBandRows)) && !band_far(s, g);
}

template <int R>
void band_launch(const DSpec& s, const DGrid& g, bool wide, float* d_field, uint64_t* S, float iso, hipStream_t stream) {
  const dim3 blocks((g.n[0] + kGridBX - 1) / kGridBX, (g.n[1] + R * kRowWaves - 1) / (R * kRowWaves), g.n[2]);
  constexpr bool W = R == kHalfBandRows;
  const auto kernel = W && wide ? (spec_composed(s) ? k_eval_grid_band<R, true, W> : k_eval_grid_band<R, false, W>)
                                : (spec_composed(s) ? k_eval_grid_band<R, true, false> : k_eval_grid_band<R, false, false>);
  hipLaunchKernelGGL(kernel, blocks, dim3(kGridBX, kRowWaves, 1), 0, stream, s, g, d_field, S, iso);
}

int field_grid_launch(const DSpec& s, const DGrid& g, float* d_field, int variant, uint64_t* S, float iso,
                      hipStream_t stream) {
  if (variant < 0 || variant > UPF_EVAL_PER_LANE) return UPF_ERR_BAD_SPEC;
  if (variant == UPF_EVAL_PER_LANE) {
    lanes_launch(s, g, d_field, S, iso, stream);
  } else if (spec_ext(s)) {  // the row form covers the layer stack and the common shapes
    exact_launch(s, g, d_field, S, iso, stream);
  } else if (band_items(g) >= kBandGridItems && g.n[1] >= kBandGridRows && band_fits(s, g) && !band_wide(s, g, kRowSlice2) && !band_far(s, g)) {
    band_launch<kBandRows>(s, g, false, d_field, S, iso, stream);
  } else if (band_items(g, kHalfBandRows) >= kHalfBandItems && half_band_rows(s, g) && band_fits(s, g)) {
    band_launch<kHalfBandRows>(s, g, band_wide(s, g, kRowSlice2), d_field, S, iso, stream);
  } else {
    constexpr int rows_per_block = kRowsPerWave * kRowWaves;
    const dim3 rblocks((g.n[0] + kGridBX - 1) / kGridBX, (g.n[1] + rows_per_block - 1) / rows_per_block, g.n[2]);
    if (spec_composed(s))
      hipLaunchKernelGGL(k_eval_grid_row<true>, rblocks, dim3(kGridBX, kRowWaves, 1), 0, stream, s, g, d_field, S, iso);
    else
      hipLaunchKernelGGL(k_eval_grid_row<false>, rblocks, dim3(kGridBX, kRowWaves, 1), 0, stream, s, g, d_field, S, iso);
  }
  UPF_LAUNCH_CHECK();
  return UPF_OK;
}

}  // namespace upf

using namespace upf;

extern "C" {

int upf_field_eval_grid_ex(const upf_field_spec* spec, const upf_grid* grid, float* d_field,
                           const upf_eval_opts* opts, void* stream) {
  if (!d_field) return UPF_ERR_NULL;
  DSpec s;
  DGrid g;
  int st = to_device(spec, &s);
  if (st) return st;
  if ((st = to_device(grid, &g))) return st;
  return field_grid_launch(s, g, d_field, opts ? opts->variant : UPF_EVAL_AUTO, nullptr, 0.0f, as_stream(stream));
}

int upf_field_eval_grid(const upf_field_spec* spec, const upf_grid* grid, float* d_field, void* stream) {
  return upf_field_eval_grid_ex(spec, grid, d_field, nullptr, stream);
}

int upf_field_eval_points(const upf_field_spec* spec, const float* d_xyz, int64_t n, float* d_f, float* d_dfdx,
                          void* stream) {
  if (n < 0) return UPF_ERR_BAD_GRID;
  if (n == 0) return UPF_OK;
  if (!d_xyz || !d_f) return UPF_ERR_NULL;
  DSpec s;
  const int st = to_device(spec, &s);
  if (st) return st;
  if (d_dfdx) return upf_field_adjoint(spec, d_xyz, n, nullptr, d_f, d_dfdx, nullptr, stream);
  const dim3 pb((unsigned)((n + 255) / 256));
  if (spec_ext(s))
    hipLaunchKernelGGL(k_eval_points<true>, pb, dim3(256), 0, as_stream(stream), s, d_xyz, n, d_f);
  else
    hipLaunchKernelGGL(k_eval_points<false>, pb, dim3(256), 0, as_stream(stream), s, d_xyz, n, d_f);
  UPF_LAUNCH_CHECK();
  return UPF_OK;
}

int upf_field_adjoint(const upf_field_spec* spec, const float* d_xyz, int64_t n, const float* d_dLdf, float* d_f,
                      float* d_dfdx, float* d_dLdtheta, void* stream) {
  if (n < 0) return UPF_ERR_BAD_GRID;
  if (n == 0) return UPF_OK;
  if (!d_xyz) return UPF_ERR_NULL;
  if (d_dLdtheta && !d_dLdf) return UPF_ERR_NULL;
  DSpec s;
  const int st = to_device(spec, &s);
  if (st) return st;
  if (d_dLdtheta && s.mode != UPF_ELEV_LAYERS) return UPF_ERR_BAD_SPEC;
  DGrid g{};
  const int nb = adjoint_blocks(n);
  const dim3 gb(nb), tb(256);
  hipStream_t hs = as_stream(stream);
  const bool ext = spec_ext(s);
  if (d_dLdtheta && ext)
    hipLaunchKernelGGL((k_adjoint<true, false, true>), gb, tb, 0, hs, s, g, d_xyz, n, d_dLdf, d_f, d_dfdx, d_dLdtheta);
  else if (d_dLdtheta)
    hipLaunchKernelGGL((k_adjoint<true, false, false>), gb, tb, 0, hs, s, g, d_xyz, n, d_dLdf, d_f, d_dfdx, d_dLdtheta);
  else if (ext)
    hipLaunchKernelGGL((k_adjoint<false, false, true>), gb, tb, 0, hs, s, g, d_xyz, n, d_dLdf, d_f, d_dfdx, d_dLdtheta);
  else
    hipLaunchKernelGGL((k_adjoint<false, false, false>), gb, tb, 0, hs, s, g, d_xyz, n, d_dLdf, d_f, d_dfdx, d_dLdtheta);
  UPF_LAUNCH_CHECK();
  return UPF_OK;
}

int upf_field_adjoint_grid(const upf_field_spec* spec, const upf_grid* grid, const float* d_dLdf, float* d_f,
                           float* d_dfdx, float* d_dLdtheta, void* stream) {
  if (d_dLdtheta && !d_dLdf) return UPF_ERR_NULL;
  DSpec s;
  DGrid g;
  int st = to_device(spec, &s);
  if (st) return st;
  if ((st = to_device(grid, &g))) return st;
  if (s.mode != UPF_ELEV_LAYERS) return UPF_ERR_BAD_SPEC;  // the parameter adjoint covers the layer stack
  if (spec_ext(s)) {  // a further shape: per lane over the nodes
    const int64_t n = (int64_t)g.n[0] * g.n[1] * g.n[2];
    const dim3 gb(adjoint_blocks(n)), tb(256);
    hipStream_t hs = as_stream(stream);
    if (d_dLdtheta)
      hipLaunchKernelGGL((k_adjoint<true, true, true>), gb, tb, 0, hs, s, g, nullptr, n, d_dLdf, d_f, d_dfdx,
                         d_dLdtheta);
    else
      hipLaunchKernelGGL((k_adjoint<false, true, true>), gb, tb, 0, hs, s, g, nullptr, n, d_dLdf, d_f, d_dfdx,
                         d_dLdtheta);
    UPF_LAUNCH_CHECK();
    return UPF_OK;
  }
  const bool bands = band_grad_items(g) >= kBandItems && band_grad_fits(s, g);
  const int64_t items = bands ? band_grad_items(g) : (int64_t)((g.n[0] + 63) / 64) * g.n[1] * g.n[2];
  const bool wide = bands && band_wide(s, g, kRowSlice);
  auto kernel = d_dLdtheta ? k_adjoint_rows<true> : k_adjoint_rows<false>;
  if (wide) kernel = d_dLdtheta ? k_adjoint_bands<true, true> : k_adjoint_bands<false, true>;
  else if (bands) kernel = d_dLdtheta ? k_adjoint_bands<true, false> : k_adjoint_bands<false, false>;
  const int waves = bands ? kBandGradWaves : 4;
  const int nb = (int)std::min<int64_t>((items + waves - 1) / waves,
                                        (int64_t)resident_blocks(reinterpret_cast<const void*>(kernel), 64 * waves));
  hipLaunchKernelGGL(kernel, dim3(nb), dim3(64 * waves), 0, as_stream(stream), s, g, items, d_dLdf, d_f, d_dfdx, d_dLdtheta);
  UPF_LAUNCH_CHECK();
  return UPF_OK;
}

}  // extern "C"
