// upf_nb.hip -- narrow-band marching cubes: coarse pass over block corners, fine
// evaluation and meshing of the active blocks only.
//
// The reference sweeps the dense grid (sources/meshGeneration.cpp:35-39); a planet's
// surface touches a few percent of the cells of a 1024^3 grid, so this path evaluates the
// field at the block corners first (every 8th node per axis, 1/512 of the nodes), keeps
// the blocks whose corners come within `band` of the iso value or straddle it, and
// evaluates and meshes only those.
//
//  coarse    one thread per block corner;
//  activity  one thread per block: a count word with the active bit; the shared scan
//            compacts the active blocks, and a dense map block -> active rank follows;
//  fine      one workgroup per active block: its 9^3 brick of fine nodes, and from the signs
//            of its 81 rows of 9 nodes, as bit masks, the crossing edges that each row owns
//            (a node owns its +x/+y/+z edges; nodes on the block's upper faces belong to the
//            next block except on the grid's upper boundary), their exclusive prefix and the
//            block's vertex and triangle counts.  A brick that the surface crosses goes to HBM
//            with a record per row; one of a single sign (two of three in a band that is
//            sure to hold the surface) leaves its zero count alone;
//  scan      vertex and triangle bases per active block, and the list of crossed blocks;
//  emit      a workgroup per crossed block at a time: its vertices and triangles listed in LDS,
//            then a thread per vertex (base + prefix + rank) and per triangle corner, whose
//            edge id comes from the owning row's record (this block's, or a neighbour's
//            through the dense map);
//  normals   one thread per vertex: the normalized analytic gradient at the vertex.
// Vertex positions use the same interpolation as the dense path on the same per-lane
// node values, so the mesh equals the dense one up to order when the band holds the
// surface.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "upf_device_grad.hpp"
#include "upf_device_row.hpp"
#include "upf_internal.hpp"
#include "upf_mc.hpp"

namespace upf {

#include "upf_mc_device.hpp"

constexpr int kB = UPF_NB_BLOCK;          // cells per block edge
constexpr int kBN = kB + 1;               // nodes per brick edge
constexpr int kBrick = kBN * kBN * kBN;   // 729 nodes
constexpr int kRows = kBN * kBN;          // 81 rows (j + 9 k) of 9 nodes
constexpr int kCells = kB * kB * kB;      // 512 cells
constexpr int kNbThreads = 256;
static_assert(kCells == 2 * kNbThreads, "fine/emit give each thread two cells");
static_assert(kRows <= kNbThreads, "fine/emit give each row a thread");

// A brick row's record: x = owned vertices of the block before the row | X << 12 | M << 21,
// y = Y | Z << 9, with M the nodes inside, X / Y / Z the nodes whose +x / +y / +z edge
// crosses (within the brick, owned or not).
struct BrickRow {
  uint32_t m, x, y, z;
};

// Row t's masks, from the rows' M.
__device__ __forceinline__ BrickRow brick_row_masks(const uint32_t* s_row, int t) {
  BrickRow r;
  r.m = s_row[t];
  r.x = (r.m ^ (r.m >> 1)) & 0xFFu;
  r.y = t % kBN < kB ? r.m ^ s_row[t + 1] : 0u;
  r.z = t < kB * kBN ? r.m ^ s_row[t + kBN] : 0u;
  return r;
}

// The nodes of row t that the block owns.
__device__ __forceinline__ uint32_t owned_nodes(int t, bool lx, bool ly, bool lz) {
  return (t % kBN < kB || ly) && (t < kB * kBN || lz) ? (lx ? 0x1FFu : 0xFFu) : 0u;
}

// The block's vertex of node i's edge along axis, from its (owned) row's record.
__device__ __forceinline__ uint32_t row_vertex(uint2 rec, int i, int axis) {
  const uint32_t below = (1u << i) - 1u;
  const uint32_t rank = ((rec.x >> (12 + i)) & (uint32_t)(axis > 0)) + ((rec.y >> i) & (uint32_t)(axis > 1));
  return (rec.x & 0xFFFu) + (uint32_t)__popc(rec.x & (below << 12)) + (uint32_t)__popc(rec.y & (below | below << 9)) + rank;
}

// Case code of the cell at the rows' masks shifted to its first node: rows (j, k),
// (j + 1, k), (j, k + 1), (j + 1, k + 1).
__device__ __forceinline__ int cell_code(uint32_t m00, uint32_t m10, uint32_t m01, uint32_t m11) {
  const auto swap = [](uint32_t m) { return ((m & 1u) << 1) | ((m >> 1) & 1u); };
  return (int)((m00 & 3u) | swap(m10) << 2 | (m01 & 3u) << 4 | swap(m11) << 6);
}

struct NbDims {
  int bx, by, bz;  // blocks per axis
  int pad;
  int64_t blocks;
};

__device__ __forceinline__ void block_coords(const NbDims& d, uint32_t b, int& bx, int& by, int& bz) {
  bx = (int)(b % (uint32_t)d.bx);
  const uint32_t r = b / (uint32_t)d.bx;
  by = (int)(r % (uint32_t)d.by);
  bz = (int)(r / (uint32_t)d.by);
}

// Workgroup-wide exclusive sum of one int per thread; *total gets the sum.
__device__ __forceinline__ int wg_exclusive_sum(int v, int* total) {
  __shared__ int s_w[kNbThreads / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int inc = wave_inclusive_sum(v);
  if (lane == 63) s_w[wave] = inc;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kNbThreads / 64; w++) {
    if (w < wave) before += s_w[w];
    all += s_w[w];
  }
  __syncthreads();
  *total = all;
  return before + inc - v;
}

template <bool EXT>
__global__ __launch_bounds__(256) void k_nb_coarse(const DSpec s, const DGrid g, const NbDims d,
                                                   float* __restrict__ coarse) {
  __shared__ float4 s_gtab[16];
  if (threadIdx.x < 16) s_gtab[threadIdx.x] = gradient_entry(threadIdx.x);
  __syncthreads();
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int cx = d.bx + 1, cy = d.by + 1;
  const int64_t n = (int64_t)cx * cy * (d.bz + 1);
  if (c >= n) return;
  const int I = (int)(c % cx);
  const int64_t r = c / cx;
  const int J = (int)(r % cy), K = (int)(r / cy);
  coarse[c] = field_eval<EXT>(s, node_coord(g.o[0], g.s[0], I * kB), node_coord(g.o[1], g.s[1], J * kB),
                              node_coord(g.o[2], g.s[2], K * kB), GradTable{s_gtab});
}

__global__ __launch_bounds__(256) void k_nb_activity(const float* __restrict__ coarse, const NbDims d, float iso,
                                                     float band, uint32_t* __restrict__ counts) {
  const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (b >= d.blocks) return;
  int bx, by, bz;
  block_coords(d, (uint32_t)b, bx, by, bz);
  const int cx = d.bx + 1;
  const int64_t cxy = (int64_t)cx * (d.by + 1);
  const int64_t c0 = (int64_t)bz * cxy + (int64_t)by * cx + bx;
  const float v[8] = {coarse[c0], coarse[c0 + 1], coarse[c0 + cx], coarse[c0 + cx + 1],
                      coarse[c0 + cxy], coarse[c0 + cxy + 1], coarse[c0 + cxy + cx], coarse[c0 + cxy + cx + 1]};
  int inside = 0;
  bool near = false;
#pragma unroll
  for (int q = 0; q < 8; q++) {
    inside += v[q] < iso;
    near |= fabsf(v[q] - iso) < band;
  }
  const bool active = near || (inside != 0 && inside != 8);
  counts[b] = active ? (1u << 17) : 0u;  // the kScanMc active bit
}

__global__ void k_nb_fill_i32(int32_t* __restrict__ p, int64_t n, int32_t v) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = v;
}

// The dense map, and in place of each active block's index its coordinates (z, x | y << 16):
// decoded once here instead of by two integer divisions (40 vector instructions) per wave.
__global__ void k_nb_map(uint2* __restrict__ act, int64_t nact, const NbDims d, int32_t* __restrict__ map) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= nact) return;
  const uint32_t b = act[r].x;
  map[b] = (int32_t)r;
  int bx, by, bz;
  block_coords(d, b, bx, by, bz);
  act[r] = make_uint2((uint32_t)bz, (uint32_t)bx | (uint32_t)by << 16);
}

template <bool EXT, bool COMPOSED = true>
__global__ __launch_bounds__(kNbThreads) void k_nb_fine(const DSpec s, const DGrid g, const NbDims d, float iso,
                                                        const uint2* __restrict__ act,
                                                        const int32_t* __restrict__ map, float* __restrict__ bricks,
                                                        uint2* __restrict__ recs, uint32_t* __restrict__ bcounts,
                                                        uint32_t* __restrict__ unresolved) {
  __shared__ float s_fe[EXT ? kBrick : 1];
  __shared__ float4 s_slice[4][EXT ? 1 : kRowSlice];
  __shared__ float4 s_gtab[16];
  __shared__ float2 s_yz[EXT ? 1 : 4 * kBrickRows * kBrickGroups];
  __shared__ uint64_t s_bits[EXT ? 1 : 4 * kBrickGroups];  // signs of the groups of rows
  __shared__ uint32_t s_row[kRows];                        // and of each row
  __shared__ int s_crossed;
  __shared__ uint8_t s_ntris[256];  // triangles per case code
  s_ntris[threadIdx.x] = upf_mc_ntris[threadIdx.x];  // read after the barriers below
  if (threadIdx.x == 0) s_crossed = 0;
  const int64_t a = blockIdx.x;
  const uint2 at = act[a];
  const int bx = (int)(at.y & 0xFFFFu), by = (int)(at.y >> 16), bz = (int)at.x;
  const int64_t b = ((int64_t)bz * d.by + by) * d.bx + bx;
  const int gi0 = bx * kB, gj0 = by * kB, gk0 = bz * kB;
  const bool lx = bx == d.bx - 1, ly = by == d.by - 1, lz = bz == d.bz - 1;
  float* __restrict__ brick = bricks + a * kBrick;
  float v[kBrickGroups];  // this lane's nodes (rows)
  const int t = threadIdx.x;
  uint32_t mask = 0;  // thread t < kRows: row t's nodes inside
  bool first;         // whether node 0 is
  if (EXT) {  // elevation modes and further shapes: per node
    for (int n = threadIdx.x; n < kBrick; n += kNbThreads) {
      const int k = n / (kBN * kBN), r = n - k * kBN * kBN;
      const int j = r / kBN, i = r - j * kBN;
      s_fe[n] = field_eval<EXT>(s, node_coord(g.o[0], g.s[0], gi0 + i), node_coord(g.o[1], g.s[1], gj0 + j),
                                node_coord(g.o[2], g.s[2], gk0 + k));
    }
    __syncthreads();
    if (t < kRows)
      for (int i = 0; i < kBN; i++) mask |= (uint32_t)(s_fe[t * kBN + i] < iso) << i;
    first = s_fe[0] < iso;
  } else {
    // the brick's 81 rows of 9 nodes (row = j + 9 k) in 12 groups of kBrickRows; wave w
    // takes groups w, w + 4, w + 8 (kBrickGroups of them), its row rho = 7 m + r being
    // brick row 7 (w + 4 m) + r (the 3 rows past 80 repeat row 80 and are not stored);
    // lane 7 * 9 = 63 stands in for node 8 of row 6
    static_assert(kBrickRows * kBrickGroups * 4 >= kBN * kBN, "four waves cover the brick's rows");
    if (threadIdx.x < 16) s_gtab[threadIdx.x] = gradient_entry(threadIdx.x);
    // the rows' coordinates, once a brick: the divisions by 9 took 50 of 877 vector
    // instructions a wave
    if (t < kBrickRows * kBrickGroups * 4) {
      const int row = min(t, kRows - 1), k = row / kBN, j = row - k * kBN;
      s_yz[t] = make_float2(node_coord(g.o[1], g.s[1], gj0 + j), node_coord(g.o[2], g.s[2], gk0 + k));
    }
    __syncthreads();
    const int wave = uniform((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const RowCtx ctx = make_row_ctx(s_slice[wave], s_gtab, nullptr, lane);
    const bool node_lane = lane < kBrickRows * kBN;
    const int rl = node_lane ? lane / kBN : kBrickRows - 1;
    const int i = node_lane ? lane - rl * kBN : kBN - 1;
    const float x = node_coord(g.o[0], g.s[0], gi0 + i);
    auto yz = [&](int rho, float& yy, float& zz) {  // row rho = 7 m + r of the wave's: 7 (wave + 4 m) + r of the brick
      const float2 c = s_yz[kBrickRows * wave + rho + 3 * kBrickRows * (rho / kBrickRows)];
      yy = c.x;
      zz = c.y;
    };
    float y[kBrickGroups], z[kBrickGroups];
#pragma unroll
    for (int m = 0; m < kBrickGroups; m++) yz(kBrickRows * m + rl, y[m], z[m]);
    brick_field<kBrickGroups, COMPOSED>(ctx, s, rl, yz, x, y, z, v);
#pragma unroll
    for (int m = 0; m < kBrickGroups; m++) {
      const bool real = node_lane && kBrickRows * (wave + 4 * m) + rl < kRows;
      const uint64_t w = ballot64(real && v[m] < iso);
      if (lane == 0) s_bits[wave + 4 * m] = w;
    }
    __syncthreads();
    if (t < kRows) mask = (uint32_t)(s_bits[t / kBrickRows] >> (kBN * (t % kBrickRows))) & 0x1FFu;
    first = s_bits[0] & 1u;
  }
  if (t < kRows) {
    s_row[t] = mask;
    if (mask != (first ? 0x1FFu : 0u)) s_crossed = 1;
  }
  __syncthreads();
  if (!s_crossed) {
    if (t == 0) bcounts[a] = 0;
    return;
  }
  if (EXT) {
    for (int n = t; n < kBrick; n += kNbThreads) brick[n] = s_fe[n];
  } else {
    const int wave = t >> 6, lane = t & 63;
#pragma unroll
    for (int m = 0; m < kBrickGroups; m++) {
      const int n = kBrickRows * kBN * (wave + 4 * m) + lane;
      if (lane < kBrickRows * kBN && n < kBrick) brick[n] = v[m];
    }
  }

  // thread t < 81: row t's crossing edges; all: cells 2t, 2t + 1
  BrickRow r{0, 0, 0, 0};
  uint32_t own = 0;
  if (t < kRows) {
    r = brick_row_masks(s_row, t);
    own = owned_nodes(t, lx, ly, lz);
    if (const uint32_t rest = (r.x | r.y | r.z) & ~own) {  // crossings of other blocks' nodes
      const int oy = t % kBN == kB && !ly, oz = t >= kB * kBN && !lz;
      const int64_t nb = b + (int64_t)oy * d.bx + (int64_t)oz * d.bx * d.by;
      const uint32_t last = lx ? 0u : rest & 0x100u, here = rest & ~last;
      if (here && map[nb] < 0) atomicAdd(unresolved, (uint32_t)__popc(here));
      if (last && map[nb + 1] < 0) atomicAdd(unresolved, 1u);
    }
  }
  const int cr = (t >> 5) * kBN + ((t >> 2) & 7), ci = 2 * (t & 3);
  const uint32_t m00 = s_row[cr] >> ci, m10 = s_row[cr + 1] >> ci;
  const uint32_t m01 = s_row[cr + kBN] >> ci, m11 = s_row[cr + kBN + 1] >> ci;
  const int nt = s_ntris[cell_code(m00, m10, m01, m11)] + s_ntris[cell_code(m00 >> 1, m10 >> 1, m01 >> 1, m11 >> 1)];
  const int nv = __popc(r.x & own) + __popc(r.y & own) + __popc(r.z & own);
  int total;  // both counts in one sum: at most 2187 vertices, 2560 triangles
  const uint32_t pre = (uint32_t)wg_exclusive_sum(nv | nt << 16, &total) & 0xFFFFu;
  if (t < kRows) recs[a * kRows + t] = make_uint2(pre | r.x << 12 | r.m << 21, r.y | r.z << 9);
  if (t == 0) bcounts[a] = (uint32_t)(total & 0xFFFF) | ((uint32_t)(total >> 16) << 12) | (1u << 24);
}

// list: the crossed blocks (active rank, first triangle), total->z of them; a workgroup
// takes every gridDim.x-th.  Bound by vector instructions; with the lists a lane has a vertex
// or a corner at a time, where a thread per three nodes and two cells left most of a wave idle.
// 1025^3 rounded cube (129,032 active blocks, a third crossed): 384 -> 120 us (143 at seven
// waves a SIMD: a block is a chain of dependent reads; one workgroup per block 25 us more,
// 2048 in all 35 us more).
__global__ __launch_bounds__(kNbThreads) __attribute__((amdgpu_waves_per_eu(8))) void k_nb_emit(const DGrid g, const NbDims d, float iso,
                                                        const uint2* __restrict__ act, const int32_t* __restrict__ map,
                                                        const float* __restrict__ bricks, const uint2* __restrict__ recs,
                                                        const uint32_t* __restrict__ bcounts,
                                                        const uint32_t* __restrict__ voff,
                                                        const uint2* __restrict__ list, const uint4* __restrict__ total,
                                                        float* __restrict__ pos, uint32_t* __restrict__ idx,
                                                        uint64_t* __restrict__ keys, int64_t cap_v, int64_t cap_t) {
  __shared__ float s_f[kBrick];
  __shared__ uint2 s_rec[kRows];
  __shared__ uint32_t s_row[kRows];
  // the block's vertices (node << 2 | axis), then its triangles (cell | triangle << 9 | code << 12)
  __shared__ uint32_t s_list[UPF_MC_MAX_TRIS * kCells];
  static_assert(3 * kBrick <= 2 * UPF_MC_MAX_TRIS * kCells, "a block's vertices fit the list");
  uint16_t* s_vert = reinterpret_cast<uint16_t*>(s_list);
  __shared__ uint8_t s_ntris[256];         // triangles per case code
  __shared__ uint4 s_tris[256];            // and their edges (c_tris16)
  __shared__ int32_t s_nrow[8];            // upper neighbour (dx | dy << 1 | dz << 2): its active row, -1: none, -2: not crossed
  __shared__ uint32_t s_nvoff[8];          // and its first vertex id
  static_assert(kNbThreads == 256, "one case code per thread");
  const int t = threadIdx.x;
  s_ntris[t] = upf_mc_ntris[t];
  s_tris[t] = *reinterpret_cast<const uint4*>(&c_tris16.v[t][0]);
  const uint8_t* tris = reinterpret_cast<const uint8_t*>(s_tris);
  const int64_t n_list = (int64_t)total->z;
  for (int64_t q = blockIdx.x; q < n_list; q += gridDim.x) {
    const int64_t a = (int64_t)uniform((int)list[q].x);
    const uint2 where = act[a];
    const int bx = (int)(where.y & 0xFFFFu), by = (int)(where.y >> 16), bz = (int)where.x;
    const int64_t b = ((int64_t)bz * d.by + by) * d.bx + bx;
    const bool lx = bx == d.bx - 1, ly = by == d.by - 1, lz = bz == d.bz - 1;
    const uint32_t vb = voff[a];
    const int nv = (int)(bcounts[a] & 0xFFFu);
    __syncthreads();  // the last block's lists are read
    // threads 1..7 look up the upper neighbours that own the vertices of the brick's upper
    // faces, published after the vertices' part
    const bool there = t >= 1 && t < 8 && !((t & 1) && lx) && !((t & 2) && ly) && !((t & 4) && lz);
    const int32_t row = there ? map[b + (t & 1) + (int64_t)((t >> 1) & 1) * d.bx + (int64_t)(t >> 2) * d.bx * d.by] : -1;
    for (int n = t; n < kBrick; n += kNbThreads) s_f[n] = bricks[a * kBrick + n];
    if (t < kRows) {  // the row's owned crossings, node after node
      const uint2 rec = recs[a * kRows + t];
      s_rec[t] = rec;
      s_row[t] = (rec.x >> 21) & 0x1FFu;
      const uint32_t own = owned_nodes(t, lx, ly, lz);
      const uint32_t x = (rec.x >> 12) & own, y = rec.y & own, z = (rec.y >> 9) & own;
      uint16_t* at = s_vert + (rec.x & 0xFFFu);
      for (uint32_t left = x | y | z; left; left &= left - 1u) {
        const int i = __ffs(left) - 1;
        const int node = 4 * (kBN * t + i);
        if ((x >> i) & 1u) *at++ = (uint16_t)node;
        if ((y >> i) & 1u) *at++ = (uint16_t)(node + 1);
        if ((z >> i) & 1u) *at++ = (uint16_t)(node + 2);
      }
    }
    __syncthreads();

    // ---- vertices (normals follow in k_nb_normals)
    for (int e = t; e < nv; e += kNbThreads) {
      const int n = s_vert[e] >> 2, ax = s_vert[e] & 3;
      const int k = n / kRows, j = (n - k * kRows) / kBN, i = n - k * kRows - j * kBN;
      const int gi[3] = {bx * kB + i, by * kB + j, bz * kB + k};
      const float p0[3] = {node_coord(g.o[0], g.s[0], gi[0]), node_coord(g.o[1], g.s[1], gi[1]),
                           node_coord(g.o[2], g.s[2], gi[2])};
      const float f0 = s_f[n], f1 = s_f[n + (ax == 0 ? 1 : (ax == 1 ? kBN : kRows))];
      const float u = (iso - f0) / (f1 - f0);
      const uint32_t vid = vb + (uint32_t)e;
      if ((int64_t)vid < cap_v) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
          const float p1 = node_coord(g.o[c], g.s[c], gi[c] + 1);
          pos[3 * (size_t)vid + c] = ax == c ? p0[c] + u * (p1 - p0[c]) : p0[c];
        }
        if (keys) {
          const int64_t node = ((int64_t)gi[2] * g.n[1] + gi[1]) * g.n[0] + gi[0];
          keys[vid] = (uint64_t)node * 3u + (uint64_t)ax;
        }
      }
    }

    // a neighbour of one sign owns none of the vertices (its record would count none)
    if (t >= 1 && t < 8) {
      s_nrow[t] = row >= 0 && bcounts[row] == 0 ? -2 : row;
      s_nvoff[t] = row >= 0 ? voff[row] : 0u;
    }

    // ---- triangles of cells 2t, 2t + 1 into the list (the sum's barriers end the vertices' part)
    const int cr = (t >> 5) * kBN + ((t >> 2) & 7), ci = 2 * (t & 3);
    const uint32_t m00 = s_row[cr] >> ci, m10 = s_row[cr + 1] >> ci;
    const uint32_t m01 = s_row[cr + kBN] >> ci, m11 = s_row[cr + kBN + 1] >> ci;
    const int code[2] = {cell_code(m00, m10, m01, m11), cell_code(m00 >> 1, m10 >> 1, m01 >> 1, m11 >> 1)};
    const int nt[2] = {s_ntris[code[0]], s_ntris[code[1]]};
    int ntot;
    int at = wg_exclusive_sum(nt[0] + nt[1], &ntot);
#pragma unroll
    for (int h = 0; h < 2; h++)
      for (int tr = 0; tr < nt[h]; tr++) s_list[at++] = (uint32_t)(2 * t + h) | (uint32_t)tr << 9 | (uint32_t)code[h] << 12;
    __syncthreads();

    // ---- their corners
    const int64_t first = (int64_t)list[q].y;
    for (int c = t; c < 3 * ntot; c += kNbThreads) {
      const int tri = c / 3;
      const uint32_t entry = s_list[tri];
      const int cell = (int)(entry & 511u);
      const int e = tris[(entry >> 12) * 16 + 3 * ((entry >> 9) & 7u) + (uint32_t)(c - 3 * tri)] & 15;  // 0..11
      const int own = (int)((kEdgeOwner >> (5 * e)) & 31u);
      const int li = (cell & 7) + (own & 1), lj = ((cell >> 3) & 7) + ((own >> 1) & 1), lk = (cell >> 6) + ((own >> 2) & 1);
      const int axis = own >> 3;
      const int ox = (li == kB && !lx), oy = (lj == kB && !ly), oz = (lk == kB && !lz);
      const int o = ox | (oy << 1) | (oz << 2);
      uint32_t id;
      if (!o) {
        id = vb + row_vertex(s_rec[lk * kBN + lj], li, axis);
      } else {
        const int32_t rnb = s_nrow[o];
        const uint2 rec = rnb >= 0 ? recs[(int64_t)rnb * kRows + (lk - kB * oz) * kBN + (lj - kB * oy)] : make_uint2(0, 0);
        id = rnb == -1 ? 0xFFFFFFFFu : s_nvoff[o] + row_vertex(rec, li - kB * ox, axis);
      }
      if (first + tri < cap_t) idx[3 * (size_t)first + c] = id;
    }
  }
}

// Normals: the normalized analytic gradient at each vertex, one thread per vertex (few
// nodes of a brick own a vertex, so evaluating the gradient inside k_nb_emit would run
// the whole gradient for mostly idle lanes).
template <bool EXT>
__global__ __launch_bounds__(256) void k_nb_normals(const DSpec s, const float* __restrict__ pos, int64_t n,
                                                    float* __restrict__ nrm) {
  __shared__ float4 s_gtab[16];
  if (threadIdx.x < 16) s_gtab[threadIdx.x] = gradient_entry(threadIdx.x);
  __syncthreads();
  const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (v >= n) return;
  ThetaAcc none{nullptr};
  float gr[3];
  (void)field_grad<false, EXT>(s, pos[3 * v], pos[3 * v + 1], pos[3 * v + 2], 0.0f, gr, none, GradTable{s_gtab});
  const float len = __builtin_sqrtf(gr[0] * gr[0] + gr[1] * gr[1] + gr[2] * gr[2]);
  const float inv = len > 0.0f ? 1.0f / len : 0.0f;
  nrm[3 * v + 0] = gr[0] * inv;
  nrm[3 * v + 1] = gr[1] * inv;
  nrm[3 * v + 2] = gr[2] * inv;
}

// ------------------------------------------------------------------ host side
struct NbLayout {
  NbDims d;
  int64_t coarse, max_active;
  size_t off_coarse, off_counts, off_tiles, off_total_a, off_act, off_map, off_bricks, off_recs, off_list,
      off_bcounts, off_voff, off_total_b, bytes;
};

inline size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

NbLayout nb_layout(const NbDims& d, int64_t max_active) {
  NbLayout L;
  L.d = d;
  L.coarse = (int64_t)(d.bx + 1) * (d.by + 1) * (d.bz + 1);
  L.max_active = max_active;
  const int64_t tiles = mc_scan_tiles(std::max<int64_t>(d.blocks, std::max<int64_t>(max_active, 1)));
  size_t o = 0;
  L.off_coarse = o; o = al256(o + 4 * (size_t)L.coarse);
  L.off_counts = o; o = al256(o + 4 * (size_t)d.blocks);
  L.off_tiles = o; o = al256(o + sizeof(uint4) * (size_t)tiles);
  L.off_total_a = o; o = al256(o + sizeof(uint4));
  L.off_act = o; o = al256(o + sizeof(uint2) * (size_t)d.blocks);
  L.off_map = o; o = al256(o + 4 * (size_t)d.blocks);
  L.off_bricks = o; o = al256(o + 4 * (size_t)kBrick * max_active);
  // the blocks' records, then their list, in the room of a two-byte table of a brick's nodes;
  // and a spare word per block: workspaces keep the sizes that callers have been given
  static_assert(sizeof(uint2) * (kRows + 1) <= 2 * (size_t)kBrick, "records and list fit");
  L.off_recs = o;
  L.off_list = o + sizeof(uint2) * (size_t)kRows * max_active;
  o = al256(o + 2 * (size_t)kBrick * max_active);
  L.off_bcounts = o; o = al256(o + 4 * (size_t)max_active);
  L.off_voff = o; o = al256(o + 4 * (size_t)max_active);
  o = al256(o + 4 * (size_t)max_active);
  L.off_total_b = o; o = al256(o + 2 * sizeof(uint4));  // totals + unresolved counter
  L.bytes = o;
  return L;
}

int nb_dims(const DGrid& g, NbDims* d) {
  for (int a = 0; a < 3; a++)
    if ((g.n[a] - 1) % kB) return UPF_ERR_BAD_GRID;
  d->bx = (g.n[0] - 1) / kB;
  d->by = (g.n[1] - 1) / kB;
  d->bz = (g.n[2] - 1) / kB;
  d->pad = 0;
  d->blocks = (int64_t)d->bx * d->by * d->bz;
  if (d->blocks >= ((int64_t)1 << 31)) return UPF_ERR_BAD_GRID;
  return UPF_OK;
}

// The workspace of a call: its layout for the largest active-block capacity it holds.
struct NbWs {
  int64_t cap;
  float* coarse;
  uint32_t* counts;
  uint4 *tiles, *total_a;
  uint2* act;
  int32_t* map;
  float* bricks;
  uint2 *recs, *list;
  uint32_t *bcounts, *voff;
  uint4* total_b;
  int64_t n_coarse;
};

int nb_workspace(const NbDims& d, void* d_ws, size_t ws_bytes, NbWs* o) {
  const NbLayout L0 = nb_layout(d, 0);
  if (!d_ws || ws_bytes < L0.bytes) return UPF_ERR_WORKSPACE;
  const size_t per = 6 * (size_t)kBrick + 12;
  int64_t cap = std::min<int64_t>(d.blocks, (int64_t)((ws_bytes - L0.bytes) / per));
  while (cap > 0 && nb_layout(d, cap).bytes > ws_bytes) cap--;
  const NbLayout L = nb_layout(d, cap);
  char* w = static_cast<char*>(d_ws);
  o->cap = cap;
  o->n_coarse = L.coarse;
  o->coarse = reinterpret_cast<float*>(w + L.off_coarse);
  o->counts = reinterpret_cast<uint32_t*>(w + L.off_counts);
  o->tiles = reinterpret_cast<uint4*>(w + L.off_tiles);
  o->total_a = reinterpret_cast<uint4*>(w + L.off_total_a);
  o->act = reinterpret_cast<uint2*>(w + L.off_act);
  o->map = reinterpret_cast<int32_t*>(w + L.off_map);
  o->bricks = reinterpret_cast<float*>(w + L.off_bricks);
  o->recs = reinterpret_cast<uint2*>(w + L.off_recs);
  o->list = reinterpret_cast<uint2*>(w + L.off_list);
  o->bcounts = reinterpret_cast<uint32_t*>(w + L.off_bcounts);
  o->voff = reinterpret_cast<uint32_t*>(w + L.off_voff);
  o->total_b = reinterpret_cast<uint4*>(w + L.off_total_b);
  return UPF_OK;
}

// The mesh from the workspace's evaluated blocks (nact of them, out->n_* their counts).
int nb_emit(const DSpec& s, const DGrid& g, const NbDims& d, const NbWs& W, float iso, int64_t nact,
            upf_mesh_buffers* out, uint64_t* d_keys, hipStream_t hs) {
  if (out->n_vertices > out->cap_vertices || out->n_triangles > out->cap_triangles) return UPF_ERR_CAPACITY;
  if (out->n_vertices == 0 && out->n_triangles == 0) return UPF_OK;
  if (!out->positions || !out->indices) return UPF_ERR_NULL;
  // the crossed blocks' number stays on the device: as many workgroups as four rounds of the
  // machine's, or as there are blocks
  hipLaunchKernelGGL(k_nb_emit, dim3((unsigned)std::min<int64_t>(nact, 8192)), dim3(kNbThreads), 0, hs, g, d, iso,
                     W.act, W.map, W.bricks, W.recs, W.bcounts, W.voff, W.list, W.total_b, out->positions, out->indices,
                     d_keys, out->cap_vertices, out->cap_triangles);
  if (out->normals && out->n_vertices) {
    const dim3 blocks((unsigned)((out->n_vertices + 255) / 256));
    const auto kernel = spec_ext(s) ? k_nb_normals<true> : k_nb_normals<false>;
    hipLaunchKernelGGL(kernel, blocks, dim3(256), 0, hs, s, out->positions, out->n_vertices, out->normals);
  }
  UPF_LAUNCH_CHECK();
  return UPF_OK;
}

}  // namespace upf

using namespace upf;

extern "C" {

size_t upf_nb_workspace_bytes(const upf_grid* grid, int64_t max_active) {
  DGrid g;
  NbDims d;
  if (to_device(grid, &g) || nb_dims(g, &d) || max_active < 0) return 0;
  return nb_layout(d, std::min<int64_t>(max_active, d.blocks)).bytes;
}

int upf_nb_extract(const upf_field_spec* spec, const upf_grid* grid, float iso, float band, upf_mesh_buffers* out,
                   uint64_t* d_keys, void* d_ws, size_t ws_bytes, upf_nb_stats* stats, void* stream) {
  if (!out || !stats) return UPF_ERR_NULL;
  if (!std::isfinite(iso) || !std::isfinite(band) || band < 0.0f) return UPF_ERR_INVALID_VALUE;
  DSpec s;
  DGrid g;
  NbDims d;
  int st = to_device(spec, &s);
  if (st || (st = to_device(grid, &g)) || (st = nb_dims(g, &d))) return st;
  *stats = upf_nb_stats{};
  stats->blocks = d.blocks;
  NbWs W;
  if ((st = nb_workspace(d, d_ws, ws_bytes, &W))) return st;
  hipStream_t hs = as_stream(stream);

  const auto nblk = [](int64_t n) { return dim3((unsigned)((n + 255) / 256)); };
  const bool modes = spec_ext(s);
  if (modes) hipLaunchKernelGGL(k_nb_coarse<true>, nblk(W.n_coarse), dim3(256), 0, hs, s, g, d, W.coarse);
  else hipLaunchKernelGGL(k_nb_coarse<false>, nblk(W.n_coarse), dim3(256), 0, hs, s, g, d, W.coarse);
  hipLaunchKernelGGL(k_nb_activity, nblk(d.blocks), dim3(256), 0, hs, W.coarse, d, iso, band, W.counts);
  UPF_LAUNCH_CHECK();
  if ((st = mc_scan_launch(W.counts, d.blocks, W.tiles, W.total_a, nullptr, W.act, nullptr, hs, kScanMc))) return st;
  hipLaunchKernelGGL(k_nb_fill_i32, nblk(d.blocks), dim3(256), 0, hs, W.map, d.blocks, -1);
  hipLaunchKernelGGL(k_nb_fill_i32, dim3(1), dim3(256), 0, hs, reinterpret_cast<int32_t*>(W.total_b), (int64_t)8, 0);
  UPF_LAUNCH_CHECK();
  uint4 ha;
  UPF_HIP_CHECK(hipMemcpyAsync(&ha, W.total_a, sizeof(uint4), hipMemcpyDeviceToHost, hs));
  UPF_HIP_CHECK(hipStreamSynchronize(hs));
  const int64_t nact = ha.z;
  stats->active_blocks = nact;
  if (nact > W.cap) return UPF_ERR_WORKSPACE;
  out->n_vertices = out->n_triangles = 0;
  if (nact == 0) return UPF_OK;

  hipLaunchKernelGGL(k_nb_map, nblk(nact), dim3(256), 0, hs, W.act, nact, d, W.map);
  const auto fine = modes ? k_nb_fine<true> : (spec_composed(s) ? k_nb_fine<false, true> : k_nb_fine<false, false>);
  hipLaunchKernelGGL(fine, dim3((unsigned)nact), dim3(kNbThreads), 0, hs, s, g, d, iso, W.act, W.map, W.bricks, W.recs,
                     W.bcounts, reinterpret_cast<uint32_t*>(W.total_b + 1));
  UPF_LAUNCH_CHECK();
  if ((st = mc_scan_launch(W.bcounts, nact, W.tiles, W.total_b, W.voff, W.list, nullptr, hs, kScanBlocks))) return st;
  uint4 hb[2];
  UPF_HIP_CHECK(hipMemcpyAsync(hb, W.total_b, 2 * sizeof(uint4), hipMemcpyDeviceToHost, hs));
  UPF_HIP_CHECK(hipStreamSynchronize(hs));
  stats->n_vertices = hb[0].x;
  stats->n_triangles = hb[0].y;
  stats->unresolved = hb[1].x;
  out->n_vertices = hb[0].x;
  out->n_triangles = hb[0].y;
  if (stats->unresolved) return UPF_ERR_BAND;
  return nb_emit(s, g, d, W, iso, nact, out, d_keys, hs);
}

int upf_nb_emit(const upf_field_spec* spec, const upf_grid* grid, float iso, upf_mesh_buffers* out, uint64_t* d_keys,
                void* d_ws, size_t ws_bytes, const upf_nb_stats* stats, void* stream) {
  if (!out || !stats) return UPF_ERR_NULL;
  if (!std::isfinite(iso)) return UPF_ERR_INVALID_VALUE;
  DSpec s;
  DGrid g;
  NbDims d;
  int st = to_device(spec, &s);
  if (st || (st = to_device(grid, &g)) || (st = nb_dims(g, &d))) return st;
  NbWs W;
  if ((st = nb_workspace(d, d_ws, ws_bytes, &W))) return st;
  if (stats->active_blocks < 0 || stats->active_blocks > W.cap) return UPF_ERR_WORKSPACE;
  if (stats->unresolved) return UPF_ERR_BAND;
  // counts that no extraction gives: a mesh of no blocks, or more than its blocks' edges and cells
  if (stats->n_vertices < 0 || stats->n_vertices > 3 * kBrick * stats->active_blocks || stats->n_triangles < 0 ||
      stats->n_triangles > UPF_MC_MAX_TRIS * kCells * stats->active_blocks)
    return UPF_ERR_INVALID_VALUE;
  out->n_vertices = stats->n_vertices;
  out->n_triangles = stats->n_triangles;
  return nb_emit(s, g, d, W, iso, stats->active_blocks, out, d_keys, as_stream(stream));
}

}  // extern "C"
