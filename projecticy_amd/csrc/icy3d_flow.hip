// Flow kernels of the 3D step: D3Q7 AA phase collision and recovery, phase
// gradients with wall/ice mirrors, force densities, HOME central collision
// and pull streaming with moving-ice reflection.
//
// Storage is SoA planes with z fastest, so a wave64 of consecutive cells
// reads 256 contiguous bytes per plane.  Every kernel is one thread per
// cell; the hot bulk paths unroll all 27 (or 26) directions at compile time
// so that each c-product folds to an add or a negation.  The rare boundary
// paths (ice links, mirrors) live in separate kernels that exit early on
// bulk cells, which keeps register pressure of the hot kernels low.
#include <mutex>

#include "icy3d_device.h"

// Event pairs around each kernel group of the fused flow step.
struct icy3d_profile {
  hipEvent_t events[ICY3D_PROFILE_GROUPS + 1];
  double total_ms[ICY3D_PROFILE_GROUPS] = {};
  int64_t count = 0;
  int pending = 0;
};

namespace icy {

// ---------------------------------------------------------------------------
// Runtime-direction reconstruction, inlined where every lane of a boundary
// group uses it; reconstruct_rt is the same code out of line for the rare
// reflection path.
__device__ __forceinline__ float reconstruct_dyn(int q, const Moments& M) {
  const float fx = (float)cx(q), fy = (float)cy(q), fz = (float)cz(q);
  const float p = M.m[0], ux = M.m[1], uy = M.m[2], uz = M.m[3];
  const float sxx = M.m[4], syy = M.m[5], szz = M.m[6], sxy = M.m[7], sxz = M.m[8], syz = M.m[9];
  float cu = fx * ux + fy * uy + fz * uz;
  float csc = fx * fx * sxx + fy * fy * syy + fz * fz * szz + 2.0f * (fx * fy * sxy + fx * fz * sxz + fy * fz * syz);
  float value = p + 3.0f * cu + 4.5f * (csc - (sxx + syy + szz) * (1.0f / 3.0f));
  float ax = fx * fx - 1.0f / 3.0f, ay = fy * fy - 1.0f / 3.0f, az = fz * fz - 1.0f / 3.0f;
  float third = 0.0f;
  third += ax * fy * (sxx * uy + 2.0f * sxy * ux - 2.0f * ux * ux * uy);
  third += ax * fz * (sxx * uz + 2.0f * sxz * ux - 2.0f * ux * ux * uz);
  third += ay * fx * (syy * ux + 2.0f * sxy * uy - 2.0f * uy * uy * ux);
  third += ay * fz * (syy * uz + 2.0f * syz * uy - 2.0f * uy * uy * uz);
  third += az * fx * (szz * ux + 2.0f * sxz * uz - 2.0f * uz * uz * ux);
  third += az * fy * (szz * uy + 2.0f * syz * uz - 2.0f * uz * uz * uy);
  third += 2.0f * fx * fy * fz * (sxz * uy + syz * ux + sxy * uz - 2.0f * ux * uy * uz);
  return w27(q) * (value + 13.5f * third);
}
__device__ __noinline__ float reconstruct_rt(int q, const Moments& M) { return reconstruct_dyn(q, M); }

// ---------------------------------------------------------------------------
// AA addressing of D3Q7 (phase.py:69-82): plane offset of logical slot q.
// 32-bit offsets: a valid grid has fewer than INT32_MAX / 16 cells, so 7 N fits.
__device__ __forceinline__ int phase_addr(const icy3d_grid& g, const Cell& c, int q, int parity) {
  const int N = (int)cells(g);
  if (parity != 0 && q != 0) {
    int i = c.i - kC7[q][0], j = c.j - kC7[q][1], k = c.k - kC7[q][2];
    if (fluid_at(g, i, j, k)) return opp7(q) * N + lin(g, i, j, k);
  }
  return q * N + c.n;
}

// home.py:262-278
__device__ __forceinline__ int boundary_flag(const icy3d_grid& g, const Cell& c) {
  if (g.id[c.n] != -1) return -1;
  int flag = 0;
  for (int q = 0; q < 27; ++q) {
    if (q == 13) continue;
    int i = c.i - cx(q), j = c.j - cy(q), k = c.k - cz(q);
    if (!fluid_at(g, i, j, k)) {
      flag = max(flag, 1);
      if (inside(g, i, j, k)) {
        int id = g.id[lin(g, i, j, k)];
        if (id >= 0 || id == -3) flag = 2;
      }
    }
  }
  return flag;
}

struct Box {
  int lo[3], hi[3];
};
__device__ __forceinline__ bool box_cell(const icy3d_grid& g, const Box& b, int t, Cell& c) {
  int ex = b.hi[0] - b.lo[0], ey = b.hi[1] - b.lo[1], ez = b.hi[2] - b.lo[2];
  if (ex <= 0 || ey <= 0 || ez <= 0 || t >= ex * ey * ez) return false;
  c.k = b.lo[2] + t % ez;
  int r = t / ez;
  c.j = b.lo[1] + r % ey;
  c.i = b.lo[0] + r / ey;
  c.n = lin(g, c.i, c.j, c.k);
  return true;
}

__global__ void k_classify(icy3d_grid g, BoxList boxes) {
  Cell c;
  if (!list_cell(g, boxes, c)) return;
  g.flag[c.n] = (int8_t)boundary_flag(g, c);
}
// Compact the tank (flag 1) and ice (flag 2) cells into lists so that the
// boundary kernels launch over the boundary only.  Three passes (count per
// block, scan of block counts, scatter) give lists in cell order without a
// contended global counter.  Block counts live in the partials buffer.
constexpr int kCompactCells = 4096;  // cells per compaction block
constexpr int kCompactPerThread = kCompactCells / 256;  // 16 consecutive cells per thread
// Bit t of *tank / *ice: cell n0 + t has flag 1 / 2.
__device__ __forceinline__ void flag_bits(const icy3d_grid& g, int n0, int N, unsigned& tank, unsigned& ice) {
  int8_t f[kCompactPerThread];
  if (n0 + kCompactPerThread <= N && (reinterpret_cast<uintptr_t>(g.flag) & 15) == 0) {
    const int4 v = *reinterpret_cast<const int4*>(g.flag + n0);
    const int w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int t = 0; t < kCompactPerThread; ++t) f[t] = (int8_t)(w[t >> 2] >> (8 * (t & 3)));
  } else {
#pragma unroll
    for (int t = 0; t < kCompactPerThread; ++t) f[t] = n0 + t < N ? g.flag[n0 + t] : (int8_t)-1;
  }
  tank = 0u;
  ice = 0u;
#pragma unroll
  for (int t = 0; t < kCompactPerThread; ++t) {
    tank |= (f[t] == 1 ? 1u : 0u) << t;
    ice |= (f[t] == 2 ? 1u : 0u) << t;
  }
}
// Exclusive prefix sum over the block (blockDim.x a multiple of 64).
__device__ __forceinline__ int block_exclusive_scan(int v) {
  __shared__ int wave_total[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) wave_total[wave] = x;
  __syncthreads();
  int base = 0;
  for (int w = 0; w < wave; ++w) base += wave_total[w];
  return base + x - v;
}
__global__ void __launch_bounds__(256) k_count_flags(icy3d_grid g) {
  const int N = (int)cells(g);
  unsigned tank, ice;
  flag_bits(g, blockIdx.x * kCompactCells + threadIdx.x * kCompactPerThread, N, tank, ice);
  const int tanks = block_sum_int(__popc(tank));
  const int ices = block_sum_int(__popc(ice));
  int* counts = reinterpret_cast<int*>(g.partials);
  if (threadIdx.x == 0) {
    counts[2 * blockIdx.x] = tanks;
    counts[2 * blockIdx.x + 1] = ices;
  }
}
// One block of 1024 threads turns block counts into exclusive offsets.
__global__ void __launch_bounds__(1024) k_scan_flag_counts(icy3d_grid g, int blocks) {
  __shared__ int tank_sum[1024], ice_sum[1024];
  int* counts = reinterpret_cast<int*>(g.partials);
  const int per = (blocks + blockDim.x - 1) / blockDim.x;
  const int begin = threadIdx.x * per, end = min(blocks, begin + per);
  int tanks = 0, ices = 0;
  for (int b = begin; b < end; ++b) {
    tanks += counts[2 * b];
    ices += counts[2 * b + 1];
  }
  tank_sum[threadIdx.x] = tanks;
  ice_sum[threadIdx.x] = ices;
  __syncthreads();
  for (int off = 1; off < (int)blockDim.x; off <<= 1) {
    int t = threadIdx.x >= (unsigned)off ? tank_sum[threadIdx.x - off] : 0;
    int i = threadIdx.x >= (unsigned)off ? ice_sum[threadIdx.x - off] : 0;
    __syncthreads();
    tank_sum[threadIdx.x] += t;
    ice_sum[threadIdx.x] += i;
    __syncthreads();
  }
  int tank_base = tank_sum[threadIdx.x] - tanks, ice_base = ice_sum[threadIdx.x] - ices;
  for (int b = begin; b < end; ++b) {
    const int t = counts[2 * b], i = counts[2 * b + 1];
    counts[2 * b] = tank_base;
    counts[2 * b + 1] = ice_base;
    tank_base += t;
    ice_base += i;
  }
  if (threadIdx.x == blockDim.x - 1) {
    g.control->tank_count = tank_sum[threadIdx.x];
    g.control->ice_count = ice_sum[threadIdx.x];
  }
}
// Each thread owns 16 consecutive cells, so one block-wide scan of the
// per-thread counts places every cell in cell order.  Both counts (at most
// 4096 per block) share one scan as the halves of an int.
__global__ void __launch_bounds__(256) k_scatter_flags(icy3d_grid g) {
  const int N = (int)cells(g);
  const int* offsets = reinterpret_cast<const int*>(g.partials);
  const int n0 = blockIdx.x * kCompactCells + threadIdx.x * kCompactPerThread;
  unsigned tank, ice;
  flag_bits(g, n0, N, tank, ice);
  const int before = block_exclusive_scan(__popc(tank) | (__popc(ice) << 16));
  int tank_at = offsets[2 * blockIdx.x] + (before & 0xffff);
  int ice_at = offsets[2 * blockIdx.x + 1] + (before >> 16);
  for (; tank; tank &= tank - 1u) g.tank_cells[tank_at++] = n0 + __ffs(tank) - 1;
  for (; ice; ice &= ice - 1u) g.ice_cells[ice_at++] = n0 + __ffs(ice) - 1;
}

// ---------------------------------------------------------------------------
// Gradients (gradients.py).
__device__ __forceinline__ void tank_mirror(const icy3d_grid& g, int& i, int& j, int& k) {
  const int b = g.boundary;
  if (i < b) i = 2 * b - 1 - i; else if (i >= g.nx - b) i = 2 * (g.nx - b) - 1 - i;
  if (j < b) j = 2 * b - 1 - j; else if (j >= g.ny - b) j = 2 * (g.ny - b) - 1 - j;
  if (k < b) k = 2 * b - 1 - k; else if (k >= g.nz - b) k = 2 * (g.nz - b) - 1 - k;
}
// gradients.py:35-46
__device__ void coverage_normal(const icy3d_grid& g, int i, int j, int k, float out[3]) {
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    int li = i - (a == 0), lj = j - (a == 1), lk = k - (a == 2);
    int hi = i + (a == 0), hj = j + (a == 1), hk = k + (a == 2);
    tank_mirror(g, li, lj, lk);
    tank_mirror(g, hi, hj, hk);
    out[a] = 0.0f;
    if (inside(g, li, lj, lk) && inside(g, hi, hj, hk))
      out[a] = 0.5f * (g.coverage[lin(g, hi, hj, hk)] - g.coverage[lin(g, li, lj, lk)]);
  }
}
// gradients.py:60-74: reflect J about the coverage-isosurface tangent plane.
__device__ void ice_mirror_point(const icy3d_grid& g, int i, int j, int k, int ji, int jj, int jk, float out[3]) {
  const float c[3] = {(float)(ji - i), (float)(jj - j), (float)(jk - k)};
  const float eta = link_fraction(g, lin(g, i, j, k), lin(g, ji, jj, jk));
  float gi[3], gj[3], n[3];
  coverage_normal(g, i, j, k, gi);
  coverage_normal(g, ji, jj, jk, gj);
#pragma unroll
  for (int a = 0; a < 3; ++a) n[a] = (1.0f - eta) * gi[a] + eta * gj[a];
  float nc = n[0] * c[0] + n[1] * c[1] + n[2] * c[2];
  float nn = n[0] * n[0] + n[1] * n[1] + n[2] * n[2];
  float cc = c[0] * c[0] + c[1] * c[1] + c[2] * c[2];
  if (nc <= 1e-6f * sqrtf(nn * cc) || nn < 1e-12f) {
    n[0] = c[0];
    n[1] = c[1];
    n[2] = c[2];
  }
  nn = n[0] * n[0] + n[1] * n[1] + n[2] * n[2];
  float inv = 1.0f / sqrtf(nn + 1e-30f);
#pragma unroll
  for (int a = 0; a < 3; ++a) n[a] *= inv;
  nc = n[0] * c[0] + n[1] * c[1] + n[2] * c[2];
  const float J[3] = {(float)ji, (float)jj, (float)jk};
#pragma unroll
  for (int a = 0; a < 3; ++a) out[a] = J[a] - 2.0f * (1.0f - eta) * nc * n[a];
}
// gradients.py:76-101: bounded trilinear sample over fluid corners only.
__device__ float fluid_interpolate(const icy3d_grid& g, const float p[3], float fallback) {
  int base[3];
  float part[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    base[a] = (int)floorf(p[a]);
    part[a] = p[a] - (float)base[a];
  }
  float value = 0.0f, total = 0.0f;
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    int a = t >> 2, b = (t >> 1) & 1, cc = t & 1;
    int i = base[0] + a, j = base[1] + b, k = base[2] + cc;
    tank_mirror(g, i, j, k);
    if (!fluid_at(g, i, j, k)) continue;
    float w = (a ? part[0] : 1.0f - part[0]) * (b ? part[1] : 1.0f - part[1]) * (cc ? part[2] : 1.0f - part[2]);
    value += w * g.phi[lin(g, i, j, k)];
    total += w;
  }
  return total > 1e-7f ? value / total : fallback;
}
// gradients.py:103-113
__device__ float wall_phase_sample(const icy3d_grid& g, int i, int j, int k, int dx, int dy, int dz) {
  int ji = i + dx, jj = j + dy, jk = k + dz;
  tank_mirror(g, ji, jj, jk);
  float value = g.phi[lin(g, i, j, k)];
  if (fluid_at(g, ji, jj, jk)) {
    value = g.phi[lin(g, ji, jj, jk)];
  } else if (inside(g, ji, jj, jk)) {
    float point[3];
    ice_mirror_point(g, i, j, k, ji, jj, jk, point);
    value = fluid_interpolate(g, point, value);
  }
  return value;
}

__device__ __forceinline__ void store_gradient(const icy3d_grid& g, int n, float gx, float gy, float gz) {
  const size_t N = cells(g);
  g.grad[n] = gx;
  g.grad[N + n] = gy;
  g.grad[2 * N + n] = gz;
}

// gradients.py:116-145: general gradient with wall and ice mirror samples.
__device__ void general_gradient(const icy3d_grid& g, const Cell& c) {
  float rx = 0.0f, ry = 0.0f, rz = 0.0f;
  if (g.id[c.n] == -1) {
    const float centre = g.phi[c.n];
    bool wall = false;
#pragma unroll
    for (int q = 0; q < 27; ++q) {
      if (q == 13) continue;
      int i = c.i + cx(q), j = c.j + cy(q), k = c.k + cz(q);
      if (fluid_at(g, i, j, k)) {
        float d = g.phi[lin(g, i, j, k)] - centre;
        const float w = w27(q);
        if (cx(q)) rx += w * (float)cx(q) * d;
        if (cy(q)) ry += w * (float)cy(q) * d;
        if (cz(q)) rz += w * (float)cz(q) * d;
      } else {
        wall = true;
      }
    }
    if (wall) {
      for (int q = 0; q < 27; ++q) {
        if (q == 13) continue;
        int dx = cx(q), dy = cy(q), dz = cz(q);
        if (fluid_at(g, c.i + dx, c.j + dy, c.k + dz)) continue;
        float d = wall_phase_sample(g, c.i, c.j, c.k, dx, dy, dz) - centre;
        const float w = w27(q);
        rx += w * (float)dx * d;
        ry += w * (float)dy * d;
        rz += w * (float)dz * d;
      }
    }
  }
  store_gradient(g, c.n, 3.0f * rx, 3.0f * ry, 3.0f * rz);
}

// Tiled regular gradient (gradients.py:359-373, flags 0 and 1).  The D3Q27
// weights factor as w(c) = w1(cx) w1(cy) w1(cz) with w1(0) = 2/3 and
// w1(+-1) = 1/6, so the isotropic gradient 3 sum_q w_q c_q phi(x + c_q) is
// separable: d/dx = 3 D_x S_y S_z phi with D u = (u+ - u-) / 6 and
// S u = (u- + 4 u0 + u+) / 6 (the centre value cancels since sum w c = 0).
// A block sweeps x over a (kGradJ x kGradK) column: each phi slab (one-cell
// halo, wall positions read through the tank mirror so that flag-1 cells see
// their mirrored neighbours) is staged once in LDS, every thread forms
// P = S_y S_z, Qy = D_y S_z and Qz = S_y D_z for its column, and the x
// combination runs in registers over three consecutive slabs.
constexpr int kGradJ = 4, kGradK = 64;
constexpr int kGradHJ = kGradJ + 2, kGradHK = kGradK + 2, kGradSlab = kGradHJ * kGradHK;
constexpr int kGradRounds = (kGradSlab + kGradJ * kGradK - 1) / (kGradJ * kGradK);

__device__ __forceinline__ float staged_phi(const icy3d_grid& g, int i, int j, int k) {
  tank_mirror(g, i, j, k);
  i = min(max(i, 0), g.nx - 1);
  j = min(max(j, 0), g.ny - 1);
  k = min(max(k, 0), g.nz - 1);
  return g.phi[lin(g, i, j, k)];
}

// Grids of the per-cell ice-list kernels (no cross-block sums): one resident
// round of 256-thread blocks on 256 CUs at each kernel's occupancy (8 and 5
// waves per SIMD), so ~10^4 listed cells run in one pass rather than two.
constexpr unsigned kGradientListBlocks = 2048, kForceListBlocks = 1280;
// gradients.py:15-20: every phase and coverage dependency of a gradient lies
// within this many cells.
constexpr int kGradientRadius = 6;
// Tiles of box m: ceil(ez / kGradK) x ceil(ey / kGradJ) x ceil(ex / slabs),
// k fastest; the boxes' tiles share one launch.
__host__ __device__ inline int grad_tiles(const int lo[3], const int hi[3], int slabs) {
  return ((hi[2] - lo[2] + kGradK - 1) / kGradK) * ((hi[1] - lo[1] + kGradJ - 1) / kGradJ) *
         ((hi[0] - lo[0] + slabs - 1) / slabs);
}
__global__ void __launch_bounds__(kGradJ* kGradK) k_gradients_tiled(icy3d_grid g, BoxList tiles, int slabs) {
  __shared__ float sp[kGradSlab];
  int m = 0;
  while (m + 1 < tiles.count && (int)blockIdx.x >= tiles.first[m + 1]) ++m;
  Box box;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    box.lo[a] = tiles.lo[m][a];
    box.hi[a] = tiles.hi[m][a];
  }
  const int tile = (int)blockIdx.x - tiles.first[m];
  const int nk = (box.hi[2] - box.lo[2] + kGradK - 1) / kGradK, nj = (box.hi[1] - box.lo[1] + kGradJ - 1) / kGradJ;
  const int tk = threadIdx.x % kGradK, tj = threadIdx.x / kGradK;
  const int k0 = box.lo[2] + (tile % nk) * kGradK, j0 = box.lo[1] + (tile / nk % nj) * kGradJ;
  const int x0 = box.lo[0] + tile / nk / nj * slabs, x_end = min(x0 + slabs, box.hi[0]);
  const int j = j0 + tj, k = k0 + tk;
  const bool mine = j < box.hi[1] && k < box.hi[2];
  int label = 0;  // of the cell that the next slab completes, loaded a slab ahead
  float fetched[kGradRounds];
#pragma unroll
  for (int r = 0; r < kGradRounds; ++r) {
    const int t = threadIdx.x + r * blockDim.x;
    fetched[r] = t < kGradSlab ? staged_phi(g, x0 - 1, j0 - 1 + t / kGradHK, k0 - 1 + t % kGradHK) : 0.0f;
  }
  float p_m2 = 0.0f, p_m1 = 0.0f, qy_m2 = 0.0f, qy_m1 = 0.0f, qz_m2 = 0.0f, qz_m1 = 0.0f;
  const float sixth = 1.0f / 6.0f;
  for (int s = x0 - 1; s <= x_end; ++s) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kGradRounds; ++r) {
      const int t = threadIdx.x + r * blockDim.x;
      if (t < kGradSlab) sp[t] = fetched[r];
    }
    if (s < x_end) {
#pragma unroll
      for (int r = 0; r < kGradRounds; ++r) {
        const int t = threadIdx.x + r * blockDim.x;
        fetched[r] = t < kGradSlab ? staged_phi(g, s + 1, j0 - 1 + t / kGradHK, k0 - 1 + t % kGradHK) : 0.0f;
      }
    }
    const int flag = label;
    if (s >= x0 && s < x_end && mine) label = g.flag[lin(g, s, j, k)];
    __syncthreads();
    float sz[3], dz[3];
#pragma unroll
    for (int dy = 0; dy < 3; ++dy) {
      const int row = (tj + dy) * kGradHK + tk;
      const float a = sp[row], b = sp[row + 1], c = sp[row + 2];
      sz[dy] = (a + 4.0f * b + c) * sixth;
      dz[dy] = (c - a) * sixth;
    }
    const float p = (sz[0] + 4.0f * sz[1] + sz[2]) * sixth;
    const float qy = (sz[2] - sz[0]) * sixth;
    const float qz = (dz[0] + 4.0f * dz[1] + dz[2]) * sixth;
    const int x = s - 1;
    if (x >= x0 && mine) {
      const int n = lin(g, x, j, k);
      if (flag == 0 || flag == 1) {
        store_gradient(g, n, 3.0f * (p - p_m2) * sixth, 3.0f * (qy_m2 + 4.0f * qy_m1 + qy) * sixth,
                       3.0f * (qz_m2 + 4.0f * qz_m1 + qz) * sixth);
      } else if (flag < 0) {
        store_gradient(g, n, 0.0f, 0.0f, 0.0f);
      }
    }
    p_m2 = p_m1;
    p_m1 = p;
    qy_m2 = qy_m1;
    qy_m1 = qy;
    qz_m2 = qz_m1;
    qz_m1 = qz;
  }
}

// gradients.py:116-145 with one lane per direction (wall links sample the
// mirror), summed within the cell's 32-lane group.
__global__ void __launch_bounds__(256) k_gradients_general_list(icy3d_grid g, BoxList boxes) {
  const int lane = threadIdx.x & (kCellLanes - 1);
  const int groups = blockDim.x / kCellLanes;
  const int count = g.control->ice_count;
  for (int t = blockIdx.x * groups + threadIdx.x / kCellLanes; t < count; t += gridDim.x * groups) {
    const int n = g.ice_cells[t];
    const Cell c = cell_of(g, n);
    if (!list_contains(boxes, c.i, c.j, c.k)) continue;
    const float centre = g.phi[n];
    float rx = 0.0f, ry = 0.0f, rz = 0.0f;
    if (lane < 27 && lane != 13) {
      const int dx = cx(lane), dy = cy(lane), dz = cz(lane);
      const int i = c.i + dx, j = c.j + dy, k = c.k + dz;
      const float sample = fluid_at(g, i, j, k) ? g.phi[lin(g, i, j, k)] : wall_phase_sample(g, c.i, c.j, c.k, dx, dy, dz);
      const float d = sample - centre, w = w27(lane);
      rx = w * (float)dx * d;
      ry = w * (float)dy * d;
      rz = w * (float)dz * d;
    }
    rx = group_sum(rx);
    ry = group_sum(ry);
    rz = group_sum(rz);
    if (lane == 0) store_gradient(g, n, 3.0f * rx, 3.0f * ry, 3.0f * rz);
  }
}
__global__ void k_write_gradient_all(icy3d_grid g) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (int)cells(g)) return;
  general_gradient(g, cell_of(g, n));
}

// Capillary stress 1.5 sigma W (|g|^2 I - g g^T), gradients.py:147-158.
__device__ __forceinline__ void stress_of(const icy3d_grid& g, float gx, float gy, float gz, float s[9]) {
  const float k = 1.5f * g.sigma * g.width;
  const float gg = gx * gx + gy * gy + gz * gz;
  const float v[3] = {gx, gy, gz};
#pragma unroll
  for (int a = 0; a < 3; ++a)
#pragma unroll
    for (int b = 0; b < 3; ++b) s[3 * a + b] = k * ((a == b ? gg : 0.0f) - v[a] * v[b]);
}
__device__ __forceinline__ void load_grad(const icy3d_grid& g, int n, float v[3]) {
  const size_t N = cells(g);
  v[0] = g.grad[n];
  v[1] = g.grad[N + n];
  v[2] = g.grad[2 * N + n];
}
__global__ void k_capillary_stress(icy3d_grid g, float* __restrict__ out) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t N = cells(g);
  if (n >= (int)N) return;
  float v[3], s[9];
  load_grad(g, n, v);
  stress_of(g, v[0], v[1], v[2], s);
#pragma unroll
  for (int t = 0; t < 9; ++t) out[t * N + n] = s[t];
}

// ---------------------------------------------------------------------------
// D3Q7 AA collision (phase.py:93-127).
// moving_walls == 2: as 1, but the link classes are current, so cells of
// class 0 or 1 (no ice or cavity cell among their 26 neighbours) skip the
// neighbour labels.
__global__ void k_collide_phase(icy3d_grid g, int parity, int moving_walls) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t N = cells(g);
  if (n >= (int)N || g.id[n] != -1) return;
  if (moving_walls == 2) moving_walls = g.flag[n] == 2;
  const Cell c = cell_of(g, n);
  const float phi = g.phi[n];
  const float u[3] = {g.u[n], g.u[N + n], g.u[2 * N + n]};
  float gr[3];
  load_grad(g, n, gr);
  const float norm = sqrtf(gr[0] * gr[0] + gr[1] * gr[1] + gr[2] * gr[2] + g.normal_eps * g.normal_eps + 1e-28f);
  const float nrm[3] = {gr[0] / norm, gr[1] / norm, gr[2] / norm};
  int addr[7];
  float in[7], post[7], fl[3];
#pragma unroll
  for (int q = 0; q < 7; ++q) {
    addr[q] = phase_addr(g, c, q, parity);
    in[q] = g.h[addr[q]];
  }
  phase_collision(in, phi, u, nrm, g.mobility, g.width, post, fl);
  const float scale = 1.0f - g.rho_air;
  g.flux[n] = scale * fl[0];
  g.flux[N + n] = scale * fl[1];
  g.flux[2 * N + n] = scale * fl[2];
#pragma unroll
  for (int q = 0; q < 7; ++q) {
    float value = post[q];
    if (q != 0 && moving_walls) {
      int i = c.i + kC7[q][0], j = c.j + kC7[q][1], k = c.k + kC7[q][2];
      if (inside(g, i, j, k)) {
        int m = lin(g, i, j, k);
        int b = g.id[m];
        if (b >= 0) {
          float eta = link_fraction(g, n, m), ub[3];
          body_velocity_at(g, c.i + 0.5f + eta * kC7[q][0], c.j + 0.5f + eta * kC7[q][1],
                           c.k + 0.5f + eta * kC7[q][2], b, ub);
          value -= phi * (kC7[q][0] * ub[0] + kC7[q][1] * ub[1] + kC7[q][2] * ub[2]);
        }
      }
    }
    // The slot that held logical opp(q) receives post[q] (AA swap).
    g.h[addr[opp7(q)]] = value;
  }
}

// simulator.py:778-794 (per-cell part).
struct Stability {
  float speed;
  int invalid;
};
__device__ __forceinline__ Stability stability_at(const icy3d_grid& g, int n, float phi, float p) {
  const size_t N = cells(g);
  float speed = fabsf(g.u[n]) + fabsf(g.u[N + n]) + fabsf(g.u[2 * N + n]);
  bool bad = !isfinite(speed) || speed > g.max_velocity || !isfinite(p) || !isfinite(phi);
  Stability s;
  s.speed = isnan(speed) ? 0.0f : speed;
  s.invalid = bad ? n : INT32_MAX;
  return s;
}
__device__ __forceinline__ void commit_stability(const icy3d_grid& g, Stability s) {
  float speed = wave_max(s.speed);
  int invalid = wave_min_int(s.invalid);
  if (wave_leader()) {
    if (speed > 0.0f) atomic_max_nonneg(&g.control->maximum_speed, speed);
    if (invalid != INT32_MAX) atomicMin(&g.control->invalid_index, invalid);
  }
}

// phase.py:132-161, fused pressure recovery and stability scan.
__global__ void k_recover_phase(icy3d_grid g, int parity, int recover_flow) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t N = cells(g);
  bool active = n < (int)N;
  float clip = 0.0f;
  Stability st = {0.0f, INT32_MAX};
  if (active) {
    if (g.id[n] != -1) {
      g.phi[n] = 0.0f;
    } else {
      const Cell c = cell_of(g, n);
      float total = g.h[n];
#pragma unroll
      for (int a = 0; a < 3; ++a) total += g.h[phase_addr(g, c, 2 * a + 1, parity)] + g.h[phase_addr(g, c, 2 * a + 2, parity)];
      float bounded = isfinite(total) ? clamp01(total) : total;
      g.h[n] += bounded - total;
      g.phi[n] = bounded;
      clip = bounded - total;
      if (recover_flow) {
        float p = g.home[n] * density(g, bounded) / 3.0f;
        g.pressure[n] = p;
        if (g.check_stability) st = stability_at(g, n, bounded, p);
      }
    }
  }
  if (!isfinite(clip)) clip = 0.0f;
  // Per-block clip sum, maximum speed and first invalid index (stored as its
  // int32 bits, INT32_MAX for none), reduced per wave and then across the
  // block's waves with one barrier; folded by k_fold_recovery.
  const bool scan = recover_flow && g.check_stability;
  __shared__ float wave_clip[kBlock / 64], wave_speed[kBlock / 64];
  __shared__ int wave_invalid[kBlock / 64];
  const float clip_w = wave_sum(clip);
  const float speed_w = scan ? wave_max(st.speed) : 0.0f;
  const int invalid_w = scan ? wave_min_int(st.invalid) : INT32_MAX;
  if (wave_leader()) {
    wave_clip[threadIdx.x >> 6] = clip_w;
    wave_speed[threadIdx.x >> 6] = speed_w;
    wave_invalid[threadIdx.x >> 6] = invalid_w;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float total = 0.0f, speed = wave_speed[0];
    int invalid = wave_invalid[0];
    for (int w = 0; w < kBlock / 64; ++w) total += wave_clip[w];
    for (int w = 1; w < kBlock / 64; ++w) {
      speed = fmaxf(speed, wave_speed[w]);
      invalid = min(invalid, wave_invalid[w]);
    }
    g.partials[blockIdx.x] = total;
    if (scan) {
      g.partials[gridDim.x + blockIdx.x] = speed;
      reinterpret_cast<int*>(g.partials)[2 * gridDim.x + blockIdx.x] = invalid;
    }
  }
}
// Folds the per-block partials of k_recover_phase: the clip volume (the
// fixed-order sum of k_finish_sum) and, with `scan`, the maximum speed and
// first invalid index (simulator.py:778-805), which replace the previous
// step's values.
__global__ void __launch_bounds__(kFinishThreads) k_fold_recovery(icy3d_grid g, int blocks, int scan) {
  const float clip = finish_total(g.partials, blocks);
  float speed = 0.0f;
  int invalid = INT32_MAX;
  if (scan) {
    // Order-free maximum and minimum, four partials in flight per thread.
    const float* speeds = g.partials + blocks;
    const int* firsts = reinterpret_cast<const int*>(g.partials + 2 * blocks);
    int b = threadIdx.x;
    for (; b + 3 * kFinishThreads < blocks; b += 4 * kFinishThreads) {
      float s4[4];
      int v4[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        s4[u] = speeds[b + u * kFinishThreads];
        v4[u] = firsts[b + u * kFinishThreads];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        speed = fmaxf(speed, s4[u]);
        invalid = min(invalid, v4[u]);
      }
    }
    for (; b < blocks; b += kFinishThreads) {
      speed = fmaxf(speed, speeds[b]);
      invalid = min(invalid, firsts[b]);
    }
    speed = block_max(speed);
    invalid = block_min_int(invalid);
  }
  if (threadIdx.x == 0) {
    g.control->phase_clip_volume += clip;
    if (scan) {
      g.control->maximum_speed = speed;
      g.control->invalid_index = invalid == INT32_MAX ? (int32_t)cells(g) : invalid;
      g.control->peak_speed = fmaxf(g.control->peak_speed, speed);
    }
  }
}

__global__ void k_recover_pressure(icy3d_grid g) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (int)cells(g) || g.id[n] != -1) return;
  g.pressure[n] = g.home[n] * density(g, g.phi[n]) / 3.0f;
}
__global__ void k_scan_stability(icy3d_grid g) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  Stability st = {0.0f, INT32_MAX};
  if (n < (int)cells(g) && g.id[n] == -1) st = stability_at(g, n, g.phi[n], g.pressure[n]);
  commit_stability(g, st);
}
__global__ void k_reset_stability(icy3d_grid g) {
  g.control->invalid_index = (int32_t)cells(g);
  g.control->maximum_speed = 0.0f;
}
__global__ void k_fold_peak(icy3d_grid g) {
  g.control->peak_speed = fmaxf(g.control->peak_speed, g.control->maximum_speed);
}

// phase.py:163-184
__global__ void k_repair_layout(icy3d_grid g, BoxList boxes) {
  if (refresh_halted(g)) return;
  Cell c;
  if (!list_cell(g, boxes, c)) return;
  const size_t N = cells(g);
  const int n = c.n;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int q = 2 * a + 1;
    int i = c.i + kC7[q][0], j = c.j + kC7[q][1], k = c.k + kC7[q][2];
    if (!inside(g, i, j, k)) continue;
    int m = lin(g, i, j, k);
    bool before = g.prev_id[n] == -1 && g.prev_id[m] == -1;
    bool after = g.id[n] == -1 && g.id[m] == -1;
    if (before != after) {
      float v = g.h[(size_t)opp7(q) * N + n];
      g.h[(size_t)opp7(q) * N + n] = g.h[(size_t)q * N + m];
      g.h[(size_t)q * N + m] = v;
    }
  }
}
// phase.py:186-191 (out is [7][N] logical populations)
__global__ void k_export_phase(icy3d_grid g, int parity, float* __restrict__ out) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t N = cells(g);
  if (n >= (int)N) return;
  const Cell c = cell_of(g, n);
#pragma unroll
  for (int q = 0; q < 7; ++q) out[(size_t)q * N + n] = g.h[phase_addr(g, c, q, parity)];
}

// ---------------------------------------------------------------------------
// Forces (simulator.py:418-519) and HOME acceleration (home.py:127-197).
// simulator.py:193-215
__device__ bool connected(const icy3d_grid& g, int i, int j, int k, int dx, int dy, int dz) {
  if (!fluid_at(g, i + dx, j + dy, k + dz)) return false;
  int distance = abs(dx) + abs(dy) + abs(dz);
  if (distance <= 1) return true;
  const int c[3] = {dx, dy, dz};
  bool valid = false;
  for (int a = 0; a < 3; ++a) {
    if (c[a] == 0) continue;
    int A[3] = {i, j, k};
    A[a] += c[a];
    if (!fluid_at(g, A[0], A[1], A[2])) continue;
    if (distance == 2) {
      valid = true;
    } else {
      for (int b = 0; b < 3; ++b) {
        if (b == a) continue;
        int B[3] = {A[0], A[1], A[2]};
        B[b] += c[b];
        if (fluid_at(g, B[0], B[1], B[2])) valid = true;
      }
    }
  }
  return valid;
}

// simulator.py:397-416: stress of the link neighbour (planar-wall mirror).
__device__ void capillary_neighbor(const icy3d_grid& g, int i, int j, int k, int dx, int dy, int dz, float s[9]) {
  float v[3];
  load_grad(g, lin(g, i, j, k), v);
  int ji = i + dx, jj = j + dy, jk = k + dz;
  if (fluid_at(g, ji, jj, jk)) {
    load_grad(g, lin(g, ji, jj, jk), v);
  } else if (inside(g, ji, jj, jk) && g.id[lin(g, ji, jj, jk)] == -2) {
    const int b = g.boundary;
    const int shape[3] = {g.nx, g.ny, g.nz};
    int J[3] = {ji, jj, jk};
    float r[3] = {1.0f, 1.0f, 1.0f};
    for (int a = 0; a < 3; ++a) {
      if (J[a] < b) {
        J[a] = 2 * b - 1 - J[a];
        r[a] = -1.0f;
      } else if (J[a] >= shape[a] - b) {
        J[a] = 2 * (shape[a] - b) - 1 - J[a];
        r[a] = -1.0f;
      }
    }
    if (fluid_at(g, J[0], J[1], J[2])) {
      load_grad(g, lin(g, J[0], J[1], J[2]), v);
      // R S(g) R = S(R g) for a diagonal sign matrix R.
      v[0] *= r[0];
      v[1] *= r[1];
      v[2] *= r[2];
    }
  }
  stress_of(g, v[0], v[1], v[2], s);
}

__device__ void force_at(const icy3d_grid& g, const Cell& c, bool with_flux, float f[3]) {
  const size_t N = cells(g);
  const int n = c.n;
  const float phi = g.phi[n], rho = density(g, phi);
  const float gy = g.gravity_y;
  const float tw = water_temperature(g, n);
  f[0] = 0.0f;
  f[1] = (rho - g.ref_density[c.j]) * gy;
  f[2] = 0.0f;
  f[1] -= fmaxf(0.0f, 2.0f * phi - 1.0f) * g.expansion * (tw - g.water_t0) * gy;
  if (g.sigma > 0.0f) {
    bool wall = false;
    const float kcap = 4.5f * g.sigma * g.width;
#pragma unroll
    for (int q = 0; q < 27; ++q) {
      if (q == 13) continue;
      int i = c.i + cx(q), j = c.j + cy(q), k = c.k + cz(q);
      float v[3];
      bool valid = false;
      if (fluid_at(g, i, j, k)) {
        load_grad(g, lin(g, i, j, k), v);
        valid = true;
      } else {
        wall = true;
      }
      if (valid) {
        const float gg = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
        const float gc = (float)cx(q) * v[0] + (float)cy(q) * v[1] + (float)cz(q) * v[2];
        const float coef = kcap * w27(q);
        f[0] += coef * (gg * (float)cx(q) - gc * v[0]);
        f[1] += coef * (gg * (float)cy(q) - gc * v[1]);
        f[2] += coef * (gg * (float)cz(q) - gc * v[2]);
      }
    }
    if (wall) {
      for (int q = 0; q < 27; ++q) {
        if (q == 13) continue;
        int dx = cx(q), dy = cy(q), dz = cz(q);
        if (fluid_at(g, c.i + dx, c.j + dy, c.k + dz)) continue;
        float s[9];
        capillary_neighbor(g, c.i, c.j, c.k, dx, dy, dz, s);
        const float w3 = 3.0f * w27(q);
#pragma unroll
        for (int a = 0; a < 3; ++a) f[a] += w3 * (s[3 * a] * dx + s[3 * a + 1] * dy + s[3 * a + 2] * dz);
      }
    }
  }
  if (with_flux) {
    const float ui[3] = {g.u[n], g.u[N + n], g.u[2 * N + n]};
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int sign = 0; sign < 2; ++sign) {
        const int d = 2 * sign - 1;
        int i = c.i + (a == 0) * d, j = c.j + (a == 1) * d, k = c.k + (a == 2) * d;
        if (!fluid_at(g, i, j, k)) continue;
        const int m = lin(g, i, j, k);
        const float mass_flux = 0.5f * (g.flux[a * N + n] + g.flux[a * N + m]);
        const bool own = (float)d * mass_flux >= 0.0f;
        float fl[3];
#pragma unroll
        for (int e = 0; e < 3; ++e) {
          float donor = own ? ui[e] : g.u[e * N + m];
          fl[e] = mass_flux * (donor - ui[e]);
        }
        if (g.flux_limit > 0.0f) {
          float budget = g.flux_limit / 6.0f * fminf(rho, density(g, g.phi[m]));
          float scale = fminf(1.0f, budget / (fabsf(fl[0]) + fabsf(fl[1]) + fabsf(fl[2]) + 1e-20f));
          fl[0] *= scale;
          fl[1] *= scale;
          fl[2] *= scale;
        }
        f[0] -= (float)d * fl[0];
        f[1] -= (float)d * fl[1];
        f[2] -= (float)d * fl[2];
      }
  }
}

// simulator.py:559-587: neighbour velocity for the stress derivative.
__device__ void stress_neighbor_velocity(const icy3d_grid& g, int i, int j, int k, int dx, int dy, int dz, float out[3]) {
  const size_t N = cells(g);
  const int n = lin(g, i, j, k);
  const float centre[3] = {g.u[n], g.u[N + n], g.u[2 * N + n]};
  out[0] = -centre[0];
  out[1] = -centre[1];
  out[2] = -centre[2];
  int ji = i + dx, jj = j + dy, jk = k + dz;
  if (fluid_at(g, ji, jj, jk)) {
    int m = lin(g, ji, jj, jk);
    out[0] = g.u[m];
    out[1] = g.u[N + m];
    out[2] = g.u[2 * N + m];
  } else if (inside(g, ji, jj, jk) && g.id[lin(g, ji, jj, jk)] >= 0) {
    int m = lin(g, ji, jj, jk);
    float eta = link_fraction(g, n, m), ub[3];
    body_velocity_at(g, i + 0.5f + eta * dx, j + 0.5f + eta * dy, k + 0.5f + eta * dz, g.id[m], ub);
    if (connected(g, i, j, k, -dx, -dy, -dz)) {
      int o = lin(g, i - dx, j - dy, k - dz);
      const float other[3] = {g.u[o], g.u[N + o], g.u[2 * N + o]};
#pragma unroll
      for (int a = 0; a < 3; ++a) out[a] = (2.0f * ub[a] + (eta - 1.0f) * other[a]) / (1.0f + eta);
    } else {
#pragma unroll
      for (int a = 0; a < 3; ++a) out[a] = 2.0f * ub[a] - centre[a];
    }
  }
}

__device__ void acceleration_at(const icy3d_grid& g, const Cell& c, const float f[3], bool moment_pressure, float a[3]) {
  const size_t N = cells(g);
  const int n = c.n;
  const float rho = density(g, g.phi[n]);
  const float inv_rho = 1.0f / rho;
  a[0] = f[0] / rho;
  a[1] = f[1] / rho;
  a[2] = f[2] / rho;
#pragma unroll
  for (int q = 0; q < 27; ++q) {
    if (q == 13) continue;
    int i = c.i + cx(q), j = c.j + cy(q), k = c.k + cz(q);
    if (!fluid_at(g, i, j, k)) continue;
    const int m = lin(g, i, j, k);
    const float rj = density(g, g.phi[m]);
    float term;
    if (moment_pressure)
      term = w27(q) * g.home[m] * ((rho - rj) / rho);
    else
      term = 3.0f * w27(q) * g.pressure[m] * (1.0f / rj - inv_rho);
    if (cx(q)) a[0] += (float)cx(q) * term;
    if (cy(q)) a[1] += (float)cy(q) * term;
    if (cz(q)) a[2] += (float)cz(q) * term;
  }
  float gr[3];
  load_grad(g, n, gr);
  const float dr = 1.0f - g.rho_air;
  gr[0] *= dr;
  gr[1] *= dr;
  gr[2] *= dr;
  if (gr[0] * gr[0] + gr[1] * gr[1] + gr[2] * gr[2] > 0.0f) {
    float G[3][3];
#pragma unroll
    for (int axis = 0; axis < 3; ++axis) {
      const int ex = axis == 0, ey = axis == 1, ez = axis == 2;
      float d[3];
      float plus[3], minus[3];
      stress_neighbor_velocity(g, c.i, c.j, c.k, ex, ey, ez, plus);
      stress_neighbor_velocity(g, c.i, c.j, c.k, -ex, -ey, -ez, minus);
#pragma unroll
      for (int e = 0; e < 3; ++e) d[e] = 0.5f * (plus[e] - minus[e]);
#pragma unroll
      for (int e = 0; e < 3; ++e) G[e][axis] = d[e];
    }
    const float coef = lattice_nu(g, n) / rho;
#pragma unroll
    for (int e = 0; e < 3; ++e)
      a[e] += coef * ((G[e][0] + G[0][e]) * gr[0] + (G[e][1] + G[1][e]) * gr[1] + (G[e][2] + G[2][e]) * gr[2]);
  }
}

// ---------------------------------------------------------------------------
// Interior forces (simulator.py:418-519 and home.py:127-197 for cells of
// flag 0 and 1: every link fluid or a tank wall).  The two 26-neighbour sums
// factor with the D3Q27 weights w(c) = w1(cx) w1(cy) w1(cz):
//   capillary  f_a = kcap sum_q w_q (c_a |g|^2 - (c.g) g_a)
//                  = kcap [D_a(|g|^2 - g_a^2) - sum_{b != a} D_b(g_a g_b)],
//   pressure   a  += sum_q w_q c p*_m (rho - rho_m) / rho = D(p*) - D(p* rho_m) / rho
//              (3 p_m (1/rho_m - 1/rho) = D(3 p/rho_m) - D(3 p) / rho without moments),
// where D_a applies (u+ - u-)/6 along a and (u- + 4 u0 + u+)/6 along the
// other two axes.  The sweep, the tiles and the order of the axes are those of
// k_stream_rows: z between lanes, y through LDS (twelve sums and the five
// values that the y faces need, double buffered), x in registers over three
// slabs.  The six face-neighbour terms (donor phase flux, viscous velocity
// gradient) take the same way.
// A position inside the tank walls is fetched from its mirror, the nearest
// cell of the fluid box, and staged as the tank formulas use it: the gradient
// with the mirrored components negated (capillary), no pressure term, the
// velocity -u of the mirror cell (halfway no-slip), and no donor flux.
// Bound by memory: 77 bytes a cell are needed, and 117 move at 256x128x128 (the
// halo's rows come again) at 89% of the copy rate, the vector ALUs 53% busy.
// Tiles of 4 x 64 cells with every quantity's 3 x 3 window read from LDS took
// 168 us there, 406 at 450x150x90 and 90 at 24x20x16; 122, 182 and 6 now (with
// twelve waves a block: sixteen spill 33 registers, 209 us at 256x128x128).
struct ForceFetch {
  float grad[3], phi, p, u[3], flux[3], volume, energy;
  int flag;
};
// Own-column values of a slab's cell, kept while the slabs after it pass.
struct ColumnCell {
  float u[3], flux_x, phi;
};
// Donor phase-flux momentum term of one face (simulator.py:499-519).
__device__ __forceinline__ void face_flux(const icy3d_grid& g, float d, float flux_own, float flux_nb, float rho,
                                          float phi_nb, const float u_own[3], const float u_nb[3], float f[3]) {
  const float mass_flux = 0.5f * (flux_own + flux_nb);
  const bool own = d * mass_flux >= 0.0f;
  float fl[3];
#pragma unroll
  for (int e = 0; e < 3; ++e) fl[e] = mass_flux * ((own ? u_own[e] : u_nb[e]) - u_own[e]);
  if (g.flux_limit > 0.0f) {
    const float budget = g.flux_limit / 6.0f * fminf(rho, density(g, phi_nb));
    const float scale = fminf(1.0f, budget / (fabsf(fl[0]) + fabsf(fl[1]) + fabsf(fl[2]) + 1e-20f));
    fl[0] *= scale;
    fl[1] *= scale;
    fl[2] *= scale;
  }
  f[0] -= d * fl[0];
  f[1] -= d * fl[1];
  f[2] -= d * fl[2];
}

__global__ void __launch_bounds__(kForceThreads) k_forces_rows(icy3d_grid g, StreamTiles T, int with_flux,
                                                                int moment_pressure) {
  __shared__ float4 quad[2][4][sweep_cells(kForceThreads)];
  __shared__ float single[2][sweep_cells(kForceThreads)];
  const size_t N = cells(g);
  const int L = T.K + 2, lane = threadIdx.x & 63, b = g.boundary;
  const int tile_k = (int)blockIdx.x % T.tiles_k, tile_j = (int)blockIdx.x / T.tiles_k % T.tiles_j;
  const int x0 = (int)blockIdx.x / T.tiles_k / T.tiles_j * T.X, x1 = min(x0 + T.X, g.nx);
  const int t = (int)(threadIdx.x >> 6) * kWaveCells + lane - 1;
  const int row = t < 0 ? 0 : t / L, col = t < 0 ? 0 : t - row * L;
  const int j = tile_j * T.J - 1 + row, k = tile_k * T.K - 1 + col;
  const bool sends = lane >= 1 && lane <= kWaveCells && row < T.J + 2;
  const bool owned = t >= 0 && sends && row >= 1 && row <= T.J && col >= 1 && col <= T.K && j < g.ny && k < g.nz;
  const int cj = min(max(j, b), g.ny - b - 1), ck = min(max(k, b), g.nz - b - 1);
  const unsigned plane = (unsigned)(g.ny * g.nz), own_plane = owned ? (unsigned)(j * g.nz + k) : 0u;
  const unsigned clamped = (unsigned)(cj * g.nz + ck);
  const bool wall_y = cj != j, wall_z = ck != k;
  // Whether the neighbours across the y and z faces are inside the walls.
  const bool open_y[2] = {j - 1 >= b, j + 1 < g.ny - b}, open_z[2] = {k - 1 >= b, k + 1 < g.nz - b};
  const float* pressure = moment_pressure ? g.home : g.pressure;

  ForceFetch f;
  auto fetch = [&](int s) __attribute__((always_inline)) {
    const unsigned o = 4u * ((unsigned)min(max(s, b), g.nx - b - 1) * plane + clamped);
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      f.grad[e] = plane_get(g.grad + e * N, o);
      f.u[e] = plane_get(g.u + e * N, o);
      f.flux[e] = plane_get(g.flux + e * N, o);
    }
    f.phi = plane_get(g.phi, o);
    f.p = plane_get(pressure, o);
    f.flag = -1;
    f.volume = f.energy = 0.0f;
    if (owned && s >= x0 && s < x1) {
      const unsigned n = (unsigned)s * plane + own_plane;
      f.flag = g.flag[n];
      f.volume = plane_get(g.water_volume, 4u * n);
      f.energy = plane_get(g.water_energy, 4u * n);
    }
  };
  fetch(x0 - 1);
  const float sixth = 1.0f / 6.0f, kcap = 4.5f * g.sigma * g.width;
  // x differences (capillary of f_x, f_y, f_z, then the pressure fields): the
  // last two slabs; x averages (the same, and the pressure fields along y and
  // z): the last two slabs.
  float diff_a[5] = {}, diff_b[5] = {}, mean_a[7] = {}, mean_b[7] = {};
  ColumnCell col_a = {}, col_b = {};
  // The last slab's cell: y and z face terms, its gradient, temperature, flag.
  float face_f[3] = {}, du_dy[3] = {}, du_dz[3] = {}, grad_b[3] = {}, temperature_b = 0.0f;
  int flag_b = -1;

  for (int s = x0 - 1; s <= x1; ++s) {
    const int buffer = s & 1;
    const bool wall_x = s < b || s >= g.nx - b, wall = wall_x || wall_y || wall_z;
    const float gx = wall_x ? -f.grad[0] : f.grad[0], gy = wall_y ? -f.grad[1] : f.grad[1];
    const float gz = wall_z ? -f.grad[2] : f.grad[2];
    const float rho = density(g, f.phi);
    ColumnCell now;
#pragma unroll
    for (int e = 0; e < 3; ++e) now.u[e] = wall ? -f.u[e] : f.u[e];
    now.flux_x = f.flux[0];
    now.phi = f.phi;
    const float flux_y = f.flux[1], flux_z = f.flux[2];
    const float temperature = water_temperature_of(g, f.volume, f.energy);
    const int flag = f.flag;
    float p1 = moment_pressure ? f.p : 3.0f * f.p / rho, p2 = moment_pressure ? f.p * rho : 3.0f * f.p;
    if (wall) p1 = p2 = 0.0f;
    // z sums and differences (6 times): of Ax, Ay, Bxy, Bxz, Byz, X1, X2 the
    // average, of Az, Bxz, Byz, X1, X2 the difference.
    const float stage[8] = {gy * gy + gz * gz, gx * gx + gz * gz, gx * gy, gx * gz, gy * gz, p1, p2, gx * gx + gy * gy};
    float below[8], above[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      below[q] = from_below(stage[q]);
      above[q] = from_above(stage[q]);
    }
    float zs[7], zd[5];
#pragma unroll
    for (int q = 0; q < 7; ++q) zs[q] = below[q] + above[q] + 4.0f * stage[q];
    zd[0] = above[7] - below[7];
#pragma unroll
    for (int q = 1; q < 5; ++q) zd[q] = above[q + 2] - below[q + 2];
    // z faces.
    float ff[3] = {0.0f, 0.0f, 0.0f}, dz_u[3];
    {
      float un[2][3];
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        un[0][e] = from_below(now.u[e]);
        un[1][e] = from_above(now.u[e]);
        dz_u[e] = 0.5f * (un[1][e] - un[0][e]);
      }
      const float flux_n[2] = {from_below(flux_z), from_above(flux_z)}, phi_n[2] = {from_below(now.phi), from_above(now.phi)};
      if (with_flux)
#pragma unroll
        for (int side = 0; side < 2; ++side)
          if (open_z[side])
            face_flux(g, side == 0 ? -1.0f : 1.0f, flux_z, flux_n[side], rho, phi_n[side], now.u, un[side], ff);
    }
    if (sends) {
      quad[buffer][0][t] = make_float4(zs[0], zs[1], zs[2], zs[3]);
      quad[buffer][1][t] = make_float4(zs[4], zs[5], zs[6], zd[0]);
      quad[buffer][2][t] = make_float4(zd[1], zd[2], zd[3], zd[4]);
      quad[buffer][3][t] = make_float4(now.u[0], now.u[1], now.u[2], flux_y);
      single[buffer][t] = now.phi;
    }
    if (s < x1) fetch(s + 1);
    __syncthreads();
    if (owned) {
      // y averages of Ax, Bxy, Bxz, X1, X2 (for the x differences), and what
      // the x averages take: y differences and the y averages of the z ones.
      float diff[5], mean[7], dy_u[3];
      {
        const float4 m0 = quad[buffer][0][t - L], p0 = quad[buffer][0][t + L];
        const float4 m1 = quad[buffer][1][t - L], p1v = quad[buffer][1][t + L];
        const float4 m2 = quad[buffer][2][t - L], p2v = quad[buffer][2][t + L];
        diff[0] = m0.x + p0.x + 4.0f * zs[0];
        diff[1] = m0.z + p0.z + 4.0f * zs[2];
        diff[2] = m0.w + p0.w + 4.0f * zs[3];
        diff[3] = m1.y + p1v.y + 4.0f * zs[5];
        diff[4] = m1.z + p1v.z + 4.0f * zs[6];
        const float az = m1.w + p1v.w + 4.0f * zd[0];
        const float bxz = m2.x + p2v.x + 4.0f * zd[1], byz = m2.y + p2v.y + 4.0f * zd[2];
        const float byz_y = p1v.x - m1.x;
        mean[0] = -((p0.z - m0.z) + bxz);
        mean[1] = (p0.y - m0.y) - byz;
        mean[2] = az - byz_y;
        mean[3] = p1v.y - m1.y;
        mean[4] = p1v.z - m1.z;
        mean[5] = m2.z + p2v.z + 4.0f * zd[3];
        mean[6] = m2.w + p2v.w + 4.0f * zd[4];
      }
      {
        const float4 m3 = quad[buffer][3][t - L], p3 = quad[buffer][3][t + L];
        const float um[3] = {m3.x, m3.y, m3.z}, up[3] = {p3.x, p3.y, p3.z};
#pragma unroll
        for (int e = 0; e < 3; ++e) dy_u[e] = 0.5f * (up[e] - um[e]);
        if (with_flux) {
          if (open_y[0]) face_flux(g, -1.0f, flux_y, m3.w, rho, single[buffer][t - L], now.u, um, ff);
          if (open_y[1]) face_flux(g, 1.0f, flux_y, p3.w, rho, single[buffer][t + L], now.u, up, ff);
        }
      }
      if (s > x0 && (flag_b == 0 || flag_b == 1)) {  // the cell s - 1
        const unsigned o = 4u * ((unsigned)(s - 1) * plane + own_plane);
        const float phi = col_b.phi, rho_b = density(g, phi);
        constexpr float kScale = 1.0f / 216.0f;
        float dx[5], avg[7];
#pragma unroll
        for (int q = 0; q < 5; ++q) dx[q] = (diff[q] - diff_a[q]) * kScale;
#pragma unroll
        for (int q = 0; q < 7; ++q) avg[q] = (mean_a[q] + 4.0f * mean_b[q] + mean[q]) * kScale;
        float force[3] = {face_f[0], (rho_b - g.ref_density[j]) * g.gravity_y + face_f[1], face_f[2]};
        force[1] -= fmaxf(0.0f, 2.0f * phi - 1.0f) * g.expansion * (temperature_b - g.water_t0) * g.gravity_y;
        if (g.sigma > 0.0f) {
          force[0] += kcap * (dx[0] + avg[0]);
          force[1] += kcap * (avg[1] - dx[1]);
          force[2] += kcap * (avg[2] - dx[2]);
        }
        if (with_flux) {
          if (s - 2 >= b) face_flux(g, -1.0f, col_b.flux_x, col_a.flux_x, rho_b, col_a.phi, col_b.u, col_a.u, force);
          if (s < g.nx - b) face_flux(g, 1.0f, col_b.flux_x, now.flux_x, rho_b, now.phi, col_b.u, now.u, force);
        }
        const float inv_rho = 1.0f / rho_b;
        float acc[3] = {force[0] / rho_b + dx[3] - dx[4] * inv_rho, force[1] / rho_b + avg[3] - avg[4] * inv_rho,
                        force[2] / rho_b + avg[5] - avg[6] * inv_rho};
        const float dr = 1.0f - g.rho_air;
        const float gr[3] = {grad_b[0] * dr, grad_b[1] * dr, grad_b[2] * dr};
        if (gr[0] * gr[0] + gr[1] * gr[1] + gr[2] * gr[2] > 0.0f) {
          float G[3][3];
#pragma unroll
          for (int e = 0; e < 3; ++e) {
            G[e][0] = 0.5f * (now.u[e] - col_a.u[e]);
            G[e][1] = du_dy[e];
            G[e][2] = du_dz[e];
          }
          const float coef =
              mixture_nu(phi, temperature_b, g.rho_water_si, g.rho_air_si, g.mu_air) * g.nu_scale / rho_b;
#pragma unroll
          for (int e = 0; e < 3; ++e)
            acc[e] += coef * ((G[e][0] + G[0][e]) * gr[0] + (G[e][1] + G[1][e]) * gr[1] + (G[e][2] + G[2][e]) * gr[2]);
        }
#pragma unroll
        for (int e = 0; e < 3; ++e) {
          plane_set(g.force + e * N, o, force[e]);
          plane_set(g.accel + e * N, o, acc[e]);
        }
      }
#pragma unroll
      for (int q = 0; q < 5; ++q) {
        diff_a[q] = diff_b[q];
        diff_b[q] = diff[q];
      }
#pragma unroll
      for (int q = 0; q < 7; ++q) {
        mean_a[q] = mean_b[q];
        mean_b[q] = mean[q];
      }
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        face_f[e] = ff[e];
        du_dy[e] = dy_u[e];
        du_dz[e] = dz_u[e];
      }
    }
    col_a = col_b;
    col_b = now;
    grad_b[0] = gx;
    grad_b[1] = gy;
    grad_b[2] = gz;
    temperature_b = temperature;
    flag_b = flag;
  }
}

// simulator.py:418-519 and home.py:127-197 for ice-adjacent cells, one lane
// per link: capillary (fluid link or mirrored stress), product-rule pressure
// term, donor phase-flux term (lanes 0..5) and the six neighbour velocities
// of the viscous derivative (lanes 0..5); lane 0 assembles the result.
__global__ void __launch_bounds__(256) k_forces_general(icy3d_grid g, int with_flux, int moment_pressure) {
  const int lane = threadIdx.x & (kCellLanes - 1);
  const int groups = blockDim.x / kCellLanes;
  const int count = g.control->ice_count;
  const size_t N = cells(g);
  for (int t = blockIdx.x * groups + threadIdx.x / kCellLanes; t < count; t += gridDim.x * groups) {
    const int n = g.ice_cells[t];
    const Cell c = cell_of(g, n);
    const float phi = g.phi[n], rho = density(g, phi);
    float f[3] = {0.0f, 0.0f, 0.0f}, acc[3] = {0.0f, 0.0f, 0.0f}, nb[3] = {0.0f, 0.0f, 0.0f};
    if (lane < 27 && lane != 13) {
      const int dx = cx(lane), dy = cy(lane), dz = cz(lane);
      const int i = c.i + dx, j = c.j + dy, k = c.k + dz;
      const bool link = fluid_at(g, i, j, k);
      const float w = w27(lane);
      if (g.sigma > 0.0f) {
        if (link) {
          float v[3];
          load_grad(g, lin(g, i, j, k), v);
          const float gg = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
          const float gc = dx * v[0] + dy * v[1] + dz * v[2];
          const float coef = 4.5f * g.sigma * g.width * w;
          f[0] = coef * (gg * dx - gc * v[0]);
          f[1] = coef * (gg * dy - gc * v[1]);
          f[2] = coef * (gg * dz - gc * v[2]);
        } else {
          float st[9];
          capillary_neighbor(g, c.i, c.j, c.k, dx, dy, dz, st);
#pragma unroll
          for (int e = 0; e < 3; ++e) f[e] = 3.0f * w * (st[3 * e] * dx + st[3 * e + 1] * dy + st[3 * e + 2] * dz);
        }
      }
      if (link) {
        const int m = lin(g, i, j, k);
        const float rj = density(g, g.phi[m]);
        const float term = moment_pressure ? w * g.home[m] * ((rho - rj) / rho)
                                           : 3.0f * w * g.pressure[m] * (1.0f / rj - 1.0f / rho);
        acc[0] = dx * term;
        acc[1] = dy * term;
        acc[2] = dz * term;
      }
    }
    if (lane < 6) {
      const int axis = lane >> 1, d = 2 * (lane & 1) - 1;
      const int ex = (axis == 0) * d, ey = (axis == 1) * d, ez = (axis == 2) * d;
      if (with_flux && fluid_at(g, c.i + ex, c.j + ey, c.k + ez)) {
        const int m = lin(g, c.i + ex, c.j + ey, c.k + ez);
        const float mass_flux = 0.5f * (g.flux[axis * N + n] + g.flux[axis * N + m]);
        const bool own = (float)d * mass_flux >= 0.0f;
        float fl[3];
#pragma unroll
        for (int e = 0; e < 3; ++e) fl[e] = mass_flux * ((own ? g.u[e * N + n] : g.u[e * N + m]) - g.u[e * N + n]);
        if (g.flux_limit > 0.0f) {
          const float budget = g.flux_limit / 6.0f * fminf(rho, density(g, g.phi[m]));
          const float scale = fminf(1.0f, budget / (fabsf(fl[0]) + fabsf(fl[1]) + fabsf(fl[2]) + 1e-20f));
#pragma unroll
          for (int e = 0; e < 3; ++e) fl[e] *= scale;
        }
#pragma unroll
        for (int e = 0; e < 3; ++e) f[e] -= (float)d * fl[e];
      }
      stress_neighbor_velocity(g, c.i, c.j, c.k, ex, ey, ez, nb);
    }
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      f[e] = group_sum(f[e]);
      acc[e] = group_sum(acc[e]);
    }
    // Neighbour velocities for the centred derivative: lane 2a+1 is +e_a.
    float plus[3][3], minus[3][3];
#pragma unroll
    for (int axis = 0; axis < 3; ++axis)
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        minus[axis][e] = __shfl(nb[e], (threadIdx.x & ~(kCellLanes - 1)) % 64 + 2 * axis, 64);
        plus[axis][e] = __shfl(nb[e], (threadIdx.x & ~(kCellLanes - 1)) % 64 + 2 * axis + 1, 64);
      }
    if (lane == 0) {
      const float gy = g.gravity_y;
      const float tw = water_temperature(g, n);
      float force[3] = {f[0], f[1], f[2]};
      force[1] += (rho - g.ref_density[c.j]) * gy - fmaxf(0.0f, 2.0f * phi - 1.0f) * g.expansion * (tw - g.water_t0) * gy;
      float a[3] = {force[0] / rho + acc[0], force[1] / rho + acc[1], force[2] / rho + acc[2]};
      float gr[3];
      load_grad(g, n, gr);
      const float dr = 1.0f - g.rho_air;
      gr[0] *= dr;
      gr[1] *= dr;
      gr[2] *= dr;
      if (gr[0] * gr[0] + gr[1] * gr[1] + gr[2] * gr[2] > 0.0f) {
        float G[3][3];
#pragma unroll
        for (int axis = 0; axis < 3; ++axis)
#pragma unroll
          for (int e = 0; e < 3; ++e) G[e][axis] = 0.5f * (plus[axis][e] - minus[axis][e]);
        const float coef = lattice_nu(g, n) / rho;
#pragma unroll
        for (int e = 0; e < 3; ++e)
          a[e] += coef * ((G[e][0] + G[0][e]) * gr[0] + (G[e][1] + G[1][e]) * gr[1] + (G[e][2] + G[2][e]) * gr[2]);
      }
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        g.force[e * N + n] = force[e];
        g.accel[e * N + n] = a[e];
      }
    }
  }
}

// simulator.py:684-706: forces and equilibrium at newly exposed cells.
__global__ void k_refill_forces(icy3d_grid g, Box box) {
  Cell c;
  if (!box_cell(g, box, blockIdx.x * blockDim.x + threadIdx.x, c)) return;
  if (!(g.id[c.n] == -1 && g.prev_id[c.n] != -1)) return;
  const size_t N = cells(g);
  float f[3], a[3];
  force_at(g, c, false, f);
  acceleration_at(g, c, f, false, a);
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    g.force[e * N + c.n] = f[e];
    g.accel[e * N + c.n] = a[e];
  }
}

__global__ void k_generic_forces(icy3d_grid g, float* __restrict__ out) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t N = cells(g);
  if (n >= (int)N) return;
  float f[3] = {0, 0, 0}, a[3] = {0, 0, 0};
  if (g.id[n] == -1) {
    const Cell c = cell_of(g, n);
    force_at(g, c, true, f);
    acceleration_at(g, c, f, true, a);
  }
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    out[e * N + n] = f[e];
    out[(3 + e) * N + n] = a[e];
  }
}

// home.py:87-100 and phase.py:84-88: equilibrium initialisation.
__device__ __forceinline__ void set_momentum_equilibrium(const icy3d_grid& g, int n, float phi, float p, float ux, float uy,
                                                         float uz) {
  const size_t N = cells(g);
  const float a[3] = {g.accel[n], g.accel[N + n], g.accel[2 * N + n]};
  const float u[3] = {ux, uy, uz};
  Moments m;
  m.m[0] = 3.0f * p / density(g, phi);
  m.m[1] = ux - 0.5f * a[0];
  m.m[2] = uy - 0.5f * a[1];
  m.m[3] = uz - 0.5f * a[2];
  const int ia[6] = {0, 1, 2, 0, 0, 1}, ib[6] = {0, 1, 2, 1, 2, 2};
#pragma unroll
  for (int t = 0; t < 6; ++t) m.m[4 + t] = u[ia[t]] * u[ib[t]] - 0.5f * (a[ia[t]] * u[ib[t]] + u[ia[t]] * a[ib[t]]);
  store_moments(g.home, N, n, m);
  g.u[n] = ux;
  g.u[N + n] = uy;
  g.u[2 * N + n] = uz;
}
__device__ __forceinline__ void set_phase_equilibrium(const icy3d_grid& g, const Cell& c, int parity, float phi, float ux,
                                                      float uy, float uz) {
#pragma unroll
  for (int q = 0; q < 7; ++q) g.h[phase_addr(g, c, q, parity)] = phase_equilibrium7(q, phi, ux, uy, uz);
}
__global__ void k_refill_equilibrium(icy3d_grid g, Box box, int parity) {
  Cell c;
  if (!box_cell(g, box, blockIdx.x * blockDim.x + threadIdx.x, c)) return;
  if (!(g.id[c.n] == -1 && g.prev_id[c.n] != -1)) return;
  const size_t N = cells(g);
  const float ux = g.u[c.n], uy = g.u[N + c.n], uz = g.u[2 * N + c.n];
  const float phi = g.phi[c.n];
  set_momentum_equilibrium(g, c.n, phi, g.pressure[c.n], ux, uy, uz);
  set_phase_equilibrium(g, c, parity, phi, ux, uy, uz);
}
// simulator.py:385-395 (zero velocity, momentum only) and the reference
// tests' seed kernels (current velocity, optional constant pressure).
__global__ void k_set_equilibrium(icy3d_grid g, int parity, int with_phase, int zero_velocity, int use_constant,
                                  float pressure) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t N = cells(g);
  if (n >= (int)N || g.id[n] != -1) return;
  float ux = 0.0f, uy = 0.0f, uz = 0.0f;
  if (!zero_velocity) {
    ux = g.u[n];
    uy = g.u[N + n];
    uz = g.u[2 * N + n];
  }
  const float phi = g.phi[n];
  set_momentum_equilibrium(g, n, phi, use_constant ? pressure : g.pressure[n], ux, uy, uz);
  if (with_phase) set_phase_equilibrium(g, cell_of(g, n), parity, phi, ux, uy, uz);
}

// ---------------------------------------------------------------------------
// HOME collision (home.py:199-211) of fluid cell n from the pre-collision
// moments in g.home: the same arithmetic in the two-kernel path (collision
// stored in home_post, then streamed) and the fused collide-stream.
__device__ __forceinline__ Moments collide_at(const icy3d_grid& g, int n) {
  const size_t N = cells(g);
  const float rate = home_shear_rate(g, g.phi[n], g.water_volume[n], g.water_energy[n]);
  return central_collision(load_moments(g.home, N, n), g.accel[n], g.accel[N + n], g.accel[2 * N + n], rate,
                           g.bulk_rate);
}
// HOME collision (home.py:199-211).
// zero_loads != 0: the first block also clears the body loads that the
// stream kernels accumulate next (one launch fewer per step).
__global__ void k_collide_momentum(icy3d_grid g, int zero_loads) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t N = cells(g);
  if (zero_loads && blockIdx.x == 0)
    for (int t = threadIdx.x; t < ICY3D_MAX_BODIES * 6; t += blockDim.x) (&g.control->loads[0][0])[t] = 0.0f;
  if (n >= (int)N || g.id[n] != -1) return;
#pragma unroll
  for (int e = 0; e < 3; ++e) g.old_u[e * N + n] = g.u[e * N + n];
  g.old_pressure[n] = g.pressure[n];
  store_moments(g.home_post, N, n, collide_at(g, n));
}

// ---------------------------------------------------------------------------
// HOME pull streaming (home.py:286-321): moment sums of the pulled populations.
struct MomentSums {
  float p, jx, jy, jz, xx, yy, zz, xy, xz, yz;
};
__device__ __forceinline__ void store_streamed(const icy3d_grid& g, float* __restrict__ dst, int n, const MomentSums& s) {
  const size_t N = cells(g);
  const float third = s.p * (1.0f / 3.0f);
  Moments m;
  m.m[0] = s.p;
  m.m[1] = s.jx;
  m.m[2] = s.jy;
  m.m[3] = s.jz;
  m.m[4] = s.xx - third;
  m.m[5] = s.yy - third;
  m.m[6] = s.zz - third;
  m.m[7] = s.xy;
  m.m[8] = s.xz;
  m.m[9] = s.yz;
  store_moments(dst, N, n, m);
  g.u[n] = s.jx + 0.5f * g.accel[n];
  g.u[N + n] = s.jy + 0.5f * g.accel[N + n];
  g.u[2 * N + n] = s.jz + 0.5f * g.accel[2 * N + n];
}

// ---------------------------------------------------------------------------
// HOME pull stream, alone and fused with the collision (home.py:199-211 then
// :286-345 for flags 0/1 and solid cells; k_stream_boundary does flag 2).
//
// With c the direction, the reconstruction of home.py:30-53 is a weight times
// a cubic in c, f(c) = w(c) sum P_abd cx^a cy^b cz^d with 17 terms P_abd per
// cell, and w(c) = w1(cx) w1(cy) w1(cz).  So the streamed moments
// sum_c c^(alpha,beta,gamma) f_c(x - c) factor into three passes of one axis:
// on the line of P0, P1, P2 along z a cell sends up = P0 + P1 + P2 to its
// upper neighbour and dn = P0 - P1 + P2 to its lower one, and gets
// U + D + 4 P0, U - D and U + D for the powers 0, 1, 2 of cz (w1 = 1/6, 4/6,
// 1/6; the 1/216 comes last); then the same along y and along x.  A non-fluid
// cell sends zeros, and its links come back by the bounce below.  About 140
// operations and 36 LDS words a cell; summing the 27 pulled populations took
// 450 and 122.  Fused, the pass is bound by memory: of 118 bytes a cell that it
// needs 188 move at 256x128x128 (the halo's rows come again), at 95% of the copy
// rate and with the vector ALUs 39% busy: 184 us, 260 with the 27 sums.
//
// A block owns J rows by K cells of a (y, z) tile and sweeps X slabs of x.
// The tile with its halo, (J + 2) rows of K + 2 cells, is laid flat over the
// lanes, 62 cells a wave: the first and last lane of a wave repeat a
// neighbour wave's cell, so the z pass is a shift between lanes, and only the
// y pass goes through LDS (nine up and nine dn values a cell, double
// buffered, one barrier a slab).  The x pass keeps the previous slabs' up
// values and centres in registers.  Loads of the next slab are issued before
// the barrier.  Fused, a staged cell is collided on load (the shear rate from
// its phase, water volume and energy, the force from its HOME acceleration):
// moments come from g.home and go to g.home_post (the caller swaps them), and
// solid cells carry their moments over, so every cell of the destination is
// defined; otherwise moments come from g.home_post and go to g.home.  u is
// written in place: no later read of the pass depends on it (the boundary
// pass reads u only at its own flag-2 cells, left alone here).
//
// Bounce: a missing link's population is R_(-c) of the cell's own
// post-collision moments.  A cell whose nine links towards one z neighbour are
// all missing and no others (the z walls, in every row) gets their sums in
// closed form from its own z lines; every other pattern goes link by link.
struct StreamFetch {
  float m[10], a[3], phi, volume, energy;
  int label, flag;
};
struct Line3 {
  float up, dn, c;
};

template <bool Fused>
__global__ void __launch_bounds__(kStreamThreads) k_stream_rows(icy3d_grid g, StreamTiles T) {
  // The y pass's values of a slab: up then dn, nine each, as 4 + 4 + 1 words.
  __shared__ float4 quad[2][4][sweep_cells(kStreamThreads)];
  __shared__ float single[2][2][sweep_cells(kStreamThreads)];
  __shared__ uint8_t links[2][sweep_cells(kStreamThreads)];  // bits 0, 1, 2: fluid at k - 1, k, k + 1
  if (Fused && blockIdx.x == 0)
    for (int t = threadIdx.x; t < ICY3D_MAX_BODIES * 6; t += blockDim.x) (&g.control->loads[0][0])[t] = 0.0f;
  const size_t N = cells(g);
  const int L = T.K + 2, lane = threadIdx.x & 63;
  const int tile_k = (int)blockIdx.x % T.tiles_k, tile_j = (int)blockIdx.x / T.tiles_k % T.tiles_j;
  const int x0 = (int)blockIdx.x / T.tiles_k / T.tiles_j * T.X, x1 = min(x0 + T.X, g.nx);
  const int t = (int)(threadIdx.x >> 6) * kWaveCells + lane - 1;
  const int row = t < 0 ? 0 : t / L, col = t < 0 ? 0 : t - row * L;
  const int j = tile_j * T.J - 1 + row, k = tile_k * T.K - 1 + col;
  const bool present = t >= 0 && row < T.J + 2 && j >= 0 && j < g.ny && k >= 0 && k < g.nz;
  const bool sends = lane >= 1 && lane <= kWaveCells && row < T.J + 2;
  const bool owned = present && sends && row >= 1 && row <= T.J && col >= 1 && col <= T.K;
  const unsigned in_plane = present ? (unsigned)(j * g.nz + k) : 0u, plane = (unsigned)(g.ny * g.nz);
  const float* source = Fused ? g.home : g.home_post;
  float* target = Fused ? g.home_post : g.home;

  StreamFetch f;
  auto fetch = [&](int s) __attribute__((always_inline)) {
    f.label = -2;
    f.flag = -1;
    if (present && s >= 0 && s < g.nx) {
      const unsigned n = (unsigned)s * plane + in_plane, o = 4u * n;
      // Every load is issued at once, without waiting for the label: a
      // non-fluid cell's values are discarded.
      f.label = g.id[n];
      f.flag = g.flag[n];
#pragma unroll
      for (int m = 0; m < 10; ++m) f.m[m] = plane_get(source + m * N, o);
#pragma unroll
      for (int e = 0; e < 3; ++e) f.a[e] = plane_get(g.accel + e * N, o);
      if (Fused) {
        f.phi = plane_get(g.phi, o);
        f.volume = plane_get(g.water_volume, o);
        f.energy = plane_get(g.water_energy, o);
      }
    }
  };
  fetch(x0 - 1);
  // Of the x lines (beta, gamma) = 00, 10, 20, 01, 11, 02: the up values of
  // the last two slabs and the centre of the last.
  float up_a[6], up_b[6], centre[6];
#pragma unroll
  for (int l = 0; l < 6; ++l) up_a[l] = up_b[l] = centre[l] = 0.0f;
  float wall[6] = {0, 0, 0, 0, 0, 0}, acc[3] = {0, 0, 0};  // of the last slab's cell
  int flag = -1;
  unsigned fluid = 0u;  // bit 9 (dx + 1) + 3 (dy + 1) + dz + 1: fluid at that neighbour of the last slab's cell

  for (int s = x0 - 1; s <= x1; ++s) {
    const int buffer = s & 1;
    const bool is_fluid = f.label == -1;
    Moments post;
#pragma unroll
    for (int m = 0; m < 10; ++m) post.m[m] = 0.0f;
    if (is_fluid) {
      Moments pre;
#pragma unroll
      for (int m = 0; m < 10; ++m) pre.m[m] = f.m[m];
      post = Fused ? central_collision(pre, f.a[0], f.a[1], f.a[2], home_shear_rate(g, f.phi, f.volume, f.energy),
                                       g.bulk_rate)
                   : pre;
    } else if (owned && s >= x0 && s < x1) {
      const unsigned n = (unsigned)s * plane + in_plane, o = 4u * n;
      float v[3] = {0.0f, 0.0f, 0.0f};
      if (f.label >= 0) body_velocity_at(g, s + 0.5f, j + 0.5f, k + 0.5f, f.label, v);
#pragma unroll
      for (int e = 0; e < 3; ++e) plane_set(g.u + e * N, o, v[e]);
      if (Fused)
#pragma unroll
        for (int m = 0; m < 10; ++m) plane_set(target + m * N, o, f.m[m]);
    }
    const float acc_s[3] = {f.a[0], f.a[1], f.a[2]};
    const int flag_s = f.flag;
    if (s < x1) fetch(s + 1);

    // z lines (a, b) = 00, 10, 01, 20, 02, 11, 12, 21.
    const float ux = post.m[1], uy = post.m[2], uz = post.m[3];
    const float sxx = post.m[4], syy = post.m[5], szz = post.m[6], sxy = post.m[7], sxz = post.m[8], syz = post.m[9];
    const float xxy = 13.5f * (sxx * uy + 2.0f * ux * (sxy - ux * uy)), xxz = 13.5f * (sxx * uz + 2.0f * ux * (sxz - ux * uz));
    const float xyy = 13.5f * (syy * ux + 2.0f * uy * (sxy - ux * uy)), yyz = 13.5f * (syy * uz + 2.0f * uy * (syz - uy * uz));
    const float xzz = 13.5f * (szz * ux + 2.0f * uz * (sxz - ux * uz)), yzz = 13.5f * (szz * uy + 2.0f * uz * (syz - uy * uz));
    const float xyz = 27.0f * (sxz * uy + syz * ux + uz * (sxy - 2.0f * ux * uy));
    const float third = 1.0f / 3.0f;
    const float z0[8] = {post.m[0] - 1.5f * (sxx + syy + szz), 3.0f * ux - third * (xyy + xzz),
                         3.0f * uy - third * (xxy + yzz), 4.5f * sxx, 4.5f * syy, 9.0f * sxy, xyy, xxy};
    const float z1[8] = {3.0f * uz - third * (xxz + yyz), 9.0f * sxz, 9.0f * syz, xxz, yyz, xyz, 0.0f, 0.0f};
    const float even[8] = {z0[0] + 4.5f * szz, z0[1] + xzz, z0[2] + yzz, z0[3], z0[4], z0[5], xyy, xxy};
    auto line = [](float p0, float p1, float p2) __attribute__((always_inline)) {
      const float sum = p0 + p2;
      return Line3{sum + p1, sum - p1, p0};
    };
    const int here = is_fluid ? 1 : 0;
    const int z_links = from_below(here) | here << 1 | from_above(here) << 2;
    // The closed-form bounce of the links towards a missing z neighbour (36
    // times their sums): c_z of the returning populations is +1 from below.
    float wall_s[6];
    {
      const float side = (z_links & 1) == 0 ? -1.0f : 1.0f;
      float e[8];
#pragma unroll
      for (int l = 0; l < 8; ++l) e[l] = even[l] + side * z1[l];
      wall_s[0] = 36.0f * e[0] + 12.0f * (e[3] + e[4]);
      wall_s[1] = -12.0f * e[1] - 4.0f * e[6];
      wall_s[2] = -12.0f * e[2] - 4.0f * e[7];
      wall_s[3] = 12.0f * (e[0] + e[3]) + 4.0f * e[4];
      wall_s[4] = 12.0f * (e[0] + e[4]) + 4.0f * e[3];
      wall_s[5] = 4.0f * e[5];
    }
    float zp[8][3];
#pragma unroll
    for (int l = 0; l < 8; ++l) {
      const float U = from_below(even[l] + z1[l]), D = from_above(even[l] - z1[l]);
      zp[l][2] = U + D;
      zp[l][1] = U - D;
      zp[l][0] = zp[l][2] + 4.0f * z0[l];
    }
    // y lines (a, gamma): powers b = 0, 1, 2 of cy are z lines (a, b).
    Line3 y[3][3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      y[0][c] = line(zp[0][c], zp[2][c], zp[4][c]);
      y[1][c] = line(zp[1][c], zp[5][c], zp[6][c]);
      y[2][c] = line(zp[3][c], zp[7][c], 0.0f);
    }
    if (sends) {
      quad[buffer][0][t] = make_float4(y[0][0].up, y[0][1].up, y[0][2].up, y[1][0].up);
      quad[buffer][1][t] = make_float4(y[1][1].up, y[1][2].up, y[2][0].up, y[2][1].up);
      quad[buffer][2][t] = make_float4(y[0][0].dn, y[0][1].dn, y[0][2].dn, y[1][0].dn);
      quad[buffer][3][t] = make_float4(y[1][1].dn, y[1][2].dn, y[2][0].dn, y[2][1].dn);
      single[buffer][0][t] = y[2][2].up;
      single[buffer][1][t] = y[2][2].dn;
      links[buffer][t] = (uint8_t)z_links;
    }
    __syncthreads();
    if (owned) {
      float U[3][3], D[3][3];
      {
        const float4 p = quad[buffer][0][t - L], q = quad[buffer][1][t - L];
        const float4 v = quad[buffer][2][t + L], w = quad[buffer][3][t + L];
        U[0][0] = p.x, U[0][1] = p.y, U[0][2] = p.z, U[1][0] = p.w;
        U[1][1] = q.x, U[1][2] = q.y, U[2][0] = q.z, U[2][1] = q.w;
        D[0][0] = v.x, D[0][1] = v.y, D[0][2] = v.z, D[1][0] = v.w;
        D[1][1] = w.x, D[1][2] = w.y, D[2][0] = w.z, D[2][1] = w.w;
        U[2][2] = single[buffer][0][t - L];
        D[2][2] = single[buffer][1][t + L];
      }
      // The cell s - 1 is complete with this slab's dn values.
      const unsigned slab_links = (unsigned)links[buffer][t - L] | (unsigned)z_links << 3 | (unsigned)links[buffer][t + L] << 6;
      fluid |= slab_links << 18;
      float h[3][6];  // power a of cx of the x lines
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        h[e][2] = U[e][0] + D[e][0];
        h[e][1] = U[e][0] - D[e][0];
        h[e][0] = h[e][2] + 4.0f * y[e][0].c;
        h[e][4] = U[e][1] - D[e][1];
        h[e][3] = U[e][1] + D[e][1] + 4.0f * y[e][1].c;
        h[e][5] = U[e][2] + D[e][2] + 4.0f * y[e][2].c;
      }
      Line3 x[6];
#pragma unroll
      for (int l = 0; l < 6; ++l) x[l] = line(h[0][l], h[1][l], h[2][l]);
      if (s > x0 && (flag == 0 || flag == 1)) {
        MomentSums m;
        float sides[6];
#pragma unroll
        for (int l = 0; l < 6; ++l) sides[l] = up_a[l] + x[l].dn;
        m.p = sides[0] + 4.0f * centre[0];
        m.jx = up_a[0] - x[0].dn;
        m.xx = sides[0];
        m.jy = sides[1] + 4.0f * centre[1];
        m.xy = up_a[1] - x[1].dn;
        m.yy = sides[2] + 4.0f * centre[2];
        m.jz = sides[3] + 4.0f * centre[3];
        m.xz = up_a[3] - x[3].dn;
        m.yz = sides[4] + 4.0f * centre[4];
        m.zz = sides[5] + 4.0f * centre[5];
        const unsigned n = (unsigned)(s - 1) * plane + in_plane;
        constexpr unsigned kAll = 0x7ffffffu, kBelow = 0x1249249u, kAbove = kBelow << 2;
        const unsigned missing = ~fluid & kAll;
        if (missing == kBelow || missing == kAbove) {
          const float c = missing == kBelow ? 1.0f : -1.0f;
          m.p += wall[0];
          m.jx += wall[1];
          m.jy += wall[2];
          m.jz += c * wall[0];
          m.xx += wall[3];
          m.yy += wall[4];
          m.zz += wall[0];
          m.xy += wall[5];
          m.xz += c * wall[1];
          m.yz += c * wall[2];
        } else if (missing) {
          const Moments own = Fused ? collide_at(g, (int)n) : load_moments(g.home_post, N, (int)n);
          for (int q = 0; q < 27; ++q) {  // the link towards neighbour q returns as direction 26 - q
            if (!__any((missing >> q) & 1u)) continue;
            const float r = (missing >> q) & 1u ? 216.0f * reconstruct_dyn(q, own) : 0.0f;
            const float cxf = (float)-cx(q), cyf = (float)-cy(q), czf = (float)-cz(q);
            m.p += r;
            m.jx += cxf * r;
            m.jy += cyf * r;
            m.jz += czf * r;
            m.xx += cxf * cxf * r;
            m.yy += cyf * cyf * r;
            m.zz += czf * czf * r;
            m.xy += cxf * cyf * r;
            m.xz += cxf * czf * r;
            m.yz += cyf * czf * r;
          }
        }
        constexpr float kScale = 1.0f / 216.0f;
        const unsigned o = 4u * n;
        const float p = kScale * m.p, p3 = p * third;
        plane_set(target, o, p);
        plane_set(target + N, o, kScale * m.jx);
        plane_set(target + 2 * N, o, kScale * m.jy);
        plane_set(target + 3 * N, o, kScale * m.jz);
        plane_set(target + 4 * N, o, kScale * m.xx - p3);
        plane_set(target + 5 * N, o, kScale * m.yy - p3);
        plane_set(target + 6 * N, o, kScale * m.zz - p3);
        plane_set(target + 7 * N, o, kScale * m.xy);
        plane_set(target + 8 * N, o, kScale * m.xz);
        plane_set(target + 9 * N, o, kScale * m.yz);
        plane_set(g.u, o, kScale * m.jx + 0.5f * acc[0]);
        plane_set(g.u + N, o, kScale * m.jy + 0.5f * acc[1]);
        plane_set(g.u + 2 * N, o, kScale * m.jz + 0.5f * acc[2]);
      }
      fluid >>= 9;
#pragma unroll
      for (int l = 0; l < 6; ++l) {
        up_a[l] = up_b[l];
        up_b[l] = x[l].up;
        centre[l] = x[l].c;
        wall[l] = wall_s[l];
      }
    }
    flag = flag_s;
#pragma unroll
    for (int e = 0; e < 3; ++e) acc[e] = acc_s[e];
  }
}

// home.py:213-254: one reflected population at an ice or tank link.  For an
// ice link it also returns the link's force and torque on body ``body``.
// ``old_u`` is the cell's velocity before the stream (home.py:203: the copy
// the collision saves; the fused path reads u itself, which is unchanged at
// flag-2 cells until this pass stores them).
__device__ float reflect_link(const icy3d_grid& g, const Cell& c, int outgoing, const Moments& post_i,
                              const float* __restrict__ old_u, int& body, float load[6]) {
  const size_t N = cells(g);
  const int dx = cx(outgoing), dy = cy(outgoing), dz = cz(outgoing);
  const int ji = c.i + dx, jj = c.j + dy, jk = c.k + dz;
  const float raw = reconstruct_rt(outgoing, post_i);
  body = -1;
  if (!inside(g, ji, jj, jk)) return raw;
  const int m = lin(g, ji, jj, jk);
  const int b = g.id[m];
  if (b < 0) return raw;  // stationary tank or unresolved cavity: bounce-back
  const Moments home_i = load_moments(g.home, N, c.n);
  const float eta = link_fraction(g, c.n, m);
  const float px = c.i + 0.5f + eta * dx, py = c.j + 0.5f + eta * dy, pz = c.k + 0.5f + eta * dz;
  float ub[3];
  body_velocity_at(g, px, py, pz, b, ub);
  const float p = home_i.m[0];
  const float neq = reconstruct_rt(outgoing, home_i) -
                    reconstruct_rt(outgoing, equilibrium_moments(p, old_u[c.n], old_u[N + c.n], old_u[2 * N + c.n]));
  const int incoming = 26 - outgoing;
  const float reflected =
      (reconstruct_rt(incoming, equilibrium_moments(p, ub[0], ub[1], ub[2])) + neq + eta * reconstruct_rt(incoming, post_i)) /
      (1.0f + eta);
  const float rho = density(g, g.phi[c.n]);
  const float cf[3] = {(float)dx, (float)dy, (float)dz};
  const float pref = (1.0f - eta) * g.ref_pressure[c.j] + eta * g.ref_pressure[jj];
  const float w = w27(outgoing);
  float impulse[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    impulse[a] = rho * ((cf[a] - ub[a]) * raw - (-cf[a] - ub[a]) * reflected);
    impulse[a] += 6.0f * w * pref * cf[a];
  }
  float own_s[9], nb_s[9], gi[3];
  load_grad(g, c.n, gi);
  stress_of(g, gi[0], gi[1], gi[2], own_s);
  capillary_neighbor(g, c.i, c.j, c.k, dx, dy, dz, nb_s);
  float cap[3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
    cap[a] = -3.0f * w *
             ((own_s[3 * a] + nb_s[3 * a]) * cf[0] + (own_s[3 * a + 1] + nb_s[3 * a + 1]) * cf[1] +
              (own_s[3 * a + 2] + nb_s[3 * a + 2]) * cf[2]);
  const float* centre = body_row(g, b) + 12;
  const float r1[3] = {px - centre[0], py - centre[1], pz - centre[2]};
  const float r2[3] = {c.i + 0.5f + 0.5f * cf[0] - centre[0], c.j + 0.5f + 0.5f * cf[1] - centre[1],
                       c.k + 0.5f + 0.5f * cf[2] - centre[2]};
#pragma unroll
  for (int a = 0; a < 3; ++a) load[a] = impulse[a] + cap[a];
  load[3] = r1[1] * impulse[2] - r1[2] * impulse[1] + (r2[1] * cap[2] - r2[2] * cap[1]);
  load[4] = r1[2] * impulse[0] - r1[0] * impulse[2] + (r2[2] * cap[0] - r2[0] * cap[2]);
  load[5] = r1[0] * impulse[1] - r1[1] * impulse[0] + (r2[0] * cap[1] - r2[1] * cap[0]);
  body = b;
  return reflected;
}

// home.py:323-345 for flag-2 cells: one lane per pulled direction; the
// 10 moment sums are reduced within the 32-lane group and body loads are
// accumulated in LDS in fixed point (units of 2^-40, so the block's sum is
// the same whatever order its lanes add in), then written as per-block
// partials; a slot that took a non-finite or out-of-range load writes NaN.  Fused: the
// post-collision moments of each pulled cell are computed from g.home here
// (collide_at) and the result goes to g.home_post, as in
// k_stream_rows<true>; otherwise they are read from home_post and the
// result goes to g.home.
constexpr double kLoadScale = 0x1p40;
template <bool Fused>
__global__ void __launch_bounds__(256) k_stream_boundary(icy3d_grid g) {
  __shared__ long long block_loads[kLoadSlots];
  __shared__ int block_bad[kLoadSlots];
  for (int t = threadIdx.x; t < kLoadSlots; t += blockDim.x) {
    block_loads[t] = 0;
    block_bad[t] = 0;
  }
  __syncthreads();
  const int lane = threadIdx.x & (kCellLanes - 1);
  const int groups = blockDim.x / kCellLanes;
  const int count = g.control->ice_count;
  const size_t N = cells(g);
  for (int t = blockIdx.x * groups + threadIdx.x / kCellLanes; t < count; t += gridDim.x * groups) {
    const int n = g.ice_cells[t];
    const Cell c = cell_of(g, n);
    float v = 0.0f;
    const int q = lane < 27 ? lane : 13;
    if (lane < 27) {
      const int i = c.i - cx(q), j = c.j - cy(q), k = c.k - cz(q);
      if (fluid_at(g, i, j, k)) {
        const int m = lin(g, i, j, k);
        v = reconstruct_dyn(q, Fused ? collide_at(g, m) : load_moments(g.home_post, N, m));
      } else {
        int body;
        float load[6];
        v = reflect_link(g, c, 26 - q, Fused ? collide_at(g, n) : load_moments(g.home_post, N, n),
                         Fused ? g.u : g.old_u, body, load);
        if (body >= 0)
#pragma unroll
          for (int e = 0; e < 6; ++e) {
            if (fabs((double)load[e] * kLoadScale) <= kFixedTermLimit)
              add_fixed(&block_loads[6 * body + e], to_fixed(load[e], kLoadScale));
            else
              block_bad[6 * body + e] = 1;
          }
      }
    }
    const float fx = (float)cx(q), fy = (float)cy(q), fz = (float)cz(q);
    MomentSums s;
    s.p = group_sum(v);
    s.jx = group_sum(fx * v);
    s.jy = group_sum(fy * v);
    s.jz = group_sum(fz * v);
    s.xx = group_sum(fx * fx * v);
    s.yy = group_sum(fy * fy * v);
    s.zz = group_sum(fz * fz * v);
    s.xy = group_sum(fx * fy * v);
    s.xz = group_sum(fx * fz * v);
    s.yz = group_sum(fy * fz * v);
    if (lane == 0) store_streamed(g, Fused ? g.home_post : g.home, n, s);
  }
  __syncthreads();
  for (int t = threadIdx.x; t < kLoadSlots; t += blockDim.x)
    g.partials[(size_t)blockIdx.x * kLoadSlots + t] =
        block_bad[t] ? __int_as_float(0x7fc00000) : (float)((double)block_loads[t] / kLoadScale);
}
// Adds the per-block load partials of k_stream_boundary to the loads: one
// block per load slot, fixed summation order.
__global__ void __launch_bounds__(256) k_finish_loads(icy3d_grid g, int blocks) {
  const int slot = blockIdx.x;
  float sum = 0.0f;
  for (int b = threadIdx.x; b < blocks; b += blockDim.x) sum += g.partials[(size_t)b * kLoadSlots + slot];
  sum = block_sum(sum);
  if (threadIdx.x == 0) (&g.control->loads[0][0])[slot] += sum;
}

__global__ void k_zero_loads(icy3d_grid g) {
  int t = threadIdx.x;
  if (t < ICY3D_MAX_BODIES * 6) (&g.control->loads[0][0])[t] = 0.0f;
}

// ---------------------------------------------------------------------------
// Probes (the reference tests' probe kernels).
__global__ void k_probe_home(const float* __restrict__ data, int rows, float* __restrict__ pops, float* __restrict__ post) {
  int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows) return;
  const float* d = data + 15 * r;
  Moments m;
#pragma unroll
  for (int t = 0; t < 10; ++t) m.m[t] = d[t];
  for (int q = 0; q < 27; ++q) pops[27 * r + q] = reconstruct_rt(q, m);
  Moments o = central_collision(m, d[10], d[11], d[12], d[13], d[14]);
#pragma unroll
  for (int t = 0; t < 10; ++t) post[10 * r + t] = o.m[t];
}
__global__ void k_probe_phase(const float* __restrict__ data, int rows, float mobility, float width, float* __restrict__ out) {
  int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows) return;
  const float* d = data + 14 * r;
  float h[7], post[7], fl[3];
#pragma unroll
  for (int q = 0; q < 7; ++q) h[q] = d[q];
  const float u[3] = {d[8], d[9], d[10]}, nrm[3] = {d[11], d[12], d[13]};
  phase_collision(h, d[7], u, nrm, mobility, width, post, fl);
#pragma unroll
  for (int q = 0; q < 7; ++q) out[10 * r + q] = post[q];
#pragma unroll
  for (int a = 0; a < 3; ++a) out[10 * r + 7 + a] = fl[a];
}
__global__ void k_probe_viscosity(const float* phi, int n_phi, const float* temps, int n_t, float rho_w, float rho_a,
                                  float mu_air, float* out) {
  int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n_phi * n_t) return;
  int i = r / n_t, t = r % n_t;
  out[r] = mixture_nu(phi[i], temps[t], rho_w, rho_a, mu_air);
}
__global__ void k_probe_stress_velocity(icy3d_grid g, int i, int j, int k, int dx, int dy, int dz, float* out) {
  if (threadIdx.x != 0) return;
  stress_neighbor_velocity(g, i, j, k, dx, dy, dz, out);
}
__global__ void k_probe_mirror(icy3d_grid g, int i, int j, int k, int dx, int dy, int dz, float* out) {
  if (threadIdx.x != 0) return;
  ice_mirror_point(g, i, j, k, i + dx, j + dy, k + dz, out);
  out[3] = wall_phase_sample(g, i, j, k, dx, dy, dz);
}

}  // namespace icy

// ===========================================================================
// C ABI
using namespace icy;

// ---------------------------------------------------------------------------
// Scratch of the allocation-free flow step (icy3d_flow_step_static): the
// block partial sums every flow kernel otherwise keeps in the caller's
// g.partials.  One copy per GPU, for the life of the process; its size
// covers grids of up to kScratchCells cells with ICY3D_MAX_BODIES bodies.
constexpr int kScratchCells = 1 << 24;
constexpr int kScratchFloats = 3 * (kScratchCells / kBlock);
static_assert(kScratchFloats >= (int)(kListBlocks * kLoadSlots), "scratch too small for the stream's load slots");
static_assert(kScratchFloats >= 2 * ((kScratchCells + kCompactCells - 1) / kCompactCells), "scratch too small");
static __device__ __align__(256) float scratch[kScratchFloats];

namespace {
// The device address of `scratch` on the current device, looked up once per
// device with hipGetSymbolAddress (each GPU holds its own copy) and kept.
constexpr int kScratchDevices = 64;
float* scratch_by_device[kScratchDevices] = {};
std::mutex scratch_lock;
int scratch_address(float** out) {
  int device = -1;
  hipError_t err = hipGetDevice(&device);
  if (err != hipSuccess) return (int)err;
  if (device < 0 || device >= kScratchDevices) return ICY3D_ERR_ARGUMENT;
  std::lock_guard<std::mutex> hold(scratch_lock);
  if (!scratch_by_device[device]) {
    void* address = nullptr;
    err = hipGetSymbolAddress(&address, HIP_SYMBOL(scratch));
    if (err != hipSuccess) return (int)err;
    scratch_by_device[device] = static_cast<float*>(address);
  }
  *out = scratch_by_device[device];
  return 0;
}

Box full_box(const icy3d_grid& g) {
  Box b = {{0, 0, 0}, {g.nx, g.ny, g.nz}};
  return b;
}
// Boxes from the caller are clamped to the grid (lo inclusive, hi exclusive).
Box make_box(const int32_t lo[3], const int32_t hi[3]) {
  Box b;
  for (int a = 0; a < 3; ++a) {
    b.lo[a] = lo[a];
    b.hi[a] = hi[a];
  }
  return b;
}
Box clamp_box(const icy3d_grid& g, Box b) {
  const int shape[3] = {g.nx, g.ny, g.nz};
  for (int a = 0; a < 3; ++a) {
    b.lo[a] = b.lo[a] < 0 ? 0 : b.lo[a];
    b.hi[a] = b.hi[a] > shape[a] ? shape[a] : b.hi[a];
  }
  return b;
}
size_t box_cells(const Box& b) {
  long ex = b.hi[0] - b.lo[0], ey = b.hi[1] - b.lo[1], ez = b.hi[2] - b.lo[2];
  if (ex <= 0 || ey <= 0 || ez <= 0) return 0;
  return (size_t)ex * ey * ez;
}
size_t grid_cells(const icy3d_grid& g) { return (size_t)g.nx * g.ny * g.nz; }
bool valid(const icy3d_grid* g) {
  return g && g->nx > 0 && g->ny > 0 && g->nz > 0 && g->bodies >= 0 && g->bodies <= ICY3D_MAX_BODIES &&
         grid_cells(*g) < (size_t)INT32_MAX / 16 && g->control;
}

// A clamped box as a one-entry list (empty when the box is).
BoxList one_box(const icy3d_grid& g, const Box& b) {
  BoxList L;
  L.count = 0;
  L.first[0] = 0;
  if (box_cells(b)) (void)make_box_list(g, 1, b.lo, b.hi, L);
  return L;
}
int launch_classify_list(const icy3d_grid& g, const BoxList& L, hipStream_t s) {
  if (list_blocks(L)) k_classify<<<list_blocks(L), kBlock, 0, s>>>(g, L);
  ICY_LAUNCH_CHECK();
  return 0;
}
int launch_classify(const icy3d_grid& g, const Box& b, hipStream_t s) {
  return launch_classify_list(g, one_box(g, b), s);
}
int launch_lists(const icy3d_grid& g, hipStream_t s) {
  const unsigned blocks = (unsigned)((grid_cells(g) + kCompactCells - 1) / kCompactCells);
  if ((int)(2 * blocks) > g.partials_capacity) return ICY3D_ERR_ARGUMENT;
  k_count_flags<<<blocks, kBlock, 0, s>>>(g);
  k_scan_flag_counts<<<1, 1024, 0, s>>>(g, (int)blocks);
  k_scatter_flags<<<blocks, kBlock, 0, s>>>(g);
  ICY_LAUNCH_CHECK();
  return 0;
}
int launch_classify_all(const icy3d_grid& g, hipStream_t s) {
  int rc = launch_classify(g, full_box(g), s);
  return rc ? rc : launch_lists(g, s);
}
// Full-grid gradients use the ice list for the mirror path; box-limited
// refreshes test the flag per cell.
// Mirror gradients always run over the ice list (one code path, so a
// box refresh reproduces a full pass bit for bit); the box only filters.
// The tiled pass per box, then one pass over the ice list filtered by the
// boxes.  Overlapping boxes write the same values twice.
int launch_gradients_list(const icy3d_grid& g, const BoxList& L, hipStream_t s) {
  if (!L.count) return 0;
  // Slabs a block sweeps: 16 where that gives every CU its eight blocks, else
  // 8 or 4 (a slab is a serial step; two more are read for the halo): with 16
  // everywhere, and each label loaded at its use, 26 us at 256x128x128 and 15
  // at 24x20x16, this way 21 and 6.
  BoxList tiles = L;
  int slabs = 32;
  do {
    slabs /= 2;
    for (int m = 0; m < L.count; ++m) tiles.first[m + 1] = tiles.first[m] + grad_tiles(L.lo[m], L.hi[m], slabs);
  } while (slabs > 4 && tiles.first[L.count] < 2048);
  k_gradients_tiled<<<(unsigned)tiles.first[L.count], kGradJ * kGradK, 0, s>>>(g, tiles, slabs);
  k_gradients_general_list<<<kGradientListBlocks, kBlock, 0, s>>>(g, L);
  ICY_LAUNCH_CHECK();
  return 0;
}
int launch_gradients(const icy3d_grid& g, const Box& b, bool, hipStream_t s) {
  return launch_gradients_list(g, one_box(g, b), s);
}
int launch_forces(const icy3d_grid& g, int with_flux, int moment_pressure, hipStream_t s) {
  const StreamTiles T = stream_tiles(g, kForceThreads);
  k_forces_rows<<<stream_blocks(g, T), stream_threads(T), 0, s>>>(g, T, with_flux, moment_pressure);  // bulk and tank cells
  k_forces_general<<<kForceListBlocks, kBlock, 0, s>>>(g, with_flux, moment_pressure);
  ICY_LAUNCH_CHECK();
  return 0;
}
int launch_recover(const icy3d_grid& g, int parity, int recover_flow, hipStream_t s) {
  bool scan = recover_flow && g.check_stability;
  const unsigned blocks = icy_blocks(grid_cells(g));
  if ((int)blocks > g.partials_capacity) return ICY3D_ERR_ARGUMENT;
  if (scan && 3 * (int)blocks > g.partials_capacity) return ICY3D_ERR_ARGUMENT;
  k_recover_phase<<<blocks, kBlock, 0, s>>>(g, parity, recover_flow);
  k_fold_recovery<<<1, kFinishThreads, 0, s>>>(g, (int)blocks, scan ? 1 : 0);
  ICY_LAUNCH_CHECK();
  return 0;
}
template <bool Fused>
void launch_stream_rows(const icy3d_grid& g, hipStream_t s) {
  const StreamTiles T = stream_tiles(g, kStreamThreads);
  k_stream_rows<Fused><<<stream_blocks(g, T), stream_threads(T), 0, s>>>(g, T);
}
int launch_stream(const icy3d_grid& g, hipStream_t s) {
  if ((int)(kListBlocks * kLoadSlots) > g.partials_capacity) return ICY3D_ERR_ARGUMENT;
  launch_stream_rows<false>(g, s);
  k_stream_boundary<false><<<kListBlocks, kBlock, 0, s>>>(g);
  if (g.bodies > 0) k_finish_loads<<<g.bodies * 6, 256, 0, s>>>(g, (int)kListBlocks);
  ICY_LAUNCH_CHECK();
  return 0;
}
// The fused collide-stream: moments from g.home into g.home_post (the
// caller swaps the buffers), body loads cleared and accumulated.
int launch_collide_stream(const icy3d_grid& g, hipStream_t s) {
  if ((int)(kListBlocks * kLoadSlots) > g.partials_capacity) return ICY3D_ERR_ARGUMENT;
  launch_stream_rows<true>(g, s);
  k_stream_boundary<true><<<kListBlocks, kBlock, 0, s>>>(g);
  if (g.bodies > 0) k_finish_loads<<<g.bodies * 6, 256, 0, s>>>(g, (int)kListBlocks);
  ICY_LAUNCH_CHECK();
  return 0;
}
// g with home and home_post traded (the state after a fused collide-stream).
icy3d_grid swapped_home(const icy3d_grid& g) {
  icy3d_grid r = g;
  r.home = g.home_post;
  r.home_post = g.home;
  return r;
}
}  // namespace

namespace icy {
// The class refresh of icy3d_refill_gradients_boxes (none when ref_lo is
// NULL), then one gradient pass over the whole grid.
int refresh_classes_full_gradients(const icy3d_grid* g, int count, const int32_t* lo, const int32_t* hi,
                                   const int32_t ref_lo[3], const int32_t ref_hi[3], hipStream_t s) {
  if (ref_lo && ref_hi) {
    const Box ref = clamp_box(*g, make_box(ref_lo, ref_hi));
    int32_t clo[kMaxBoxes * 3], chi[kMaxBoxes * 3];
    for (int m = 0; m < count; ++m)
      for (int a = 0; a < 3; ++a) {
        clo[3 * m + a] = max(lo[3 * m + a] - 1, ref.lo[a]);
        chi[3 * m + a] = min(hi[3 * m + a] + 1, ref.hi[a]);
      }
    BoxList classes;
    if (!make_box_list(*g, count, clo, chi, classes)) return ICY3D_ERR_ARGUMENT;
    int rc = launch_classify_list(*g, classes, s);
    if (!rc) rc = launch_lists(*g, s);
    if (rc) return rc;
  }
  return launch_gradients(*g, full_box(*g), true, s);
}
}  // namespace icy

extern "C" {

int icy3d_copy_async(void* dst, const void* src, size_t bytes, void* stream) {
  if (!bytes) return 0;
  if (!dst || !src) return ICY3D_ERR_ARGUMENT;
  return (int)hipMemcpyAsync(dst, src, bytes, hipMemcpyDefault, (hipStream_t)stream);
}
// A blocking copy: asynchronous and followed by a synchronisation of the
// stream it took the 24x20x16 tank's eight steps from 1760 to 1950 us.
int icy3d_read_control(const icy3d_grid* g, icy3d_control* host, void* stream) {
  if (!valid(g) || !host) return ICY3D_ERR_ARGUMENT;
  return (int)hipMemcpyWithStream(host, g->control, sizeof(*host), hipMemcpyDeviceToHost, (hipStream_t)stream);
}
int icy3d_abi_sizes(int32_t* grid_bytes, int32_t* control_bytes) {
  *grid_bytes = (int32_t)sizeof(icy3d_grid);
  *control_bytes = (int32_t)sizeof(icy3d_control);
  return 0;
}

int icy3d_classify(const icy3d_grid* g, const int32_t lo[3], const int32_t hi[3], void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  int rc = launch_classify(*g, lo ? clamp_box(*g, make_box(lo, hi)) : full_box(*g), s);
  return rc ? rc : launch_lists(*g, s);
}
int icy3d_gradients(const icy3d_grid* g, const int32_t lo[3], const int32_t hi[3], void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  return launch_gradients(*g, lo ? clamp_box(*g, make_box(lo, hi)) : full_box(*g), lo == nullptr, (hipStream_t)stream);
}
int icy3d_refill_gradients_boxes(const icy3d_grid* g, int count, const int32_t* lo, const int32_t* hi,
                                 const int32_t ref_lo[3], const int32_t ref_hi[3], void* stream) {
  if (!valid(g) || !ref_lo || !ref_hi || count < 0 || count > kMaxBoxes || (count && (!lo || !hi)))
    return ICY3D_ERR_ARGUMENT;
  // Classes depend on labels one cell away, gradients on cells within the
  // dependency radius (gradients.py:15-20): only there, inside the reference
  // box, can the refreshed values differ from the stored ones.
  const Box ref = clamp_box(*g, make_box(ref_lo, ref_hi));
  int32_t clo[kMaxBoxes * 3], chi[kMaxBoxes * 3], glo[kMaxBoxes * 3], ghi[kMaxBoxes * 3];
  for (int m = 0; m < count; ++m)
    for (int a = 0; a < 3; ++a) {
      clo[3 * m + a] = max(lo[3 * m + a] - 1, ref.lo[a]);
      chi[3 * m + a] = min(hi[3 * m + a] + 1, ref.hi[a]);
      glo[3 * m + a] = max(lo[3 * m + a] - kGradientRadius, ref.lo[a]);
      ghi[3 * m + a] = min(hi[3 * m + a] + kGradientRadius, ref.hi[a]);
    }
  BoxList classes, gradients;
  if (!make_box_list(*g, count, clo, chi, classes) || !make_box_list(*g, count, glo, ghi, gradients))
    return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  int rc = launch_classify_list(*g, classes, s);
  if (!rc) rc = launch_lists(*g, s);
  return rc ? rc : launch_gradients_list(*g, gradients, s);
}
int icy3d_refill_gradients(const icy3d_grid* g, const int32_t lo[3], const int32_t hi[3], void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  Box b = clamp_box(*g, make_box(lo, hi));
  int rc = launch_classify(*g, b, s);
  if (!rc) rc = launch_lists(*g, s);
  return rc ? rc : launch_gradients(*g, b, false, s);
}
int icy3d_build_boundary_lists(const icy3d_grid* g, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  return launch_lists(*g, (hipStream_t)stream);
}
int icy3d_collide_phase(const icy3d_grid* g, int parity, int moving_walls, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  k_collide_phase<<<icy_blocks(grid_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g, parity, moving_walls ? 1 : 0);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_recover_phase(const icy3d_grid* g, int parity, int recover_flow, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  return launch_recover(*g, parity, recover_flow, (hipStream_t)stream);
}
int icy3d_phase_warmup(const icy3d_grid* g, int steps, int* parity, void* stream) {
  if (!valid(g) || !parity || steps < 0) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  Box b = full_box(*g);
  const unsigned blocks = icy_blocks(grid_cells(*g));
  // Labels do not change during the warm-up: classify once.
  int rc0 = launch_classify_all(*g, s);
  if (rc0) return rc0;
  for (int t = 0; t < steps; ++t) {
    int rc = launch_gradients(*g, b, true, s);
    if (rc) return rc;
    k_collide_phase<<<blocks, kBlock, 0, s>>>(*g, *parity, 0);
    *parity = 1 - *parity;
    rc = launch_recover(*g, *parity, 0, s);
    if (rc) return rc;
  }
  return 0;
}
int icy3d_recover_pressure(const icy3d_grid* g, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  k_recover_pressure<<<icy_blocks(grid_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_scan_stability(const icy3d_grid* g, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  k_reset_stability<<<1, 1, 0, s>>>(*g);
  k_scan_stability<<<icy_blocks(grid_cells(*g)), kBlock, 0, s>>>(*g);
  k_fold_peak<<<1, 1, 0, s>>>(*g);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_forces(const icy3d_grid* g, int with_flux, int moment_pressure, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  int rc = launch_classify_all(*g, s);
  return rc ? rc : launch_forces(*g, with_flux, moment_pressure, s);
}
int icy3d_collide_momentum(const icy3d_grid* g, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  k_collide_momentum<<<icy_blocks(grid_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g, 0);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_stream_home(const icy3d_grid* g, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  return launch_stream(*g, (hipStream_t)stream);
}
int icy3d_collide_stream_home(const icy3d_grid* g, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  return launch_collide_stream(*g, (hipStream_t)stream);
}
int icy3d_flow_step_profiled(const icy3d_grid* g, int parity, int refresh_gradients, int classify,
                             icy3d_profile* prof, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  const icy3d_grid& G = *g;
  const unsigned blocks = icy_blocks(grid_cells(G));
  Box b = full_box(G);
  int rc = 0;
  auto mark = [&](int event) {
    if (prof) (void)hipEventRecord(prof->events[event], s);
  };
  if (classify || refresh_gradients) {
    rc = launch_classify_all(G, s);
    if (rc) return rc;
  }
  if (refresh_gradients) {
    rc = launch_gradients(G, b, true, s);
    if (rc) return rc;
  }
  mark(0);
  k_collide_phase<<<blocks, kBlock, 0, s>>>(G, parity, 2);
  parity = 1 - parity;
  mark(1);
  rc = launch_forces(G, 1, 1, s);
  if (rc) return rc;
  mark(2);
  rc = launch_collide_stream(G, s);
  mark(3);
  const icy3d_grid H = swapped_home(G);  // the streamed moments
  if (!rc) rc = launch_recover(H, parity, 1, s);
  mark(4);
  if (!rc) rc = launch_gradients(H, b, true, s);
  mark(5);
  if (prof) prof->pending = 1;
  return rc;
}
int icy3d_flow_step(const icy3d_grid* g, int parity, int refresh_gradients, int classify, void* stream) {
  return icy3d_flow_step_profiled(g, parity, refresh_gradients, classify, nullptr, stream);
}
// The same launches in two parts: everything up to the stream (after which
// the body loads in the control block are final), then recovery and the
// gradients.  A caller copies the loads out between the two and integrates
// the rigid bodies on the host while the second part runs.
int icy3d_flow_step_begin(const icy3d_grid* g, int parity, int refresh_gradients, int classify, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  const icy3d_grid& G = *g;
  const unsigned blocks = icy_blocks(grid_cells(G));
  int rc = 0;
  if (classify || refresh_gradients) {
    rc = launch_classify_all(G, s);
    if (rc) return rc;
  }
  if (refresh_gradients) {
    rc = launch_gradients(G, full_box(G), true, s);
    if (rc) return rc;
  }
  k_collide_phase<<<blocks, kBlock, 0, s>>>(G, parity, 2);
  rc = launch_forces(G, 1, 1, s);
  if (rc) return rc;
  return launch_collide_stream(G, s);
}
int icy3d_flow_step_end(const icy3d_grid* g, int parity, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  int rc = launch_recover(*g, 1 - parity, 1, s);
  if (!rc) rc = launch_gradients(*g, full_box(*g), true, s);
  return rc;
}
int icy3d_flow_step_recover(const icy3d_grid* g, int parity, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  return launch_recover(*g, 1 - parity, 1, (hipStream_t)stream);
}
int icy3d_profile_create(icy3d_profile** out) {
  if (!out) return ICY3D_ERR_ARGUMENT;
  icy3d_profile* p = new icy3d_profile();
  for (int e = 0; e <= ICY3D_PROFILE_GROUPS; ++e) {
    hipError_t err = hipEventCreate(&p->events[e]);
    if (err != hipSuccess) {
      for (int k = 0; k < e; ++k) (void)hipEventDestroy(p->events[k]);
      delete p;
      return (int)err;
    }
  }
  *out = p;
  return 0;
}
int icy3d_profile_destroy(icy3d_profile* p) {
  if (!p) return 0;
  for (int e = 0; e <= ICY3D_PROFILE_GROUPS; ++e) (void)hipEventDestroy(p->events[e]);
  delete p;
  return 0;
}
int icy3d_profile_collect(icy3d_profile* p) {
  if (!p) return ICY3D_ERR_ARGUMENT;
  if (!p->pending) return 0;
  hipError_t err = hipEventSynchronize(p->events[ICY3D_PROFILE_GROUPS]);
  if (err != hipSuccess) return (int)err;
  for (int k = 0; k < ICY3D_PROFILE_GROUPS; ++k) {
    float ms = 0.0f;
    err = hipEventElapsedTime(&ms, p->events[k], p->events[k + 1]);
    if (err != hipSuccess) return (int)err;
    p->total_ms[k] += ms;
  }
  p->count += 1;
  p->pending = 0;
  return 0;
}
int icy3d_profile_read(const icy3d_profile* p, double* total_ms, int64_t* count) {
  if (!p || !total_ms || !count) return ICY3D_ERR_ARGUMENT;
  for (int k = 0; k < ICY3D_PROFILE_GROUPS; ++k) total_ms[k] = p->total_ms[k];
  *count = p->count;
  return 0;
}
int icy3d_repair_phase_layout_boxes(const icy3d_grid* g, int parity, int count, const int32_t* lo, const int32_t* hi,
                                    void* stream) {
  BoxList L;
  if (!valid(g) || !make_box_list(*g, count, lo, hi, L)) return ICY3D_ERR_ARGUMENT;
  if (!parity) return 0;
  if (list_blocks(L)) k_repair_layout<<<list_blocks(L), kBlock, 0, (hipStream_t)stream>>>(*g, L);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_repair_phase_layout(const icy3d_grid* g, int parity, const int32_t lo[3], const int32_t hi[3],
                              void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  const Box b = lo ? clamp_box(*g, make_box(lo, hi)) : full_box(*g);
  if (!box_cells(b)) return 0;
  return icy3d_repair_phase_layout_boxes(g, parity, 1, b.lo, b.hi, stream);
}
int icy3d_export_phase(const icy3d_grid* g, int parity, float* out, void* stream) {
  if (!valid(g) || !out) return ICY3D_ERR_ARGUMENT;
  k_export_phase<<<icy_blocks(grid_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g, parity, out);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_project_refill(const icy3d_grid* g, int parity, const int32_t lo[3], const int32_t hi[3], void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  Box b = clamp_box(*g, make_box(lo, hi));
  size_t n = box_cells(b);
  if (!n) return 0;
  hipStream_t s = (hipStream_t)stream;
  k_refill_forces<<<icy_blocks(n), kBlock, 0, s>>>(*g, b);
  k_refill_equilibrium<<<icy_blocks(n), kBlock, 0, s>>>(*g, b, parity);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_seed_populations(const icy3d_grid* g, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  k_set_equilibrium<<<icy_blocks(grid_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g, 0, 0, 1, 0, 0.0f);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_set_equilibrium_all(const icy3d_grid* g, int parity, int with_phase, int use_constant_pressure,
                              float pressure, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  k_set_equilibrium<<<icy_blocks(grid_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g, parity, with_phase, 0,
                                                                                   use_constant_pressure, pressure);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_capillary_stress(const icy3d_grid* g, float* out, void* stream) {
  if (!valid(g) || !out) return ICY3D_ERR_ARGUMENT;
  k_capillary_stress<<<icy_blocks(grid_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g, out);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_generic_forces(const icy3d_grid* g, float* out, void* stream) {
  if (!valid(g) || !out) return ICY3D_ERR_ARGUMENT;
  k_generic_forces<<<icy_blocks(grid_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g, out);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_write_gradient_all(const icy3d_grid* g, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  k_write_gradient_all<<<icy_blocks(grid_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_probe_home(const float* data, int rows, float* populations, float* collided, void* stream) {
  if (!data || rows < 0 || !populations || !collided) return ICY3D_ERR_ARGUMENT;
  if (rows) k_probe_home<<<icy_blocks(rows), kBlock, 0, (hipStream_t)stream>>>(data, rows, populations, collided);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_probe_phase(const float* data, int rows, float mobility, float width, float* out, void* stream) {
  if (!data || rows < 0 || !out) return ICY3D_ERR_ARGUMENT;
  if (rows) k_probe_phase<<<icy_blocks(rows), kBlock, 0, (hipStream_t)stream>>>(data, rows, mobility, width, out);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_probe_viscosity(const float* phi, int n_phi, const float* temps, int n_t, float rho_w, float rho_a,
                          float mu_air, float* out, void* stream) {
  if (!phi || !temps || !out || n_phi < 0 || n_t < 0) return ICY3D_ERR_ARGUMENT;
  int total = n_phi * n_t;
  if (total)
    k_probe_viscosity<<<icy_blocks(total), kBlock, 0, (hipStream_t)stream>>>(phi, n_phi, temps, n_t, rho_w, rho_a,
                                                                             mu_air, out);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_probe_stress_velocity(const icy3d_grid* g, const int32_t cell[3], const int32_t c[3], float* out,
                                void* stream) {
  if (!valid(g) || !out) return ICY3D_ERR_ARGUMENT;
  // The probe reads the cell and its two link neighbours: keep all inside.
  for (int a = 0; a < 3; ++a) {
    int extent = a == 0 ? g->nx : (a == 1 ? g->ny : g->nz);
    if (cell[a] - 1 < 0 || cell[a] + 1 >= extent || c[a] < -1 || c[a] > 1) return ICY3D_ERR_ARGUMENT;
  }
  k_probe_stress_velocity<<<1, 64, 0, (hipStream_t)stream>>>(*g, cell[0], cell[1], cell[2], c[0], c[1], c[2], out);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_probe_mirror(const icy3d_grid* g, const int32_t cell[3], const int32_t c[3], float* out, void* stream) {
  if (!valid(g) || !out) return ICY3D_ERR_ARGUMENT;
  for (int a = 0; a < 3; ++a) {
    int extent = a == 0 ? g->nx : (a == 1 ? g->ny : g->nz);
    if (cell[a] - 1 < 0 || cell[a] + 1 >= extent || c[a] < -1 || c[a] > 1) return ICY3D_ERR_ARGUMENT;
  }
  k_probe_mirror<<<1, 64, 0, (hipStream_t)stream>>>(*g, cell[0], cell[1], cell[2], c[0], c[1], c[2], out);
  ICY_LAUNCH_CHECK();
  return 0;
}

int icy3d_flow_step_static(const icy3d_grid* g, int parity, int refresh_gradients, int classify, void* stream) {
  if (!valid(g)) return ICY3D_ERR_ARGUMENT;
  if (grid_cells(*g) > (size_t)kScratchCells) return ICY3D_ERR_SCRATCH;
  float* device_scratch = nullptr;
  if (const int rc = scratch_address(&device_scratch)) return rc;
  icy3d_grid G = *g;
  G.partials = device_scratch;
  G.partials_capacity = kScratchFloats;
  return icy3d_flow_step(&G, parity, refresh_gradients, classify, stream);
}
int64_t icy3d_flow_step_static_max_cells(void) { return kScratchCells; }

}  // extern "C"

#ifndef ICY_SOURCE_HASH
#define ICY_SOURCE_HASH "unrecorded"
#endif
extern "C" const char* icy3d_source_hash(void) { return ICY_SOURCE_HASH; }
