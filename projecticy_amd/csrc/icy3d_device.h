// Device helpers shared by the icy3d HIP translation units (gfx950 only).
//
// Lattice conventions follow the reference (iceflow3d/lattice.py:11-46):
// D3Q27 direction q = 9(cx+1) + 3(cy+1) + (cz+1), rest q = 13, weights
// rounded once per order (8/27, 2/27, 1/54, 1/216); D3Q7 order
// 0,+x,-x,+y,-y,+z,-z (phase.py:15-24).  Populations are never stored: the
// HOME moments (p*, u, S) are reconstructed per direction in registers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/icy3d.h"

namespace icy {

constexpr int kBlock = 256;

__host__ __device__ constexpr int cx(int q) { return q / 9 - 1; }
__host__ __device__ constexpr int cy(int q) { return q / 3 % 3 - 1; }
__host__ __device__ constexpr int cz(int q) { return q % 3 - 1; }
__host__ __device__ constexpr int order(int q) {
  return (cx(q) != 0) + (cy(q) != 0) + (cz(q) != 0);
}
__host__ __device__ constexpr float w27(int q) {
  return order(q) == 0 ? 8.0f / 27.0f : (order(q) == 1 ? 2.0f / 27.0f : (order(q) == 2 ? 1.0f / 54.0f : 1.0f / 216.0f));
}

constexpr int kC7[7][3] = {{0, 0, 0}, {1, 0, 0}, {-1, 0, 0}, {0, 1, 0}, {0, -1, 0}, {0, 0, 1}, {0, 0, -1}};
__host__ __device__ constexpr int opp7(int q) { return q == 0 ? 0 : (q % 2 == 1 ? q + 1 : q - 1); }

struct Cell {
  int i, j, k, n;
};

__device__ __forceinline__ Cell cell_of(const icy3d_grid& g, int n) {
  Cell c;
  c.n = n;
  c.k = n % g.nz;
  int t = n / g.nz;
  c.j = t % g.ny;
  c.i = t / g.ny;
  return c;
}
__device__ __forceinline__ int lin(const icy3d_grid& g, int i, int j, int k) { return (i * g.ny + j) * g.nz + k; }
__device__ __forceinline__ bool inside(const icy3d_grid& g, int i, int j, int k) {
  return (unsigned)i < (unsigned)g.nx && (unsigned)j < (unsigned)g.ny && (unsigned)k < (unsigned)g.nz;
}
__device__ __forceinline__ bool fluid_at(const icy3d_grid& g, int i, int j, int k) {
  return inside(g, i, j, k) && g.id[lin(g, i, j, k)] == -1;
}
__device__ __forceinline__ size_t cells(const icy3d_grid& g) { return (size_t)g.nx * g.ny * g.nz; }
// A launch of icy3d_refresh_begin_boxes after a stability scan that found an
// invalid cell: the kernel leaves every field as it is.
__device__ __forceinline__ bool refresh_halted(const icy3d_grid& g) {
  return g.refresh_guard && g.control->invalid_index < (int)cells(g);
}

__device__ __forceinline__ float clamp01(float v) { return fminf(1.0f, fmaxf(0.0f, v)); }
__device__ __forceinline__ float density(const icy3d_grid& g, float phi) {
  return g.rho_air + (1.0f - g.rho_air) * clamp01(phi);
}

// IAPWS-style water viscosity, lattice.py:131-137, as 1e-6 sum c t^e with
// t^e evaluated as exp2(e log2 t) (one log, four exponentials).
__device__ __forceinline__ float water_mu(float t_c) {
  float lt = log2f((t_c + 273.15f) / 300.0f);
  return 1e-6f * (280.68f * exp2f(-1.9f * lt) + 511.45f * exp2f(-7.7f * lt) + 61.131f * exp2f(-19.6f * lt) +
                  0.45903f * exp2f(-40.0f * lt));
}
// lattice.py:49-55
__device__ __forceinline__ float mixture_nu(float phi, float t_c, float rho_w, float rho_a, float mu_air) {
  float f = clamp01(phi);
  float mu = f * water_mu(t_c) + (1.0f - f) * mu_air;
  float rho = f * rho_w + (1.0f - f) * rho_a;
  return mu / rho;
}
// thermal.py:71-78
__device__ __forceinline__ float water_temperature(const icy3d_grid& g, int n) {
  float v = g.water_volume[n];
  return v > 1e-30f ? g.tm + g.water_energy[n] / (g.rho_cp * v) : g.air_t;
}
__device__ __forceinline__ float water_temperature_of(const icy3d_grid& g, float volume, float energy) {
  return volume > 1e-30f ? g.tm + energy / (g.rho_cp * volume) : g.air_t;
}
// The HOME shear relaxation rate s = 1 / (1/2 + 3 nu) of home.py:199-211
// from a cell's phase, water volume and water energy.
__device__ __forceinline__ float home_shear_rate(const icy3d_grid& g, float phi, float volume, float energy) {
  const float nu = mixture_nu(phi, water_temperature_of(g, volume, energy), g.rho_water_si, g.rho_air_si, g.mu_air) *
                   g.nu_scale;
  return 1.0f / (0.5f + 3.0f * nu);
}
__device__ __forceinline__ float lattice_nu(const icy3d_grid& g, int n) {
  return mixture_nu(g.phi[n], water_temperature(g, n), g.rho_water_si, g.rho_air_si, g.mu_air) * g.nu_scale;
}

// HOME moment vector: p*, u(3), Sxx, Syy, Szz, Sxy, Sxz, Syz (home.py:16-27).
struct Moments {
  float m[10];
};

__device__ __forceinline__ Moments load_moments(const float* __restrict__ base, size_t stride, int n) {
  Moments r;
#pragma unroll
  for (int t = 0; t < 10; ++t) r.m[t] = base[t * stride + n];
  return r;
}
__device__ __forceinline__ void store_moments(float* __restrict__ base, size_t stride, int n, const Moments& r) {
#pragma unroll
  for (int t = 0; t < 10; ++t) base[t * stride + n] = r.m[t];
}

// Third-order filtered reconstruction of direction (x,y,z), home.py:30-53,
// with the direction known at compile time so every c-product folds.
template <int X, int Y, int Z>
__device__ __forceinline__ float reconstruct_c(const Moments& M) {
  const float p = M.m[0], ux = M.m[1], uy = M.m[2], uz = M.m[3];
  const float sxx = M.m[4], syy = M.m[5], szz = M.m[6], sxy = M.m[7], sxz = M.m[8], syz = M.m[9];
  constexpr float fx = X, fy = Y, fz = Z;
  float cu = fx * ux + fy * uy + fz * uz;
  float csc = fx * fx * sxx + fy * fy * syy + fz * fz * szz + 2.0f * (fx * fy * sxy + fx * fz * sxz + fy * fz * syz);
  float value = p + 3.0f * cu + 4.5f * (csc - (sxx + syy + szz) * (1.0f / 3.0f));
  // sum over ordered pairs a != b of (c_a^2 - 1/3) c_b (S_aa u_b + 2 S_ab u_a - 2 u_a^2 u_b)
  float third = 0.0f;
  constexpr float ax = fx * fx - 1.0f / 3.0f, ay = fy * fy - 1.0f / 3.0f, az = fz * fz - 1.0f / 3.0f;
  if (Y != 0) third += ax * fy * (sxx * uy + 2.0f * sxy * ux - 2.0f * ux * ux * uy);
  if (Z != 0) third += ax * fz * (sxx * uz + 2.0f * sxz * ux - 2.0f * ux * ux * uz);
  if (X != 0) third += ay * fx * (syy * ux + 2.0f * sxy * uy - 2.0f * uy * uy * ux);
  if (Z != 0) third += ay * fz * (syy * uz + 2.0f * syz * uy - 2.0f * uy * uy * uz);
  if (X != 0) third += az * fx * (szz * ux + 2.0f * sxz * uz - 2.0f * uz * uz * ux);
  if (Y != 0) third += az * fy * (szz * uy + 2.0f * syz * uz - 2.0f * uz * uz * uy);
  if (X != 0 && Y != 0 && Z != 0)
    third += 2.0f * fx * fy * fz * (sxz * uy + syz * ux + sxy * uz - 2.0f * ux * uy * uz);
  constexpr float w = (X != 0) + (Y != 0) + (Z != 0) == 0   ? 8.0f / 27.0f
                      : (X != 0) + (Y != 0) + (Z != 0) == 1 ? 2.0f / 27.0f
                      : (X != 0) + (Y != 0) + (Z != 0) == 2 ? 1.0f / 54.0f
                                                            : 1.0f / 216.0f;
  return w * (value + 13.5f * third);
}
template <int Q>
__device__ __forceinline__ float reconstruct(const Moments& M) {
  return reconstruct_c<cx(Q), cy(Q), cz(Q)>(M);
}

// Runtime-direction reconstruction for the rare boundary paths.
__device__ __noinline__ float reconstruct_rt(int q, const Moments& M);

// home.py:56-58
__device__ __forceinline__ Moments equilibrium_moments(float p, float ux, float uy, float uz) {
  Moments r;
  r.m[0] = p;
  r.m[1] = ux;
  r.m[2] = uy;
  r.m[3] = uz;
  r.m[4] = ux * ux;
  r.m[5] = uy * uy;
  r.m[6] = uz * uz;
  r.m[7] = ux * uy;
  r.m[8] = ux * uz;
  r.m[9] = uy * uz;
  return r;
}

// home.py:61-78: forced central-moment collision of the HOME moments.
__device__ __forceinline__ Moments central_collision(const Moments& M, float ax, float ay, float az, float rate,
                                                     float bulk) {
  const float u[3] = {M.m[1] + 0.5f * ax, M.m[2] + 0.5f * ay, M.m[3] + 0.5f * az};
  const float a[3] = {ax, ay, az};
  // S in (xx, yy, zz, xy, xz, yz) order
  const int ia[6] = {0, 1, 2, 0, 0, 1}, ib[6] = {0, 1, 2, 1, 2, 2};
  float R[6], F[6], uu[6];
#pragma unroll
  for (int t = 0; t < 6; ++t) {
    uu[t] = u[ia[t]] * u[ib[t]];
    R[t] = M.m[4 + t] - uu[t];
    F[t] = a[ia[t]] * u[ib[t]] + u[ia[t]] * a[ib[t]];
  }
  const float tr_r = (R[0] + R[1] + R[2]) * (1.0f / 3.0f);
  const float tr_f = (F[0] + F[1] + F[2]) * (1.0f / 3.0f);
  const float keep_shear = 1.0f - rate, keep_bulk = 1.0f - bulk;
  const float force_shear = 1.0f - 0.5f * rate, force_bulk = 1.0f - 0.5f * bulk;
  Moments out;
  out.m[0] = M.m[0];
  out.m[1] = M.m[1] + ax;
  out.m[2] = M.m[2] + ay;
  out.m[3] = M.m[3] + az;
#pragma unroll
  for (int t = 0; t < 3; ++t)
    out.m[4 + t] = uu[t] + keep_shear * (R[t] - tr_r) + keep_bulk * tr_r + force_shear * (F[t] - tr_f) +
                   force_bulk * tr_f;
#pragma unroll
  for (int t = 3; t < 6; ++t) out.m[4 + t] = uu[t] + keep_shear * R[t] + force_shear * F[t];
  return out;
}

// phase.py:38-60: D3Q7 CM-MRT Allen-Cahn collision.
__device__ __forceinline__ void phase_collision(const float h[7], float phi, const float u[3], const float n[3],
                                                float mobility, float width, float post[7], float flux[3]) {
  const float rate = 1.0f / (0.5f + 4.0f * mobility);
  float second_sum = 0.0f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    float first = h[2 * a + 1] - h[2 * a + 2];
    float source = phi * (1.0f - phi) / width * n[a];
    float delta = (1.0f - rate) * (first - phi * u[a]) + (1.0f - 0.5f * rate) * source;
    float j = phi * u[a] + delta;
    float second = phi * 0.25f + 2.0f * u[a] * (delta - 0.5f * source);
    post[2 * a + 1] = 0.5f * (second + j);
    post[2 * a + 2] = 0.5f * (second - j);
    flux[a] = 0.5f * (first + j) - phi * u[a];
    second_sum += second;
  }
  post[0] = phi - second_sum;
}
__device__ __forceinline__ float phase_equilibrium7(int q, float phi, float ux, float uy, float uz) {
  float w = q == 0 ? 0.25f : 0.125f;
  return w * phi * (1.0f + 4.0f * (kC7[q][0] * ux + kC7[q][1] * uy + kC7[q][2] * uz));
}

// Body state row: origin[3], R[9] (row-major), centre[3], v[3], omega[3].
__device__ __forceinline__ const float* body_row(const icy3d_grid& g, int b) { return g.body + ICY3D_STATE_STRIDE * b; }
// simulator.py:253-257
__device__ __forceinline__ void body_velocity_at(const icy3d_grid& g, float px, float py, float pz, int b, float out[3]) {
  const float* s = body_row(g, b);
  float rx = px - s[12], ry = py - s[13], rz = pz - s[14];
  const float* v = s + 15;
  const float* w = s + 18;
  out[0] = v[0] + (w[1] * rz - w[2] * ry);
  out[1] = v[1] + (w[2] * rx - w[0] * rz);
  out[2] = v[2] + (w[0] * ry - w[1] * rx);
}
// simulator.py:217-223: world point -> material-grid coordinates of body b.
__device__ __forceinline__ void material_grid(const icy3d_grid& g, float px, float py, float pz, int b, float out[3]) {
  const float* s = body_row(g, b);
  float dx = px - s[0], dy = py - s[1], dz = pz - s[2];
  const int* size = g.material_size + 3 * b;
#pragma unroll
  for (int a = 0; a < 3; ++a)
    out[a] = (s[3 + a] * dx + s[6 + a] * dy + s[9 + a] * dz) + 0.5f * (float)size[a] - 0.5f;
}
__device__ __forceinline__ size_t mat_index(const icy3d_grid& g, int b, int i, int j, int k) {
  return (((size_t)b * g.mx + i) * g.my + j) * g.mz + k;
}
__device__ __forceinline__ bool mat_inside(const icy3d_grid& g, int b, int i, int j, int k) {
  const int* s = g.material_size + 3 * b;
  return (unsigned)i < (unsigned)s[0] && (unsigned)j < (unsigned)s[1] && (unsigned)k < (unsigned)s[2];
}
// thermal.py:80-86
__device__ __forceinline__ float ice_temperature(const icy3d_grid& g, int b, int i, int j, int k) {
  size_t m = mat_index(g, b, i, j, k);
  float mass = g.material_mass[m];
  float t = g.tm;
  if (mass > 1e-30f) t += g.material_energy[m] / (g.cp_ice * mass);
  return t;
}

// gradients.py:48-58 (shared by mirror sampling and population reflection)
__device__ __forceinline__ float link_fraction(const icy3d_grid& g, int n_i, int n_j) {
  float ci = g.coverage[n_i], cj = g.coverage[n_j];
  return fminf(0.95f, fmaxf(0.05f, (g.threshold - ci) / fmaxf(cj - ci, 1e-6f)));
}

// ---- wave-level reductions (wave64) ---------------------------------------
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ int wave_min_int(int v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ int wave_max_int(int v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ int wave_sum_int(int v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}
__device__ __forceinline__ bool wave_leader() { return (threadIdx.x & 63) == 0; }
// Non-negative float max through the ordered integer image; the relaxed
// pre-read skips the atomic once the running maximum is already larger, so
// a full-grid reduction issues only a handful of atomics.
__device__ __forceinline__ void atomic_max_nonneg(float* address, float value) {
  if (value > *reinterpret_cast<volatile float*>(address))
    atomicMax(reinterpret_cast<int*>(address), __float_as_int(value));
}

// Block-wide sum (blockDim.x a multiple of 64, at most 1024); every thread
// of the block must call it.  The result is valid in thread 0 only.
// Block-wide maximum / minimum; the result is valid in thread 0.
__device__ __forceinline__ float block_max(float v) {
  __shared__ float wave_part[16];
  v = wave_max(v);
  if ((threadIdx.x & 63) == 0) wave_part[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = v;
  if (threadIdx.x == 0)
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r = fmaxf(r, wave_part[w]);
  __syncthreads();
  return r;
}
__device__ __forceinline__ int block_min_int(int v) {
  __shared__ int wave_part[16];
  v = wave_min_int(v);
  if ((threadIdx.x & 63) == 0) wave_part[threadIdx.x >> 6] = v;
  __syncthreads();
  int r = v;
  if (threadIdx.x == 0)
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r = min(r, wave_part[w]);
  __syncthreads();
  return r;
}
__device__ __forceinline__ float block_sum(float v) {
  __shared__ float wave_part[16];
  v = wave_sum(v);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) wave_part[wave] = v;
  __syncthreads();
  float total = 0.0f;
  if (threadIdx.x == 0)
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) total += wave_part[w];
  __syncthreads();
  return total;
}

}  // namespace icy

namespace {
// Second stage of a deterministic sum: one block folds the per-block
// partials in a fixed order and adds the total to *target.
// Four loads are in flight per thread per round.
constexpr int kFinishThreads = 1024;
// The fold itself (blockDim.x == kFinishThreads); the total is valid in
// thread 0.
__device__ __forceinline__ float finish_total(const float* __restrict__ partials, int count) {
  float v = 0.0f;
  int t = threadIdx.x;
  for (; t + 3 * kFinishThreads < count; t += 4 * kFinishThreads) {
    const float a = partials[t], b = partials[t + kFinishThreads];
    const float c = partials[t + 2 * kFinishThreads], d = partials[t + 3 * kFinishThreads];
    v += (a + b) + (c + d);
  }
  for (; t < count; t += kFinishThreads) v += partials[t];
  return icy::block_sum(v);
}
__global__ void __launch_bounds__(kFinishThreads) k_finish_sum(const float* __restrict__ partials, int count,
                                                              float* target) {
  const float total = finish_total(partials, count);
  if (threadIdx.x == 0) *target += total;
}
}  // namespace

namespace icy {

// Grid-stride iteration over a device-resident cell list.
#define ICY_FOR_LIST(list, count_expr, var)                                                       \
  for (int _t = blockIdx.x * blockDim.x + threadIdx.x, _count = (count_expr); _t < _count;       \
       _t += gridDim.x * blockDim.x)                                                              \
    if (const int var = (list)[_t]; true)

constexpr unsigned kListBlocks = 1024;
// Boundary kernels give each listed cell a group of 32 lanes, one lane per
// D3Q27 direction (lanes 27..31 idle), and reduce within the group.
constexpr int kCellLanes = 32;
__device__ __forceinline__ float group_sum(float v) {
#pragma unroll
  for (int off = kCellLanes / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kCellLanes);
  return v;
}
__device__ __forceinline__ int block_sum_int(int v) {
  __shared__ int wave_part_int[16];
  v = wave_sum_int(v);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) wave_part_int[wave] = v;
  __syncthreads();
  int total = 0;
  if (threadIdx.x == 0)
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) total += wave_part_int[w];
  __syncthreads();
  return total;
}
// Partial load slots written by each boundary-stream block.
constexpr int kLoadSlots = ICY3D_MAX_BODIES * 6;

// Fixed-point accumulation for scatters whose targets collect contributions
// from many threads.  Integer addition is associative, so the total does not
// depend on the order in which the atomics land and a step repeats bit for
// bit.  A contribution is rounded to a multiple of 1/scale; the caller keeps
// |contribution * scale| at most kFixedTermLimit, so the sum of up to 2^10
// such terms stays inside an int64.
constexpr double kFixedTermLimit = 0x1p52;
__device__ __forceinline__ long long to_fixed(double value, double scale) { return __double2ll_rn(value * scale); }
__device__ __forceinline__ void add_fixed(long long* sum, long long q) {
  atomicAdd(reinterpret_cast<unsigned long long*>(sum), static_cast<unsigned long long>(q));
}

}  // namespace icy

#define ICY_LAUNCH_CHECK()                         \
  do {                                             \
    hipError_t _e = hipGetLastError();             \
    if (_e != hipSuccess) return static_cast<int>(_e); \
  } while (0)

inline unsigned icy_blocks(size_t count) {
  return static_cast<unsigned>((count + icy::kBlock - 1) / icy::kBlock);
}

namespace icy {
// Disjoint cell boxes covered by one launch of kBlock-thread blocks: box b
// owns blocks [first[b], first[b + 1]), so a block's box is uniform.
constexpr int kMaxBoxes = ICY3D_MAX_BODIES + 1;
struct BoxList {
  int count;
  int first[kMaxBoxes + 1];
  int lo[kMaxBoxes][3], hi[kMaxBoxes][3];
};
__device__ __forceinline__ bool list_cell(const icy3d_grid& g, const BoxList& L, Cell& c) {
  int b = 0;
  while (b + 1 < L.count && (int)blockIdx.x >= L.first[b + 1]) ++b;
  const int t = ((int)blockIdx.x - L.first[b]) * (int)blockDim.x + (int)threadIdx.x;
  const int ex = L.hi[b][0] - L.lo[b][0], ey = L.hi[b][1] - L.lo[b][1], ez = L.hi[b][2] - L.lo[b][2];
  if (t >= ex * ey * ez) return false;
  c.k = L.lo[b][2] + t % ez;
  const int r = t / ez;
  c.j = L.lo[b][1] + r % ey;
  c.i = L.lo[b][0] + r / ey;
  c.n = lin(g, c.i, c.j, c.k);
  return true;
}
__device__ __forceinline__ bool list_contains(const BoxList& L, int i, int j, int k) {
  for (int b = 0; b < L.count; ++b)
    if (i >= L.lo[b][0] && i < L.hi[b][0] && j >= L.lo[b][1] && j < L.hi[b][1] && k >= L.lo[b][2] && k < L.hi[b][2])
      return true;
  return false;
}
// Host side: the list of `count` boxes [lo, hi) (clamped to the grid, empty
// boxes dropped) with its block table; false if count is out of range or a
// box leaves the grid.
inline bool make_box_list(const icy3d_grid& g, int count, const int32_t* lo, const int32_t* hi, BoxList& L) {
  if (count < 0 || count > kMaxBoxes || (count && (!lo || !hi))) return false;
  const int shape[3] = {g.nx, g.ny, g.nz};
  L.count = 0;
  L.first[0] = 0;
  for (int b = 0; b < count; ++b) {
    long cells = 1;
    for (int a = 0; a < 3; ++a) {
      if (lo[3 * b + a] < 0 || hi[3 * b + a] > shape[a]) return false;
      cells *= hi[3 * b + a] > lo[3 * b + a] ? hi[3 * b + a] - lo[3 * b + a] : 0;
    }
    if (!cells) continue;
    const int m = L.count++;
    for (int a = 0; a < 3; ++a) {
      L.lo[m][a] = lo[3 * b + a];
      L.hi[m][a] = hi[3 * b + a];
    }
    L.first[m + 1] = L.first[m] + (int)((cells + kBlock - 1) / kBlock);
  }
  return true;
}
inline unsigned list_blocks(const BoxList& L) { return (unsigned)L.first[L.count]; }

// ---------------------------------------------------------------------------
// Tiles of the row sweeps (k_forces_rows, k_stream_rows,
// k_water_rows): J rows by K cells of
// y and z, X slabs; the tile with its halo laid flat over the lanes, 62 cells
// a wave.
struct StreamTiles {
  int J, K, X, tiles_j, tiles_k;
};
constexpr int kWaveCells = 62;
constexpr int kStreamThreads = 1024, kForceThreads = 768, kWaterThreads = 1024;
constexpr int sweep_cells(int threads) { return threads / 64 * kWaveCells; }
// v of the previous / next lane of the wave.
__device__ __forceinline__ float from_below(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float from_above(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ int from_below(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, true); }
__device__ __forceinline__ int from_above(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, true); }
// An element of a plane at a byte offset below 2^31 (a grid has fewer than
// 2^27 cells): a uniform base and a 32-bit lane offset.
__device__ __forceinline__ float plane_get(const float* base, unsigned offset) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + offset);
}
__device__ __forceinline__ void plane_set(float* base, unsigned offset, float v) {
  *reinterpret_cast<float*>(reinterpret_cast<char*>(base) + offset) = v;
}

// The row sweeps' tiles.  z is cut into as few tiles as leave ten rows a block
// (eight of them its own).  Then the rows and slabs a block owns: a block
// takes a CU to itself, a slab costs it a fixed latency and a time for each
// wave, and it stages two rows and two slabs more than it owns, so the
// cheapest cut is searched over the row tiles that fit and the slab chunks
// that fill whole rounds of the 256 CUs (kSlabLatency, kWaveTime: microseconds
// measured at 24x20x16 and 256x128x128).  A block has tens of rows, however
// many the grid has, so a launch searches tens of cuts.
inline StreamTiles stream_tiles(const icy3d_grid& g, int threads) {
  constexpr int kCus = 256;
  constexpr double kSlabLatency = 1.6, kWaveTime = 0.24;
  const int cells_most = sweep_cells(threads);
  StreamTiles best = {};
  int tiles_k = 1;
  while (10 * ((g.nz + tiles_k - 1) / tiles_k + 2) > cells_most) ++tiles_k;
  const int K = (g.nz + tiles_k - 1) / tiles_k, L = K + 2;
  tiles_k = (g.nz + K - 1) / K;
  const int most = cells_most / L - 2;
  double least = 0.0;
  for (int J = most < g.ny ? most : g.ny; J >= 1; --J) {
    const int tiles_j = (g.ny + J - 1) / J;
    if ((g.ny + tiles_j - 1) / tiles_j != J) continue;  // as many tiles of fewer rows do
    const int waves = ((J + 2) * L + kWaveCells - 1) / kWaveCells, yz = tiles_k * tiles_j;
    for (int rounds = 1; rounds <= 4; ++rounds) {
      const int chunks = yz >= kCus * rounds ? 1 : kCus * rounds / yz;
      const int X = (g.nx + chunks - 1) / chunks, blocks = yz * ((g.nx + X - 1) / X);
      const double cost = (double)((blocks + kCus - 1) / kCus) * (X + 2) * (kSlabLatency + kWaveTime * waves);
      if (best.J == 0 || cost < least) {
        least = cost;
        best = {J, K, X, tiles_j, tiles_k};
      }
    }
  }
  return best;
}
inline unsigned stream_blocks(const icy3d_grid& g, const StreamTiles& T) {
  return (unsigned)(T.tiles_k * T.tiles_j * ((g.nx + T.X - 1) / T.X));
}
inline unsigned stream_threads(const StreamTiles& T) {
  return (unsigned)(((T.J + 2) * (T.K + 2) + kWaveCells - 1) / kWaveCells * 64);
}
}  // namespace icy
