// MI355X (gfx950) kernels of the 2D falling-and-melting ice step.
//
// One thread per cell (n = i * ny + j, 256-thread blocks over the flat
// index, so a wavefront reads 64 consecutive j of one column: coalesced
// q-plane loads).  Flow arithmetic is FP32 like the reference; the thermal
// state, the projection and melt-momentum sums and the rigid mass
// properties are FP64 like the reference.  Every FP64 sum is a two-stage
// reduction (per-block partials, then one block folding them in a fixed
// order), so results do not depend on scheduling.  Rigid-body updates run
// as single-thread kernels on the control block so the pose never leaves
// the device between the kernels that use it.
//
// Differences in structure from the reference, with identical results:
//   - momentum and phase collision of a cell run in one pass (the phase
//     collision reads the acceleration the momentum collision just wrote
//     for the same cell, as the reference's second kernel does);
//   - streaming is written as a pull: cell x takes population q from
//     x - c_q when that cell is fluid, else the bounce-back of its own
//     outgoing population opp(q) (with the moving-ice phase correction), which is
//     exactly what the reference's push writes into x; the same thread then
//     forms phi, u and the pressure's population sum from registers.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstddef>

#include "icy2d.h"

namespace icy2 {

constexpr int kBlock = 256;

__host__ __device__ constexpr int cxq(int q) { return (q == 1 || q == 5 || q == 8) ? 1 : (q == 3 || q == 6 || q == 7) ? -1 : 0; }
__host__ __device__ constexpr int cyq(int q) { return (q == 2 || q == 5 || q == 6) ? 1 : (q == 4 || q == 7 || q == 8) ? -1 : 0; }
__host__ __device__ constexpr int oppq(int q) { return q == 0 ? 0 : q <= 4 ? ((q + 1) % 4) + 1 : ((q - 3) % 4) + 5; }
__host__ __device__ constexpr float wq(int q) { return q == 0 ? 4.0f / 9.0f : q <= 4 ? 1.0f / 9.0f : 1.0f / 36.0f; }
static_assert(oppq(1) == 3 && oppq(2) == 4 && oppq(3) == 1 && oppq(4) == 2, "axis opposites");
static_assert(oppq(5) == 7 && oppq(6) == 8 && oppq(7) == 5 && oppq(8) == 6, "diagonal opposites");

__device__ __forceinline__ int cells(const icy2d_grid& g) { return g.nx * g.ny; }
__device__ __forceinline__ int at(const icy2d_grid& g, int i, int j) { return i * g.ny + j; }
__device__ __forceinline__ bool inside(const icy2d_grid& g, int i, int j) { return i >= 0 && i < g.nx && j >= 0 && j < g.ny; }
// simulator.py:4566-4574
__device__ __forceinline__ bool wall_at(const icy2d_grid& g, int i, int j) {
  const int b = g.boundary;
  return i < b || i >= g.nx - b || j < b || j >= g.ny - b;
}
// simulator.py:2300-2301
__device__ __forceinline__ bool fluid_at(const icy2d_grid& g, int i, int j) { return !wall_at(g, i, j) && g.solid[at(g, i, j)] == 0; }
// Row and column of cell n, one of the cells first .. first + 255: on long
// rows the division is that of the first cell, the same for all lanes (a
// lane's own takes some 30 vector instructions).  For the reductions that run
// over several such blocks of cells; the kernels of one cell a thread gained
// nothing by it.
__device__ __forceinline__ void row_col(const icy2d_grid& g, int first, int n, int& i, int& j) {
  if (g.ny >= 512) {
    i = first / g.ny;
    j = n - i * g.ny;
    if (j >= g.ny) {
      j -= g.ny;
      ++i;
    }
  } else {
    i = n / g.ny;
    j = n - i * g.ny;
  }
}
__device__ __forceinline__ float clamp01(float v) { return fminf(1.0f, fmaxf(0.0f, v)); }
__device__ __forceinline__ double clamp01d(double v) { return fmin(1.0, fmax(0.0, v)); }

// Population storage: FP32, or FP16 holding the population times
// population_scale (a power of two, so the scaling is exact) with FP32
// arithmetic in registers.  Bit 0 of half_populations selects FP16 for the
// momentum populations (f, fbuf), bit 1 for the phase populations (h, hbuf);
// bit 2 rounds FP16 stores stochastically instead of to nearest, so that
// updates smaller than half an FP16 step (the equilibrium lifts of the
// volume projection and the melt-momentum closure) survive in expectation
// instead of being dropped.  The random number is a hash of the value's
// FP32 bits, its index and the control block's step counter: deterministic
// for a given state and step, and fresh every step, so a cell that receives
// the same sub-step lift on an unchanged value is not rounded the same way
// every time.
// The Liang populations are small (O(u) and O(p)); the scale keeps them in
// the FP16 normal range.
template <int Kind>
__device__ __forceinline__ bool half_storage(const icy2d_grid& g) {
  return (g.half_populations >> Kind) & 1;
}
__device__ __forceinline__ uint32_t mix32(uint32_t h) {
  h ^= h >> 16;
  h *= 0x7feb352du;
  h ^= h >> 15;
  h *= 0x846ca68bu;
  h ^= h >> 16;
  return h;
}
__device__ __forceinline__ __half half_stochastic(float x, uint32_t salt, uint32_t step) {
  const __half lo = __float2half_rz(x);
  const float flo = __half2float(lo);
  if (flo == x || !(fabsf(x) < 65504.0f)) return __float2half(x);
  const __half hi = __ushort_as_half((unsigned short)(__half_as_ushort(lo) + 1));  // next step away from zero
  // The step is a power of two and x - flo has no more bits than x, so the
  // quotient is exact as a product with the step's inverse.
  const uint32_t step_bits = __float_as_uint(__half2float(hi) - flo), sign = step_bits & 0x80000000u;
  const float p = (x - flo) * __uint_as_float(sign | ((254u << 23) - (step_bits & 0x7f800000u)));
  const uint32_t key = mix32(salt * 0x9e3779b1u ^ mix32(step + 0x7f4a7c15u));
  const float r = (float)(mix32(__float_as_uint(x) ^ key) >> 8) * (1.0f / 16777216.0f);
  return r < p ? hi : lo;
}
// The step counter as a constant: no kernel that stores populations changes
// it.  Read like any other word it would be loaded again, and waited for with
// all stores before it, at every store.
__device__ __forceinline__ uint32_t rounding_step(const icy2d_grid& g) {
  return *(const __attribute__((address_space(4))) uint32_t*)&g.control->rounding_step;
}
// A stored population's bits, and its value from them.
template <int Kind>
__device__ __forceinline__ uint32_t pop_raw(const float* base, const icy2d_grid& g, int idx) {
  if (half_storage<Kind>(g)) return reinterpret_cast<const uint16_t*>(base)[idx];
  return reinterpret_cast<const uint32_t*>(base)[idx];
}
template <int Kind>
__device__ __forceinline__ float pop_value(const icy2d_grid& g, uint32_t raw) {
  if (half_storage<Kind>(g)) return __half2float(__ushort_as_half((unsigned short)raw)) * g.population_inverse_scale;
  return __uint_as_float(raw);
}
template <int Kind>
__device__ __forceinline__ float pop_get(const float* base, const icy2d_grid& g, int idx) {
  if (half_storage<Kind>(g)) return __half2float(reinterpret_cast<const __half*>(base)[idx]) * g.population_inverse_scale;
  return base[idx];
}
template <int Kind>
__device__ __forceinline__ void pop_set(float* base, const icy2d_grid& g, int idx, float v) {
  if (half_storage<Kind>(g)) {
    const float x = v * g.population_scale;
    reinterpret_cast<__half*>(base)[idx] =
        (g.half_populations & 4) ? half_stochastic(x, (uint32_t)idx * 2u + (uint32_t)Kind, rounding_step(g))
                                 : __float2half(x);
  } else {
    base[idx] = v;
  }
}
template <int Kind>
__device__ __forceinline__ void pop_add(float* base, const icy2d_grid& g, int idx, float v) {
  pop_set<Kind>(base, g, idx, pop_get<Kind>(base, g, idx) + v);
}
constexpr int kMomentum = 0, kPhase = 1;

// Bit 3 of half_populations stores each phase population as its deviation
// from w_q * ref, where ref is the cell's phase: phi[n] for h (every kernel
// that changes a fluid cell's phi re-encodes its h), and phase_ref[n], the
// phase the collision saw, for hbuf (the stream rewrites phi while it pulls
// hbuf from the neighbours).  Near the bulk the deviation is O(u) instead of
// the O(1) equilibrium part, so FP16 keeps ~100x finer absolute steps.
// The projection's flag planes in hbuf use pop_get/pop_set directly.
__device__ __forceinline__ bool phase_relative(const icy2d_grid& g) { return (g.half_populations & 8) != 0; }
__device__ __forceinline__ float phase_get(const float* base, const icy2d_grid& g, int q, int n, float ref) {
  const float v = pop_get<kPhase>(base, g, q * cells(g) + n);
  return phase_relative(g) ? v + wq(q) * ref : v;
}
__device__ __forceinline__ void phase_set(float* base, const icy2d_grid& g, int q, int n, float ref, float v) {
  pop_set<kPhase>(base, g, q * cells(g) + n, phase_relative(g) ? v - wq(q) * ref : v);
}
// The same for the kernels that are compiled for a storage too.  Whether
// w_q * ref is fused with the sum or rounded before it is written out there: a
// stochastic rounding draws another sample for another last bit, and the
// compiler's choice changes with what else a kernel does with the product.
template <bool Fused>
__device__ __forceinline__ float phase_decoded(const icy2d_grid& g, int q, float stored, float ref) {
#pragma clang fp contract(off)
  if (!phase_relative(g)) return stored;
  return Fused ? fmaf(wq(q), ref, stored) : stored + wq(q) * ref;
}
template <bool Fused>
__device__ __forceinline__ float phase_encoded(const icy2d_grid& g, int q, float v, float ref) {
#pragma clang fp contract(off)
  if (!phase_relative(g)) return v;
  return Fused ? fmaf(-wq(q), ref, v) : v - wq(q) * ref;
}
// Bit q of Fused: as above for direction q.
template <unsigned Fused>
__device__ __forceinline__ void phase_store(float* base, const icy2d_grid& g, int q, int n, float ref, float v) {
  const float x = (Fused >> q) & 1u ? phase_encoded<true>(g, q, v, ref) : phase_encoded<false>(g, q, v, ref);
  pop_set<kPhase>(base, g, q * cells(g) + n, x);
}
// The saved phase of a cell whose hbuf is read (0 when unused).
__device__ __forceinline__ float hbuf_ref(const icy2d_grid& g, int n) { return phase_relative(g) ? g.phase_ref[n] : 0.0f; }

// lattice.py:64-104
template <int Q>
__device__ __forceinline__ float momentum_eq(float p, float rho, float ux, float uy) {
  const float cu = (float)cxq(Q) * ux + (float)cyq(Q) * uy, uu = ux * ux + uy * uy;
  float value = 3.0f * wq(Q) * p + wq(Q) * rho * (3.0f * cu + 4.5f * cu * cu - 1.5f * uu);
  if (Q == 0) value -= 3.0f * p;
  return value;
}
// c_q . (x, y) without the products by zero (which a compiler has to keep).
__device__ __forceinline__ float along(int q, float x, float y) {
  const float cx = (float)cxq(q), cy = (float)cyq(q);
  return cxq(q) && cyq(q) ? cx * x + cy * y : cxq(q) ? cx * x : cyq(q) ? cy * y : 0.0f;
}
// The velocity's part of the momentum equilibrium and the whole from it, for the
// kernels that are compiled for a storage.  Which operations are fused is
// written out there (Square: -1.5 u.u): left to the compiler it depends on
// what else of a kernel shares a product, and a stochastic rounding draws
// another sample for another last bit.
template <bool Square>
__device__ __forceinline__ float momentum_poly(int q, float uu, float ux, float uy) {
#pragma clang fp contract(off)
  const float cu = along(q, ux, uy), linear = fmaf(3.0f, cu, 4.5f * cu * cu);
  return Square ? fmaf(-1.5f, uu, linear) : linear - 1.5f * uu;
}
__device__ __forceinline__ float momentum_eq_of(int q, float p, float rho, float poly) {
  const float value = fmaf(wq(q) * rho, poly, 3.0f * wq(q) * p);
  return q == 0 ? fmaf(-3.0f, p, value) : value;
}
__device__ __forceinline__ float momentum_eq_rt(int q, float p, float rho, float ux, float uy) {
  const float cu = (float)cxq(q) * ux + (float)cyq(q) * uy, uu = ux * ux + uy * uy;
  float value = 3.0f * wq(q) * p + wq(q) * rho * (3.0f * cu + 4.5f * cu * cu - 1.5f * uu);
  if (q == 0) value -= 3.0f * p;
  return value;
}
template <int Q>
__device__ __forceinline__ float phase_eq(float phi, float ux, float uy) {
  const float cu = (float)cxq(Q) * ux + (float)cyq(Q) * uy, uu = ux * ux + uy * uy;
  return wq(Q) * phi * (1.0f + 3.0f * cu + 4.5f * cu * cu - 1.5f * uu);
}
__device__ __forceinline__ float phase_eq_rt(int q, float phi, float ux, float uy) {
  const float cu = (float)cxq(q) * ux + (float)cyq(q) * uy, uu = ux * ux + uy * uy;
  return wq(q) * phi * (1.0f + 3.0f * cu + 4.5f * cu * cu - 1.5f * uu);
}
// The velocity's part of phase_eq, as momentum_poly (Products: 3 c.u + 4.5 (c.u)^2).
template <bool Products, bool Square>
__device__ __forceinline__ float phase_poly(int q, float uu, float ux, float uy) {
#pragma clang fp contract(off)
  const float cu = along(q, ux, uy);
  const float linear = Products ? fmaf(4.5f * cu, cu, fmaf(3.0f, cu, 1.0f)) : 1.0f + 3.0f * cu + 4.5f * cu * cu;
  return Square ? fmaf(-1.5f, uu, linear) : linear - 1.5f * uu;
}
// lattice.py:112-115
__device__ __forceinline__ float mixture(const icy2d_grid& g, float phi) {
  const float w = clamp01(phi);
  return g.rho_w * w + g.rho_a * (1.0f - w);
}
// lattice.py:118-177: separable inverse central-moment basis, m = {00,10,01,20,02,11,21,12,22}
template <int C>
__device__ __forceinline__ void basis(float u, float b[3]) {
  if (C == 0) {
    b[0] = 1.0f - u * u;
    b[1] = -2.0f * u;
    b[2] = -1.0f;
  } else if (C == 1) {
    b[0] = 0.5f * u * (u + 1.0f);
    b[1] = u + 0.5f;
    b[2] = 0.5f;
  } else {
    b[0] = 0.5f * u * (u - 1.0f);
    b[1] = u - 0.5f;
    b[2] = 0.5f;
  }
}
// s + a b with the product fused or rounded.
template <bool Fused>
__device__ __forceinline__ float add_product(float s, float a, float b) {
#pragma clang fp contract(off)
  return Fused ? fmaf(a, b, s) : s + a * b;
}
// Bit m of Rounded: moment m's product is rounded before it is added.
template <int Q, unsigned Rounded>
__device__ __forceinline__ float reconstruct_cm(float ux, float uy, const float m[9]) {
  float bx[3], by[3];
  basis<cxq(Q)>(ux, bx);
  basis<cyq(Q)>(uy, by);
  float s = bx[0] * by[0] * m[0] + bx[1] * by[0] * m[1] + bx[0] * by[1] * m[2];
  s = add_product<!(Rounded >> 3 & 1u)>(s, bx[2] * by[0], m[3]);
  s = add_product<!(Rounded >> 4 & 1u)>(s, bx[0] * by[2], m[4]);
  s += bx[1] * by[1] * m[5];
  s = add_product<!(Rounded >> 6 & 1u)>(s, bx[2] * by[1], m[6]);
  s = add_product<!(Rounded >> 7 & 1u)>(s, bx[1] * by[2], m[7]);
  return s + bx[2] * by[2] * m[8];
}
// sums[m] += c_q's raw moment m times v, without the moments that vanish.
template <int M>
__device__ __forceinline__ void add_raw(float (&sums)[M], int q, float v) {
  const int cx = cxq(q), cy = cyq(q);
  const int k[9] = {1, cx, cy, cx * cx, cy * cy, cx * cy, cx * cx * cy, cx * cy * cy, cx * cx * cy * cy};
#pragma unroll
  for (int m = 0; m < M; ++m) {
    if (k[m] > 0) sums[m] += v;
    if (k[m] < 0) sums[m] -= v;
  }
}

// --------------------------------------------------------------- body
// The pose transform, the bilinear coverage sample and the signed distance
// are evaluated in FP64: the cut-link fraction sdf_f / (sdf_f - sdf_s)
// with sdf = threshold - coverage amplifies coverage rounding, and the
// stored FP32 coverage is then the correctly rounded value.
struct Pose {
  double ox, oy, c, s;  // origin and rotation (cos, sin) of the material frame
  float cx, cy, vx, vy, omega;
};
// simulator.py:4835-4845 (centre rounded to FP32 like the reference's) and :2449-2453
__device__ __forceinline__ Pose load_pose(const icy2d_grid& g) {
  const icy2d_control* ctl = g.control;
  Pose p;
  p.ox = ctl->origin[0];
  p.oy = ctl->origin[1];
  p.c = cos((double)ctl->angle);
  p.s = sin((double)ctl->angle);
  const double lx = ctl->local_com[0], ly = ctl->local_com[1];
  p.cx = (float)(p.ox + (p.c * lx - p.s * ly));
  p.cy = (float)(p.oy + (p.s * lx + p.c * ly));
  p.vx = ctl->velocity[0];
  p.vy = ctl->velocity[1];
  p.omega = ctl->omega;
  return p;
}
__device__ __forceinline__ void body_velocity(const Pose& p, float px, float py, float v[2]) {
  const float rx = px - p.cx, ry = py - p.cy;
  v[0] = p.vx + p.omega * -ry;
  v[1] = p.vy + p.omega * rx;
}
// simulator.py:2482-2496
__device__ __forceinline__ void local_coords(const Pose& p, double px, double py, double& lx, double& ly) {
  const double rx = px - p.ox, ry = py - p.oy;
  lx = p.c * rx + p.s * ry;
  ly = -p.s * rx + p.c * ry;
}
// Whether the cell may touch the body's material grid in any orientation: its
// centre lies within the grid's half diagonal and 2 cells of the body's
// origin.  Beyond, the coverage is zero and the signed distance positive, and
// the pose (FP64 sine and cosine, most of these kernels' time) is not needed.
__device__ __forceinline__ bool within_reach(const icy2d_grid& g, int i, int j) {
  const double hw = 0.5 * g.body_nx, hh = 0.5 * g.body_ny;
  const double dx = i + 0.5 - g.control->origin[0], dy = j + 0.5 - g.control->origin[1];
  const float reach = sqrtf((float)(hw * hw + hh * hh)) + 2.0f;
  return !(dx * dx + dy * dy > (double)reach * reach);
}
// simulator.py:1586-1594
__device__ __forceinline__ float body_fraction(const icy2d_grid& g, int bi, int bj) {
  const double mass = fmin(g.cell_mass, fmax(0.0, g.body_mass[bi * g.body_ny + bj]));
  double fraction = mass / g.cell_mass;
  if (mass > 0.0) fraction = fmax(fraction, 1.0e-30);
  return (float)fraction;
}
// simulator.py:1596-1603
__device__ __forceinline__ double body_temperature(const icy2d_grid& g, int k) {
  double t = g.t_melt;
  const double mass = g.body_mass[k];
  if (mass > 1.0e-30) t += g.body_energy[k] / (mass * g.cp_i);
  return fmin(g.t_melt, t);
}
// simulator.py:1605-1613
__device__ __forceinline__ double water_temperature(const icy2d_grid& g, int n) {
  const double v = g.water_v[n];
  if (v > 1.0e-30) return g.t_melt + g.water_e[n] / (g.rho_w_si * g.cp_w * v);
  return g.t_air;
}
// Fixed point for the thermal scatters (exchange heat onto body cells, melt
// onto water cells): integer addition is associative, so the sums do not
// depend on the order in which the atomics land and a step repeats bit for
// bit.  Heat is counted in units of 2^-54 of the latent heat of a full body
// cell, injected volume in 2^-52 of a cell area and injected energy in 2^-52
// of the latent heat.  A term beyond 2^52 units (a quarter of a cell's latent
// heat, or a whole cell for the injection) sets bit 2 of error_flags and adds
// nothing; the host raises at its next read.
constexpr double kFixedTermLimit = 0x1p52;
__device__ __forceinline__ double heat_fixed_scale(const icy2d_grid& g) { return 0x1p54 / (g.latent * g.cell_mass); }
__device__ __forceinline__ double energy_fixed_scale(const icy2d_grid& g) { return 0x1p52 / (g.latent * g.cell_mass); }
__device__ __forceinline__ double volume_fixed_scale(const icy2d_grid& g) { return 0x1p52 / g.area; }
__device__ __forceinline__ long long to_fixed(const icy2d_grid& g, double value, double scale) {
  const double x = value * scale;
  if (!(fabs(x) <= kFixedTermLimit)) {
    atomicOr(&g.control->error_flags, 4);
    return 0;
  }
  return __double2ll_rn(x);
}
__device__ __forceinline__ long long heat_to_fixed(const icy2d_grid& g, double value) {
  return to_fixed(g, value, heat_fixed_scale(g));
}
__device__ __forceinline__ void add_fixed(int64_t* sum, long long q) {
  if (q) atomicAdd(reinterpret_cast<unsigned long long*>(sum), static_cast<unsigned long long>(q));
}
// simulator.py:2508-2530
__device__ __forceinline__ float sample_fraction(const icy2d_grid& g, double lx, double ly) {
  const double gx = lx + (0.5 * g.body_nx - 0.5), gy = ly + (0.5 * g.body_ny - 0.5);
  const int bi0 = (int)floor(gx), bj0 = (int)floor(gy);
  double fraction = 0.0;
#pragma unroll
  for (int di = 0; di < 2; ++di)
#pragma unroll
    for (int dj = 0; dj < 2; ++dj) {
      const int bi = bi0 + di, bj = bj0 + dj;
      if (bi >= 0 && bi < g.body_nx && bj >= 0 && bj < g.body_ny) {
        const double wx = 1.0 - fabs(gx - bi), wy = 1.0 - fabs(gy - bj);
        fraction += fmax(0.0, wx) * fmax(0.0, wy) * (double)body_fraction(g, bi, bj);
      }
    }
  return (float)clamp01d(fraction);
}
// simulator.py:4587-4603 (lattice cells; scaled by dx where the reference uses metres)
__device__ __forceinline__ float signed_distance(const icy2d_grid& g, const Pose& p, int i, int j) {
  double lx, ly;
  local_coords(p, i + 0.5, j + 0.5, lx, ly);
  const double hw = 0.5 * g.body_nx, hh = 0.5 * g.body_ny;
  const int bi = (int)floor(lx + hw), bj = (int)floor(ly + hh);
  if (bi >= 0 && bi < g.body_nx && bj >= 0 && bj < g.body_ny) return g.threshold - g.coverage[at(g, i, j)];
  const double dx = fabs(lx) - hw, dy = fabs(ly) - hh;
  const double ox = fmax(dx, 0.0), oy = fmax(dy, 0.0);
  return (float)(sqrt(ox * ox + oy * oy) + fmin(fmax(dx, dy), 0.0));
}
// simulator.py:4782-4796
__device__ __forceinline__ float cut_fraction(const icy2d_grid& g, const Pose& p, int i, int j, int ni, int nj) {
  const float fluid = fmaxf(signed_distance(g, p, i, j) * g.dx, 1.0e-6f);
  return fminf(0.95f, fmaxf(0.05f, fluid / (fluid - signed_distance(g, p, ni, nj) * g.dx + 1.0e-12f)));
}

// ------------------------------------------------------- reductions
// Wave-wide, the result in every lane: lane l takes in lanes l ^ 32, 16, 8, 4,
// 2 and 1 in turn, as two swaps of rows and four moves within a row of 16
// lanes (rotations by 8 and 4, which are l ^ 8 and l ^ 4 on values of that
// period, then quads and pairs), all between registers.  ds_bpermute shuffles,
// two a step for FP64, took most of the block sums' time: the aperture's six
// 31 us at 1024x2048, 17 with a cell a thread.  The order of the adds is part of the
// results: a stochastically rounded FP16 population hashes its value's bits,
// so that a sum off by its last bit leads to another sample everywhere.
template <int Ctrl>
__device__ __forceinline__ double row_move(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), Ctrl, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), Ctrl, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
// What a swap of 16-lane rows (32-lane halves) leaves in each lane: of v and w
// the even rows (lower halves), and the odd rows (upper halves).
struct Pair {
  double a, b;
};
__device__ __forceinline__ Pair swap_rows(double v, double w) {
  const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(w), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(w), false, false);
  return {__hiloint2double((int)hi[0], (int)lo[0]), __hiloint2double((int)hi[1], (int)lo[1])};
}
__device__ __forceinline__ Pair swap_halves(double v, double w) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(w), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(w), false, false);
  return {__hiloint2double((int)hi[0], (int)lo[0]), __hiloint2double((int)hi[1], (int)lo[1])};
}
// The last four steps: over the lanes of each row.
template <class Op>
__device__ __forceinline__ double row_fold(double v, Op op) {
  v = op(v, row_move<0x128>(v));   // rotated by 8
  v = op(v, row_move<0x124>(v));   // rotated by 4
  v = op(v, row_move<0x4e>(v));    // lanes 2 3 0 1
  return op(v, row_move<0xb1>(v)); // lanes 1 0 3 2
}
template <class Op>
__device__ __forceinline__ double wave_fold(double v, Op op) {
  Pair p = swap_halves(v, v);
  v = op(p.a, p.b);
  p = swap_rows(v, v);
  return row_fold(op(p.a, p.b), op);
}
// Four values at once, each in wave_fold's order: on return row 0 of the wave
// (lanes 0 to 15) holds the first's result, rows 1, 2 and 3 the third's, the
// second's and the fourth's.  A swap of two values leaves the halves of one in
// the lower lanes and those of the other in the upper, so one fold of 64 lanes
// and three adds do for four.
template <class Op>
__device__ __forceinline__ double wave_fold4(double v0, double v1, double v2, double v3, Op op) {
  const Pair p = swap_halves(v0, v1), q = swap_halves(v2, v3);
  const Pair r = swap_rows(op(p.a, p.b), op(q.a, q.b));
  return row_fold(op(r.a, r.b), op);
}
__device__ __forceinline__ double wave_sum(double v) {
  return wave_fold(v, [](double a, double b) { return a + b; });
}
__device__ __forceinline__ double wave_min(double v) {
  return wave_fold(v, [](double a, double b) { return fmin(a, b); });
}
__device__ __forceinline__ double wave_max(double v) {
  return wave_fold(v, [](double a, double b) { return fmax(a, b); });
}
// Writes the block's sums of v[0..K) to partials[blk * K + k] (blocks of at
// most 1024 threads).
template <int K>
__device__ __forceinline__ void block_partials(double (&v)[K], double* partials, int blk) {
  __shared__ double part[K][16];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const double s = wave_sum(v[k]);
    if (lane == 0) part[k][wave] = s;
  }
  __syncthreads();
  if (threadIdx.x < K) {
    double total = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) total += part[threadIdx.x][w];
    partials[blk * K + threadIdx.x] = total;
  }
}
// Reductions over all cells take kRun cells a thread (kRuns): the FP64 wave
// sums, the quotients that are the same for all cells and the block sums' fold
// were a light kernel's largest part.  Each run of kBlock cells keeps its own
// partials, those of a block of its own, so the sums' order is the one of the
// kernels with a cell a thread; the four runs' wave sums share their steps.
// Over the 64-case ensemble, with a cell a thread and this way: evaluation 47
// and 26 us, aperture 74 and 57, targets 76 and 60, transfer 81 and 74, and
// support (minima and maxima only) 46 and 22.
constexpr int kRun = 4;
__device__ __forceinline__ int run_blocks(const icy2d_grid& g) { return (cells(g) + kBlock - 1) / kBlock; }
// Writes the sums (minima, maxima: bit k of the masks) of v[r][0..K) over run r
// of the block to partials[(blk * kRun + r) * K + k].
template <int K, unsigned kMins = 0u, unsigned kMaxs = 0u>
__device__ __forceinline__ void run_partials(const icy2d_grid& g, double (&v)[kRun][K], int blk) {
  static_assert(kRun == 4, "a run for each row of 16 lanes");
  __shared__ double part[kRun][K][kBlock / 64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int row = lane >> 4, run = (row & 1) * 2 + (row >> 1);  // the run whose result wave_fold4 leaves in the row
  auto combine = [](int k, double a, double b) {
    return (kMins >> k) & 1u ? fmin(a, b) : (kMaxs >> k) & 1u ? fmax(a, b) : a + b;
  };
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const double s = wave_fold4(v[0][k], v[1][k], v[2][k], v[3][k], [&](double a, double b) { return combine(k, a, b); });
    if ((lane & 15) == 0) part[run][k][wave] = s;
  }
  __syncthreads();
  if ((int)threadIdx.x < kRun * K) {
    const int r = (int)threadIdx.x / K, k = (int)threadIdx.x - r * K;
    double total = part[r][k][0];
#pragma unroll
    for (int w = 1; w < kBlock / 64; ++w) total = combine(k, total, part[r][k][w]);
    if (blk * kRun + r < run_blocks(g)) g.partials[(blk * kRun + r) * K + k] = total;
  }
}
// Folds partials[b * K + k] over b in a fixed order: one block per k,
// each thread summing a strided subset with four loads in flight, then a
// fixed-order combination of the thread results.  Bit k of min_mask /
// max_mask selects a minimum / maximum instead of a sum; bit k of add_mask
// adds the result to out[k] instead of replacing it.
constexpr int kFinishThreads = 1024;
__device__ __forceinline__ void finish_fold(const double* __restrict__ partials, int blocks, int K, int k,
                                            double* out, unsigned min_mask, unsigned max_mask, unsigned add_mask) {
  __shared__ double part[kFinishThreads];
  const bool is_min = (min_mask >> k) & 1u, is_max = (max_mask >> k) & 1u;
  const double identity = is_min ? 1.0e300 : is_max ? -1.0e300 : 0.0;
  auto combine = [&](double a, double b) { return is_min ? fmin(a, b) : is_max ? fmax(a, b) : a + b; };
  double v = identity;
  int b = threadIdx.x;
  for (; b + 3 * kFinishThreads < blocks; b += 4 * kFinishThreads) {
    const double x0 = partials[b * K + k], x1 = partials[(b + kFinishThreads) * K + k];
    const double x2 = partials[(b + 2 * kFinishThreads) * K + k], x3 = partials[(b + 3 * kFinishThreads) * K + k];
    v = combine(v, combine(combine(x0, x1), combine(x2, x3)));
  }
  for (; b < blocks; b += kFinishThreads) v = combine(v, partials[b * K + k]);
  part[threadIdx.x] = v;
  __syncthreads();
  for (int width = kFinishThreads / 2; width > 0; width >>= 1) {
    if ((int)threadIdx.x < width) part[threadIdx.x] = combine(part[threadIdx.x], part[threadIdx.x + width]);
    __syncthreads();
  }
  if (threadIdx.x == 0) out[k] = ((add_mask >> k) & 1u) ? out[k] + part[0] : part[0];
}

__global__ void __launch_bounds__(kFinishThreads) k2_finish(const double* __restrict__ partials, int blocks, int K,
                                                            double* out, unsigned min_mask, unsigned max_mask,
                                                            unsigned add_mask) {
  finish_fold(partials, blocks, K, (int)blockIdx.x, out, min_mask, max_mask, add_mask);
}

__device__ __forceinline__ int cell_index(int blk) { return blk * (int)blockDim.x + (int)threadIdx.x; }

// ---------------------------------------------------- geometry kernels
// simulator.py:2532-2537; only_if_projected repeats the pass after a
// contact projection (simulator.py:4109-4111) without a host round trip.
__device__ __forceinline__ void k2_body_fraction(const icy2d_grid& g, const int blk, int only_if_projected) {
  if (only_if_projected && g.control->projected == 0) return;
  const int n = cell_index(blk);
  if (n >= cells(g)) return;
  const int i = n / g.ny, j = n - i * g.ny;
  float fraction = 0.0f;
  if (within_reach(g, i, j)) {
    const Pose p = load_pose(g);
    double lx, ly;
    local_coords(p, i + 0.5, j + 0.5, lx, ly);
    fraction = sample_fraction(g, lx, ly);
  }
  g.coverage[n] = fraction;
}
// simulator.py:2539-2544
__device__ __forceinline__ void k2_commit_raster(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk);
  if (n >= cells(g)) return;
  const int i = n / g.ny, j = n - i * g.ny;
  if (wall_at(g, i, j)) g.coverage[n] = 0.0f;
}
// simulator.py:3940-3965: per-block extrema (min x, max x, min y, max y) as partials
__device__ __forceinline__ void k2_support_partials(const icy2d_grid& g, const int blk, int only_if_projected) {
  if (only_if_projected && g.control->projected == 0) return;
  double v[4] = {1.0e30, -1.0e30, 1.0e30, -1.0e30};
  bool covered[kRun], any = false;
#pragma unroll
  for (int r = 0; r < kRun; ++r) {
    const int n = (blk * kRun + r) * kBlock + (int)threadIdx.x;
    covered[r] = n < cells(g) && g.coverage[n] >= g.threshold;
    any = any || covered[r];
  }
  if (!__syncthreads_or(any ? 1 : 0)) {  // a block without ice: the identities
    if (threadIdx.x < 4) g.partials[blk * 4 + threadIdx.x] = v[threadIdx.x & 1];
    return;
  }
  if (any) {
    const Pose p = load_pose(g);
#pragma unroll
    for (int r = 0; r < kRun; ++r) {
      if (!covered[r]) continue;
      const int first = (blk * kRun + r) * kBlock;
      int i, j;
      row_col(g, first, first + (int)threadIdx.x, i, j);
      if (signed_distance(g, p, i, j) <= 0.0f) {
        v[0] = fmin(v[0], (double)(float)(i - p.ox));
        v[1] = fmax(v[1], (double)(float)(i + 1 - p.ox));
        v[2] = fmin(v[2], (double)(float)(j - p.oy));
        v[3] = fmax(v[3], (double)(float)(j + 1 - p.oy));
      }
    }
  }
  // Minima (even k) and maxima (odd k) over the block: per wave by
  // shuffles, then over the waves.
  __shared__ double part[4][16];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const double r = (k & 1) ? wave_max(v[k]) : wave_min(v[k]);
    if (lane == 0) part[k][wave] = r;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    const int k = threadIdx.x;
    double r = part[k][0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r = (k & 1) ? fmax(r, part[k][w]) : fmin(r, part[k][w]);
    g.partials[blk * 4 + k] = r;
  }
}
// simulator.py:3932-3938 and :3966-3971: store the extrema
__device__ __forceinline__ void k2_support_store(const icy2d_grid& g, const int blk, int reduce, int only_if_projected) {
  icy2d_control* ctl = g.control;
  if (only_if_projected && ctl->projected == 0) return;
  double* e = g.partials + g.partials_capacity - 4;
  if (!reduce) {
    // simulator.py:4115-4119: a fixed-pose refresh resets the flag and the extrema
    ctl->projected = 0;
    e[0] = e[2] = 1.0e30;
    e[1] = e[3] = -1.0e30;
  } else if (!(e[2] < 1.0e20)) {
    e[0] = e[1] = e[2] = e[3] = 0.0;
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) ctl->support[k] = (float)e[k];
}
// simulator.py:3973-4017
__device__ __forceinline__ void k2_integrate_rigid(const icy2d_grid& g, const int blk) {
  icy2d_control* ctl = g.control;
  if (ctl->inertia > 0.0) {
    const float mass = (float)ctl->mass, inertia = (float)ctl->inertia;
    const float jx = (float)ctl->impulse[0] + mass * g.gx, jy = (float)ctl->impulse[1] + mass * g.gy;
    const float torque = (float)ctl->impulse[2];
    const float vx = g.linear_damping * (ctl->velocity[0] + jx / mass);
    const float vy = g.linear_damping * (ctl->velocity[1] + jy / mass);
    const float omega = g.angular_damping * (ctl->omega + torque / inertia);
    const float lcx = (float)ctl->local_com[0], lcy = (float)ctl->local_com[1];
    const Pose p = load_pose(g);
    const float angle = ctl->angle + omega;
    const float cx = p.cx + vx, cy = p.cy + vy;
    const float c = cosf(angle), s = sinf(angle);
    ctl->velocity[0] = vx;
    ctl->velocity[1] = vy;
    ctl->angle = angle;
    ctl->omega = omega;
    ctl->origin[0] = cx - (c * lcx - s * lcy);
    ctl->origin[1] = cy - (s * lcx + c * lcy);
  } else {
    ctl->velocity[0] = ctl->velocity[1] = 0.0f;
    ctl->omega = 0.0f;
  }
  ctl->impulse[0] = ctl->impulse[1] = ctl->impulse[2] = 0.0;
  ctl->rounding_step += 1u;
}
// simulator.py:4019-4080
__device__ __forceinline__ void k2_project_inside(const icy2d_grid& g, const int blk) {
  icy2d_control* ctl = g.control;
  int projected = 0;
  const Pose p = load_pose(g);
  float cx = p.cx, cy = p.cy, vx = ctl->velocity[0], vy = ctl->velocity[1];
  const float lcx = (float)ctl->local_com[0], lcy = (float)ctl->local_com[1];
  const float rcx = p.c * lcx - p.s * lcy, rcy = p.s * lcx + p.c * lcy;
  if (ctl->inertia > 0.0 && ctl->support[1] > ctl->support[0]) {
    const float lower = (float)g.boundary, upper_x = (float)(g.nx - g.boundary), upper_y = (float)(g.ny - g.boundary);
    const float lo_x = lower - (ctl->support[0] - rcx), hi_x = upper_x - (ctl->support[1] - rcx);
    const float lo_y = lower - (ctl->support[2] - rcy), hi_y = upper_y - (ctl->support[3] - rcy);
    if (cx <= lo_x) {
      if (cx < lo_x) projected = 1;
      cx = lo_x;
      vx = fmaxf(vx, 0.0f);
    } else if (cx >= hi_x) {
      if (cx > hi_x) projected = 1;
      cx = hi_x;
      vx = fminf(vx, 0.0f);
    }
    if (cy <= lo_y) {
      if (cy < lo_y) projected = 1;
      cy = lo_y;
      vy = fmaxf(vy, 0.0f);
    } else if (cy >= hi_y) {
      if (cy > hi_y) projected = 1;
      cy = hi_y;
      vy = fminf(vy, 0.0f);
    }
  }
  ctl->velocity[0] = vx;
  ctl->velocity[1] = vy;
  ctl->projected = projected;
  if (projected) {
    ctl->origin[0] = cx - rcx;
    ctl->origin[1] = cy - rcy;
  }
}
// simulator.py:2699-2711 (init) and :2713-2727
__device__ __forceinline__ void k2_update_solid_mask(const icy2d_grid& g, const int blk, int init) {
  const int n = cell_index(blk);
  if (n >= cells(g)) return;
  const int i = n / g.ny, j = n - i * g.ny;
  bool solid = false;
  if (g.control->inertia > 0.0 && !wall_at(g, i, j) && within_reach(g, i, j))
    solid = signed_distance(g, load_pose(g), i, j) <= 0.0f;
  if (!init) g.prev_solid[n] = g.solid[n];
  g.solid[n] = (int8_t)solid;
  if (init) g.prev_solid[n] = (int8_t)solid;
}

// -------------------------------------------------------- initialisation
// simulator.py:2595-2624
__device__ __forceinline__ void k2_initialize_fluid(const icy2d_grid& g, const int blk, int water_width, int water_height) {
  const int n = cell_index(blk), N = cells(g);
  if (n >= N) return;
  const Pose p = load_pose(g);
  const int i = n / g.ny, j = n - i * g.ny;
  const float indicator = (i < water_width && j < water_height) ? 1.0f : 0.0f;
  const bool active = fluid_at(g, i, j);
  const float phi0 = active ? indicator : 0.0f;
  float v[2] = {0.0f, 0.0f};
  if (g.solid[n] == 1) body_velocity(p, i + 0.5f, j + 0.5f, v);
  const float phase = g.solid[n] == 1 ? indicator : phi0;
  g.phi[n] = phase;
  g.u[n] = v[0];
  g.u[N + n] = v[1];
  g.a[n] = g.a[N + n] = 0.0f;
  g.p[n] = 0.0f;
  const float rho = mixture(g, phi0);
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    pop_set<kMomentum>(g.f, g, q * N + n, momentum_eq_rt(q, 0.0f, rho, v[0], v[1]));
    phase_set(g.h, g, q, n, phase, active ? phase_eq_rt(q, phi0, v[0], v[1]) : 0.0f);
  }
}
// simulator.py:2664-2697
__device__ __forceinline__ void k2_hydrostatic_equilibrium(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk), N = cells(g);
  if (n >= N) return;
  const int i = n / g.ny, j = n - i * g.ny;
  if (fluid_at(g, i, j)) {
    const float phi = g.phi[n], rho = mixture(g, phi);
    g.u[n] = g.u[N + n] = 0.0f;
    g.p[n] = g.p_ref[j];
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      pop_set<kMomentum>(g.f, g, q * N + n, momentum_eq_rt(q, 0.0f, rho, 0.0f, 0.0f));
      phase_set(g.h, g, q, n, phi, phase_eq_rt(q, phi, 0.0f, 0.0f));
    }
  } else {
    float v[2] = {0.0f, 0.0f};
    if (g.solid[n] == 1) body_velocity(load_pose(g), i + 0.5f, j + 0.5f, v);
    g.u[n] = v[0];
    g.u[N + n] = v[1];
    g.p[n] = 0.0f;
  }
}
// simulator.py:4125-4133 (partials of the fluid phase sum)
__device__ __forceinline__ void k2_water_volume_partials(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk);
  double v[1] = {0.0};
  if (n < cells(g)) {
    const int i = n / g.ny, j = n - i * g.ny;
    if (fluid_at(g, i, j)) v[0] = (double)g.phi[n];
  }
  block_partials<1>(v, g.partials, blk);
}
__device__ __forceinline__ void k2_copy_initial_volume(const icy2d_grid& g, const int blk) { g.control->water[1] = g.control->water[0]; }
// simulator.py:3833-3858
__device__ __forceinline__ void k2_recover_initial_moments(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk), N = cells(g);
  if (n >= N) return;
  const int i = n / g.ny, j = n - i * g.ny;
  if (fluid_at(g, i, j)) {
    float phi = 0.0f, mx = 0.0f, my = 0.0f, h[9];
    const float old_phase = g.phi[n];
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      h[q] = phase_get(g.h, g, q, n, old_phase);
      phi += h[q];
      const float fv = pop_get<kMomentum>(g.f, g, q * N + n);
      if (cxq(q)) mx += (float)cxq(q) * fv;
      if (cyq(q)) my += (float)cyq(q) * fv;
    }
    g.phi[n] = phi;
    if (phase_relative(g)) {
#pragma unroll
      for (int q = 0; q < 9; ++q) phase_set(g.h, g, q, n, phi, h[q]);
    }
    const float rho = fmaxf(mixture(g, phi), 1.0e-12f);
    g.u[n] = mx / rho;
    g.u[N + n] = my / rho;
  } else if (g.solid[n] == 1) {
    float v[2];
    body_velocity(load_pose(g), i + 0.5f, j + 0.5f, v);
    g.u[n] = v[0];
    g.u[N + n] = v[1];
  } else {
    g.phi[n] = 0.0f;
    g.u[n] = g.u[N + n] = 0.0f;
  }
}

// --------------------------------------------------------------- flow
// simulator.py:2459-2477
__device__ __forceinline__ float phase_neighbor(const icy2d_grid& g, int i, int j, int sx, int sy, int distance,
                                                float centre) {
  float value = centre;
  const int i1 = i + sx, j1 = j + sy;
  if (inside(g, i1, j1) && fluid_at(g, i1, j1)) {
    value = g.phi[at(g, i1, j1)];
    if (distance == 2) {
      const int i2 = i + 2 * sx, j2 = j + 2 * sy;
      value = (inside(g, i2, j2) && fluid_at(g, i2, j2)) ? g.phi[at(g, i2, j2)] : centre;
    }
  }
  return value;
}
// Blended isotropic gradient of simulator.py:3263-3290 / :3566-3589.
struct PhaseStencil {
  float g[2], source[2], laplacian;
};
__device__ __forceinline__ PhaseStencil phase_stencil(const icy2d_grid& g, int i, int j, float phi) {
  PhaseStencil s = {{0.0f, 0.0f}, {0.0f, 0.0f}, 0.0f};
  const float alpha = 1.0f / 3.0f;
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const float p1 = phase_neighbor(g, i, j, cxq(q), cyq(q), 1, phi);
    const float p2 = phase_neighbor(g, i, j, cxq(q), cyq(q), 2, phi);
    const float c[2] = {(float)cxq(q), (float)cyq(q)};
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      s.source[e] += 3.0f * wq(q) * c[e] * (p1 - phi);
      s.g[e] += (1.0f - alpha) * 3.0f * wq(q) * c[e] * (p1 - phi);
      s.g[e] += alpha * 1.5f * wq(q) * c[e] * (4.0f * p1 - p2 - 3.0f * phi);
    }
    s.laplacian += 6.0f * wq(q) * (p1 - phi);
  }
  return s;
}

// Tao single-node reflection into the cut link's outgoing slot and its
// momentum exchange (simulator.py:4798-4866).  Returns true when a link was cut.
// pdyn and poly: the cell's dynamic pressure and momentum_poly of its velocity
// with half its force density, as the collision has just computed them.
__device__ __forceinline__ bool prepare_cut_links(const icy2d_grid& g, const Pose& p, int i, int j, float pdyn,
                                                  const float poly[9], float raw[9], double load[3]) {
  const int N = cells(g), n = at(g, i, j);
  const float rho = mixture(g, g.phi[n]);
  float prepared[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) prepared[q] = raw[q];
  bool cut = false;
#pragma unroll
  for (int q = 1; q < 9; ++q) {
    const int ni = i + cxq(q), nj = j + cyq(q);
    if (!(inside(g, ni, nj) && g.solid[at(g, ni, nj)] == 1)) continue;
    const float eta = cut_fraction(g, p, i, j, ni, nj);
    const float bx = (i + 0.5f) + eta * (float)cxq(q), by = (j + 0.5f) + eta * (float)cyq(q);
    float ub[2];
    body_velocity(p, bx, by, ub);
    const int o = oppq(q);
    const float noneq = pop_get<kMomentum>(g.f, g, q * N + n) - momentum_eq_of(q, pdyn, rho, poly[q]);
    const float wall = momentum_eq_rt(o, pdyn, rho, ub[0], ub[1]);
    const float reflected = (wall + noneq + eta * raw[o]) / (1.0f + eta);
    prepared[q] = reflected;
    float ix = ((float)cxq(q) - ub[0]) * raw[q] - ((float)-cxq(q) - ub[0]) * reflected;
    float iy = ((float)cyq(q) - ub[1]) * raw[q] - ((float)-cyq(q) - ub[1]) * reflected;
    // (1 - eta) p_ref[j] + eta p_ref[nj]; written out as either product could be the fused one
    const float keep = 1.0f - eta, own_ref = g.p_ref[j];
    const float pref = cyq(q) ? fmaf(keep, own_ref, eta * g.p_ref[nj]) : fmaf(eta, own_ref, keep * own_ref);
    ix += 6.0f * wq(q) * pref * (float)cxq(q);
    iy += 6.0f * wq(q) * pref * (float)cyq(q);
    const double rx = (double)(bx - p.cx), ry = (double)(by - p.cy);
    load[0] += (double)ix;
    load[1] += (double)iy;
    load[2] += rx * (double)iy - ry * (double)ix;
    cut = true;
  }
#pragma unroll
  for (int q = 0; q < 9; ++q) raw[q] = prepared[q];
  return cut;
}

// The collision reads a 5x5 phase stencil (the blended gradient uses
// neighbours at distance 2) and a 3x3 velocity stencil.  A block covers a
// tile of Rows x 64 cells (Rows = blockDim.x / 64) and stages, once, the
// phase and fluid flags of the tile with a PH-cell halo and its velocities
// and neighbour kinds with a VH-cell halo in LDS: PH = 2, VH = 1 for the
// tile's own collisions, one more of each when the block also collides a
// one-cell ring around the tile (the fused collide-stream).
constexpr int kTileCols = 64, kTileMaxRows = 8;
template <int Rows, int PH, int VH>
struct StencilWindow {
  static constexpr int kPhaseHalo = PH, kVelocityHalo = VH;
  static constexpr int kPR = Rows + 2 * PH, kPC = kTileCols + 2 * PH, kUR = Rows + 2 * VH, kUC = kTileCols + 2 * VH;
  float phi[kPR][kPC];
  float u[2][kUR][kUC];
  uint8_t fluid[kPR][kPC];
  uint8_t kind[kUR][kUC];  // 0 fluid, 1 ice (solid == 1), 2 wall or outside
};
using CollideTile = StencilWindow<kTileMaxRows, 2, 1>;
// simulator.py:2459-2477 on the staged window (a, b: window row/column of the cell).
template <class W>
__device__ __forceinline__ float phase_neighbor_tile(const W& t, int a, int b, int sx, int sy, int distance,
                                                     float centre) {
  float value = centre;
  if (t.fluid[a + sx][b + sy]) {
    value = t.phi[a + sx][b + sy];
    if (distance == 2) value = t.fluid[a + 2 * sx][b + 2 * sy] ? t.phi[a + 2 * sx][b + 2 * sy] : centre;
  }
  return value;
}
template <class W>
__device__ __forceinline__ PhaseStencil phase_stencil_tile(const W& t, int a, int b, float phi) {
  PhaseStencil s = {{0.0f, 0.0f}, {0.0f, 0.0f}, 0.0f};
  const float alpha = 1.0f / 3.0f;
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const float p1 = phase_neighbor_tile(t, a, b, cxq(q), cyq(q), 1, phi);
    const float p2 = phase_neighbor_tile(t, a, b, cxq(q), cyq(q), 2, phi);
    const float c[2] = {(float)cxq(q), (float)cyq(q)};
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      s.source[e] += 3.0f * wq(q) * c[e] * (p1 - phi);
      s.g[e] += (1.0f - alpha) * 3.0f * wq(q) * c[e] * (p1 - phi);
      s.g[e] += alpha * 1.5f * wq(q) * c[e] * (4.0f * p1 - p2 - 3.0f * phi);
    }
    s.laplacian += 6.0f * wq(q) * (p1 - phi);
  }
  return s;
}
template <class W>
__device__ __forceinline__ void stage_window(const icy2d_grid& g, W& t, int i0, int j0, int rows) {
  constexpr int PH = W::kPhaseHalo, VH = W::kVelocityHalo;
  const int N = cells(g), threads = (int)blockDim.x;
  // All of a thread's values are loaded before the first is used (one after
  // the other they cost a memory latency each): up to four of the phase and
  // three of the velocity for tiles of 2, 4 or 8 rows of 64 threads.
  constexpr int kPhases = ((2 + 2 * PH) * W::kPC + 127) / 128, kVelocities = ((2 + 2 * VH) * W::kUC + 127) / 128;
  const int phases = (rows + 2 * PH) * W::kPC, velocities = (rows + 2 * VH) * W::kUC;
  float phase[kPhases], vx[kVelocities], vy[kVelocities];
  int label[kPhases], solid[kVelocities];
  bool free[kPhases], in[kVelocities], open[kVelocities];
#pragma unroll
  for (int f = 0; f < kPhases; ++f) {
    if (f * threads >= phases) continue;
    const int e = (int)threadIdx.x + f * threads, a = e / W::kPC, b = e - a * W::kPC, i = i0 - PH + a, j = j0 - PH + b;
    const bool inner = inside(g, i, j);
    const int m = inner ? at(g, i, j) : 0;
    phase[f] = g.phi[m];
    label[f] = g.solid[m];
    free[f] = inner && !wall_at(g, i, j);
  }
#pragma unroll
  for (int f = 0; f < kVelocities; ++f) {
    if (f * threads >= velocities) continue;
    const int e = (int)threadIdx.x + f * threads, a = e / W::kUC, b = e - a * W::kUC, i = i0 - VH + a, j = j0 - VH + b;
    in[f] = inside(g, i, j);
    const int m = in[f] ? at(g, i, j) : 0;
    solid[f] = g.solid[m];
    vx[f] = g.u[m];
    vy[f] = g.u[N + m];
    open[f] = in[f] && !wall_at(g, i, j);
  }
#pragma unroll
  for (int f = 0; f < kPhases; ++f) {
    const int e = (int)threadIdx.x + f * threads, a = e / W::kPC, b = e - a * W::kPC;
    if (e >= phases) continue;
    const bool fluid = free[f] && label[f] == 0;  // a wall's or ice cell's phase is dropped
    t.fluid[a][b] = fluid;
    t.phi[a][b] = fluid ? phase[f] : 0.0f;
  }
#pragma unroll
  for (int f = 0; f < kVelocities; ++f) {
    const int e = (int)threadIdx.x + f * threads, a = e / W::kUC, b = e - a * W::kUC;
    if (e >= velocities) continue;
    const bool fluid = open[f] && solid[f] == 0;
    t.kind[a][b] = fluid ? 0 : in[f] && solid[f] == 1 ? 1 : 2;
    t.u[0][a][b] = fluid ? vx[f] : 0.0f;
    t.u[1][a][b] = fluid ? vy[f] : 0.0f;
  }
}

// What a cell's collision reads of its own, loaded before the block waits for
// the window: the populations as stored, velocity, pressure and water.
struct OwnCell {
  uint32_t f[9], h[9];
  float u[2], p;
  double water_v, water_e;
};
__device__ __forceinline__ void load_own(const icy2d_grid& g, int n, int with_momentum, OwnCell& o) {
  const int N = cells(g);
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    o.h[q] = pop_raw<kPhase>(g.h, g, q * N + n);
    if (with_momentum) o.f[q] = pop_raw<kMomentum>(g.f, g, q * N + n);
  }
  o.u[0] = g.u[n];
  o.u[1] = g.u[N + n];
  if (with_momentum) {
    o.p = g.p[n];
    o.water_v = g.water_v[n];
    o.water_e = g.water_e[n];
  }
}
// simulator.py:3241-3552 (momentum, with the cut-link preparation of
// :4798-4866) then :3554-3697 (phase) for one fluid cell (i, j) = n from a
// staged window: (a, b) is the cell in the window's phase arrays, (av, bv) in
// its velocity arrays.  The post-collision populations go to pf and ph, the
// force density to (ax, ay) (read from g.a when with_momentum is 0) and the
// cut links' momentum exchange is added to load.
// Populations are moved by kernels compiled for their storage (one_case):
// with a branch around each access an FP16 load was converted, and so waited
// for, before the next was issued.
// The moments of the populations, equilibria and forces are sums over the nine
// directions in the reference's order, which is part of the results: the
// momentum populations are small differences of terms of order one (the same
// moments as polynomials in u moved them by 2e-4 in eight steps), and a
// stochastically rounded FP16 one draws another sample for another last bit.
// What costs nothing is left out: the products by a direction's zeros and the
// vanishing moments (a compiler has to keep 0 * x), and the body's pose (FP64
// sine and cosine) where no neighbour is ice.  Bound by the vector ALUs: 149 us
// at 1024x2048 (its bytes take 85) and 699 over the 64-case ensemble; 247 and
// 1503 with all products, a pose in every lane and branches around the loads.
template <bool Push, class W>
__device__ __forceinline__ void collide_cell(const icy2d_grid& g, const OwnCell& own, bool near, const Pose& pose,
                                             const W& tile, int a0, int b0, int av, int bv, int i, int j, int n,
                                             int with_momentum, float pf[9], float ph[9], float& ax, float& ay, double load[3]) {
  const int N = cells(g);
  const float phi = tile.phi[a0][b0];
  const PhaseStencil st = phase_stencil_tile(tile, a0, b0, phi);
  if (with_momentum) {
    // _fluid_force_viscosity_and_gradient (simulator.py:3241-3368)
    const float bounded = clamp01(phi), rho_b = g.rho_w * bounded + g.rho_a * (1.0f - bounded);
    const float beta = 12.0f * g.sigma / g.width, kappa = 1.5f * g.sigma * g.width;
    const float anomaly_rho = rho_b - g.rho_ref[j];
    const double v = own.water_v;
    const float temperature = (float)(v > 1.0e-30 ? g.t_melt + own.water_e / (g.rho_w_si * g.cp_w * v) : g.t_air);
    const float ratio = -g.expansion * (temperature - g.t_ref);
    const float ww = clamp01(2.0f * bounded - 1.0f);
    float fx = anomaly_rho * g.gx, fy = anomaly_rho * g.gy;
    fx += ww * g.rho_w * ratio * g.gx;
    fy += ww * g.rho_w * ratio * g.gy;
    fx /= rho_b;
    fy /= rho_b;
    const float chemical = 4.0f * beta * bounded * (bounded - 1.0f) * (bounded - 0.5f) - kappa * st.laplacian;
    fx += chemical * st.g[0] / rho_b;
    fy += chemical * st.g[1] / rho_b;
    const float ux0 = own.u[0], uy0 = own.u[1];
    float gxx = 0.0f, gxy = 0.0f, gyx = 0.0f, gyy = 0.0f;
#pragma unroll
    for (int q = 1; q < 9; ++q) {
      const int ni = i + cxq(q), nj = j + cyq(q);
      const int a = av + cxq(q), b = bv + cyq(q);
      float v[2] = {tile.u[0][a][b], tile.u[1][a][b]};  // zero at walls and ice
      if (near && tile.kind[a][b] == 1) body_velocity(pose, ni + 0.5f, nj + 0.5f, v);
      const float dxv = v[0] - ux0, dyv = v[1] - uy0, w3 = 3.0f * wq(q);
      if (cxq(q)) gxx += w3 * (float)cxq(q) * dxv;
      if (cyq(q)) gxy += w3 * (float)cyq(q) * dxv;
      if (cxq(q)) gyx += w3 * (float)cxq(q) * dyv;
      if (cyq(q)) gyy += w3 * (float)cyq(q) * dyv;
    }
    const float near_solid = near ? 1.0f : 0.0f;
    const float cs = g.smagorinsky;
    const float nu_t = cs * cs * sqrtf(2.0f * (gxx * gxx + gyy * gyy + 0.5f * (gxy + gyx) * (gxy + gyx)));
    ax = fx;
    ay = fy;
    // _collide_momentum (simulator.py:3370-3552)
    const float ux = ux0 + 0.5f * ax, uy = uy0 + 0.5f * ay;
    const float fraction = clamp01(phi);
    const float nu = fraction * g.nu_w + (1.0f - fraction) * g.nu_a + nu_t;
    const float tau = 0.5f + 3.0f * nu;
    const float indicator = fmaxf(1.0f - fraction, near_solid);
    const float shear_tau = fmaxf(tau, 0.5f + (g.interface_tau - 0.5f) * indicator);
    const float rho = mixture(g, phi), pdyn = own.p - g.p_ref[j];
    const float Fx = rho * ax, Fy = rho * ay, drho = g.rho_w - g.rho_a;
    const float gsx = st.source[0], gsy = st.source[1];
    // Raw moments m = {00, 10, 01, 20, 02, 11, 21, 12, 22}.
    float raw[6] = {0, 0, 0, 0, 0, 0}, eq[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, src[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, poly[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      add_raw(raw, q, pop_value<kMomentum>(g, own.f[q]));
      poly[q] = momentum_poly<true>(q, fmaf(uy, uy, ux * ux), ux, uy);
      add_raw(eq, q, momentum_eq_of(q, pdyn, rho, poly[q]));
      if (q > 0) add_raw(src, q, wq(q) * 3.0f * (along(q, Fx, Fy) + drho * along(q, ux, uy) * along(q, gsx, gsy)));
    }
    const float w_phys = 1.0f / tau, w_shear = 1.0f / shear_tau;
    const float sp = 1.0f - 0.5f * w_phys, ss = 1.0f - 0.5f * w_shear;
    float post[9];
#pragma unroll
    for (int m = 0; m < 3; ++m) post[m] = raw[m] - w_phys * (raw[m] - eq[m]) + sp * src[m];
    const float trace = eq[3] + eq[4] + 0.5f * (src[3] + src[4]);
    const float diff = raw[3] - raw[4];
    const float post_diff = diff - w_shear * (diff - (eq[3] - eq[4])) + ss * (src[3] - src[4]);
    post[3] = 0.5f * (trace + post_diff);
    post[4] = 0.5f * (trace - post_diff);
    post[5] = raw[5] - w_shear * (raw[5] - eq[5]) + ss * src[5];
#pragma unroll
    for (int m = 6; m < 9; ++m) post[m] = eq[m] + 0.5f * src[m];
    // reconstruct_cm at u = 0: factors 1, 1/2 and 1/4, so every product is exact.
    pf[0] = post[0] - post[3] - post[4] + post[8];
    pf[1] = 0.5f * (post[1] + post[3] - post[7] - post[8]);
    pf[2] = 0.5f * (post[2] + post[4] - post[6] - post[8]);
    pf[3] = 0.5f * (post[3] - post[1] + post[7] - post[8]);
    pf[4] = 0.5f * (post[4] - post[2] + post[6] - post[8]);
    pf[5] = 0.25f * (post[5] + post[6] + post[7] + post[8]);
    pf[6] = 0.25f * (post[6] - post[5] - post[7] + post[8]);
    pf[7] = 0.25f * (post[5] - post[6] - post[7] + post[8]);
    pf[8] = 0.25f * (post[7] - (post[5] + post[6]) + post[8]);
    if (near) prepare_cut_links(g, pose, i, j, pdyn, poly, pf, load);
  } else {
    ax = g.a[n];
    ay = g.a[N + n];
  }
  // _collide_phase (simulator.py:3554-3697)
  const float ux = own.u[0] + 0.5f * ax, uy = own.u[1] + 0.5f * ay;
  const float rate = 1.0f / (3.0f * g.mobility + 0.5f);
  const float norm = sqrtf(st.g[0] * st.g[0] + st.g[1] * st.g[1]) + 1.0e-14f;
  const float compression = 4.0f * phi * (1.0f - phi) / g.width;
  const float nx_ = st.g[0] / norm, ny_ = st.g[1] / norm;
  // Central moments, m = {00, 10, 01, 20, 02, 11, 21, 12, 22}.
  const float uu = Push ? fmaf(uy, uy, ux * ux) : fmaf(ux, ux, uy * uy);  // as momentum_poly: written out
  float r10 = 0.0f, r01 = 0.0f, eq[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, src[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const float rx = (float)cxq(q) - ux, ry = (float)cyq(q) - uy;
    const float hv = phase_decoded<true>(g, q, pop_value<kPhase>(g, own.h[q]), phi);
    const float he = wq(q) * phi * phase_poly<!Push, !Push>(q, uu, ux, uy);
    const float force = wq(q) * compression * along(q, nx_, ny_);
    const float rx2 = rx * rx, ry2 = ry * ry;
    const float k[9] = {1.0f, rx, ry, rx2, ry2, rx * ry, rx2 * ry, rx * ry2, rx2 * ry2};
    r10 += hv * rx;
    r01 += hv * ry;
#pragma unroll
    for (int m = 0; m < 9; ++m) {
      eq[m] += he * k[m];
      if (q > 0) src[m] += force * k[m];
    }
  }
  float post[9];
#pragma unroll
  for (int m = 0; m < 9; ++m) post[m] = eq[m] + 0.5f * src[m];
  post[1] = r10 - rate * (r10 - eq[1]) + (1.0f - 0.5f * rate) * src[1];
  post[2] = r01 - rate * (r01 - eq[2]) + (1.0f - 0.5f * rate) * src[2];
  // Opposite directions of an axis share two products: fused where they are
  // used first, rounded where they are used again. Written out like momentum_poly's.
  ph[0] = reconstruct_cm<0, 0u>(ux, uy, post);
  ph[1] = reconstruct_cm<1, 0u>(ux, uy, post);
  ph[2] = reconstruct_cm<2, 0u>(ux, uy, post);
  ph[3] = reconstruct_cm<3, 0x48u>(ux, uy, post);
  ph[4] = reconstruct_cm<4, 0x90u>(ux, uy, post);
  ph[5] = reconstruct_cm<5, 0u>(ux, uy, post);
  ph[6] = reconstruct_cm<6, 0x48u>(ux, uy, post);
  ph[7] = reconstruct_cm<7, 0x90u>(ux, uy, post);
  ph[8] = reconstruct_cm<8, 0xd8u>(ux, uy, post);
}
// Whether one of the cell's eight neighbours is ice (the window's kinds).
template <class W>
__device__ __forceinline__ bool beside_ice(const W& t, int av, int bv) {
  bool near = false;
#pragma unroll
  for (int q = 1; q < 9; ++q) near = near || t.kind[av + cxq(q)][bv + cyq(q)] == 1;
  return near;
}

// The collisions of the tile's fluid cells into fbuf and hbuf (and the
// force density into a).
__device__ __forceinline__ void k2_collide(const icy2d_grid& g, const int blk, int with_momentum) {
  __shared__ CollideTile tile;
  const int N = cells(g);
  const int rows = (int)blockDim.x / kTileCols, tiles_j = (g.ny + kTileCols - 1) / kTileCols;
  const int i0 = (blk / tiles_j) * rows, j0 = (blk % tiles_j) * kTileCols;
  const int li = (int)threadIdx.x / kTileCols, lj = (int)threadIdx.x % kTileCols;
  const int i = i0 + li, j = j0 + lj;
  OwnCell own = {};
  if (i < g.nx && j < g.ny) load_own(g, at(g, i, j), with_momentum, own);
  stage_window(g, tile, i0, j0, rows);
  __syncthreads();
  double load[3] = {0.0, 0.0, 0.0};
  if (i < g.nx && j < g.ny && tile.fluid[li + 2][lj + 2]) {
    const int n = at(g, i, j);
    const float phi = tile.phi[li + 2][lj + 2];
    float pf[9], ph[9], ax, ay;
    const bool near = beside_ice(tile, li + 1, lj + 1);
    Pose pose = {};
    if (near) pose = load_pose(g);
    collide_cell<false>(g, own, near, pose, tile, li + 2, lj + 2, li + 1, lj + 1, i, j, n, with_momentum, pf, ph, ax, ay,
                        load);
    if (with_momentum) {
      g.a[n] = ax;
      g.a[N + n] = ay;
#pragma unroll
      for (int q = 0; q < 9; ++q) pop_set<kMomentum>(g.fbuf, g, q * N + n, pf[q]);
    }
#pragma unroll
    for (int q = 0; q < 9; ++q) phase_store<0x1u>(g.hbuf, g, q, n, phi, ph[q]);
    if (phase_relative(g)) g.phase_ref[n] = phi;
  }
  if (with_momentum) block_partials<3>(load, g.partials, blk);
}
// The cut-link preparation alone, in place on fbuf (test helper of the
// reference's own tests around simulator.py:4798-4866).
__device__ __forceinline__ void k2_prepare_cut_links(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk), N = cells(g);
  double load[3] = {0.0, 0.0, 0.0};
  if (n < N) {
    const int i = n / g.ny, j = n - i * g.ny;
    if (fluid_at(g, i, j)) {
      float raw[9];
#pragma unroll
      for (int q = 0; q < 9; ++q) raw[q] = pop_get<kMomentum>(g.fbuf, g, q * N + n);
      const float ux = g.u[n] + 0.5f * g.a[n], uy = g.u[N + n] + 0.5f * g.a[N + n];
      float poly[9];
#pragma unroll
      for (int q = 0; q < 9; ++q) poly[q] = momentum_poly<true>(q, ux * ux + uy * uy, ux, uy);
      prepare_cut_links(g, load_pose(g), i, j, g.p[n] - g.p_ref[j], poly, raw, load);
#pragma unroll
      for (int q = 0; q < 9; ++q) pop_set<kMomentum>(g.fbuf, g, q * N + n, raw[q]);
    }
  }
  block_partials<3>(load, g.partials, blk);
}

// Pull streaming + macroscopic update (simulator.py:3699-3825).
template <int Q>
__device__ __forceinline__ void pull(const icy2d_grid& g, const Pose& pose, int i, int j, int n, float phi_old,
                                     bool phase_only, float& fq, float& hq) {
  const int N = cells(g);
  const int si = i - cxq(Q), sj = j - cyq(Q);  // source of population Q
  if (Q == 0 || (inside(g, si, sj) && fluid_at(g, si, sj))) {
    const int m = Q == 0 ? n : at(g, si, sj);
    if (!phase_only) fq = pop_get<kMomentum>(g.fbuf, g, Q * N + m);
    hq = phase_decoded<false>(g, Q, pop_get<kPhase>(g.hbuf, g, Q * N + m), hbuf_ref(g, m));
  } else {
    constexpr int out = oppq(Q);  // own population sent towards (si, sj)
    if (!phase_only) fq = pop_get<kMomentum>(g.fbuf, g, out * N + n);
    float ho = phase_decoded<false>(g, out, pop_get<kPhase>(g.hbuf, g, out * N + n), hbuf_ref(g, n));
    if (inside(g, si, sj) && g.solid[at(g, si, sj)] == 1) {
      const float eta = cut_fraction(g, pose, i, j, si, sj);
      float ub[2];
      body_velocity(pose, (i + 0.5f) + eta * (float)cxq(out), (j + 0.5f) + eta * (float)cyq(out), ub);
      ho -= 6.0f * wq(out) * phi_old * ((float)cxq(out) * ub[0] + (float)cyq(out) * ub[1]);
    }
    hq = ho;
  }
}
// mode bit 0: stream (pull); bit 1: update phi, u (and the pressure's
// population sum) from the cell's populations, as the reference's separate
// macroscopic kernel does after streaming.  The step runs both in one pass.
constexpr int kStreamPull = 1, kStreamUpdate = 2;
// A kernel for each mode: the pulls' registers (cut links) would leave the
// update alone, which moves most bytes, five waves a SIMD instead of eight, and its
// loads wait for the label (269 us over the 64-case ensemble, 146).
template <int mode>
__device__ __forceinline__ void k2_stream(const icy2d_grid& g, const int blk, int phase_only) {
  const int n = cell_index(blk), N = cells(g);
  if (n >= N) return;
  const int i = n / g.ny, j = n - i * g.ny;
  // FP64 sine and cosine: for the pulled links and ice cells only.
  const bool posed = (mode & kStreamPull) || g.solid[n] == 1;
  Pose pose = {};
  if (posed) pose = load_pose(g);
  const bool po = phase_only != 0;
  constexpr bool pulling = mode & kStreamPull, update = mode & kStreamUpdate;
  const float phi_old = g.phi[n];
  uint32_t own_f[9] = {}, own_h[9] = {};  // loaded before the label is waited for
  if (!pulling) {
#pragma unroll
    for (int q = 0; q < 9; ++q) {
      own_h[q] = pop_raw<kPhase>(g.h, g, q * N + n);
      if (!po) own_f[q] = pop_raw<kMomentum>(g.f, g, q * N + n);
    }
  }
  if (fluid_at(g, i, j)) {
    float f[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, h[9];
    if (pulling) {
      pull<0>(g, pose, i, j, n, phi_old, po, f[0], h[0]);
      pull<1>(g, pose, i, j, n, phi_old, po, f[1], h[1]);
      pull<2>(g, pose, i, j, n, phi_old, po, f[2], h[2]);
      pull<3>(g, pose, i, j, n, phi_old, po, f[3], h[3]);
      pull<4>(g, pose, i, j, n, phi_old, po, f[4], h[4]);
      pull<5>(g, pose, i, j, n, phi_old, po, f[5], h[5]);
      pull<6>(g, pose, i, j, n, phi_old, po, f[6], h[6]);
      pull<7>(g, pose, i, j, n, phi_old, po, f[7], h[7]);
      pull<8>(g, pose, i, j, n, phi_old, po, f[8], h[8]);
    } else {
#pragma unroll
      for (int q = 0; q < 9; ++q) {
        h[q] = phase_decoded<true>(g, q, pop_value<kPhase>(g, own_h[q]), phi_old);
        if (!po) f[q] = pop_value<kMomentum>(g, own_f[q]);
      }
    }
    float phi = phi_old;
    if (update) {
      phi = 0.0f;
#pragma unroll
      for (int q = 0; q < 9; ++q) phi += h[q];
    }
    // h is stored against the phase this pass leaves in phi[n]
    if (pulling || (update && phase_relative(g))) {
#pragma unroll
      for (int q = 0; q < 9; ++q) {
        phase_store<0x23u>(g.h, g, q, n, phi, h[q]);
        if (pulling && !po) pop_set<kMomentum>(g.f, g, q * N + n, f[q]);
      }
    }
    if (!update) return;
    g.phi[n] = phi;
    if (!po) {
      float mx = 0.0f, my = 0.0f, moving = 0.0f;
#pragma unroll
      for (int q = 0; q < 9; ++q) {
        if (cxq(q)) mx += (float)cxq(q) * f[q];
        if (cyq(q)) my += (float)cyq(q) * f[q];
        if (q) moving += f[q];
      }
      const float rho = fmaxf(mixture(g, phi), 1.0e-12f);
      g.u[n] = mx / rho;
      g.u[N + n] = my / rho;
      g.moving[n] = moving;
    }
  } else if (update) {
    if (wall_at(g, i, j)) g.phi[n] = 0.0f;
    if (!po) {
      float v[2] = {0.0f, 0.0f};
      if (g.solid[n] == 1) body_velocity(pose, i + 0.5f, j + 0.5f, v);
      g.u[n] = v[0];
      g.u[N + n] = v[1];
      g.a[n] = g.a[N + n] = 0.0f;
    }
  }
}
// A population plane element copied as stored (FP16 or FP32).
template <int Kind>
__device__ __forceinline__ void pop_copy(float* dst, const float* src, const icy2d_grid& g, int idx) {
  if (half_storage<Kind>(g)) reinterpret_cast<__half*>(dst)[idx] = reinterpret_cast<const __half*>(src)[idx];
  else dst[idx] = src[idx];
}

// The step's collision and streaming in one pass (simulator.py:3241-3738):
// each fluid cell collides as k2_collide does and pushes every
// post-collision population straight to its destination in fbuf and hbuf
// (population q to x + c_q when that cell is fluid; otherwise it comes back
// to x itself as population opp(q), with the moving-ice phase term), which
// is where the pull stream of k2_stream would fetch it from.  No block reads
// what another writes: f and h are read, fbuf and hbuf written.  A
// non-fluid cell's stored populations are carried over to fbuf and hbuf.
// The caller swaps f/fbuf and h/hbuf and then runs the macroscopic update
// (k2_stream<2>), which reads only the cell's own populations.  A phase
// population stored relative to the phase (bit 3) is stored against its
// destination's phase, which the update decodes it with.
__device__ __forceinline__ void k2_collide_push(const icy2d_grid& g, const int blk) {
  __shared__ CollideTile tile;
  const int N = cells(g);
  const int rows = (int)blockDim.x / kTileCols, tiles_j = (g.ny + kTileCols - 1) / kTileCols;
  const int i0 = (blk / tiles_j) * rows, j0 = (blk % tiles_j) * kTileCols;
  const int li = (int)threadIdx.x / kTileCols, lj = (int)threadIdx.x % kTileCols;
  const int i = i0 + li, j = j0 + lj;
  OwnCell own = {};
  if (i < g.nx && j < g.ny) load_own(g, at(g, i, j), 1, own);
  stage_window(g, tile, i0, j0, rows);
  __syncthreads();
  double load[3] = {0.0, 0.0, 0.0};
  if (i < g.nx && j < g.ny) {
    const int n = at(g, i, j);
    if (tile.fluid[li + 2][lj + 2]) {
      const bool near = beside_ice(tile, li + 1, lj + 1);
      Pose pose = {};
      if (near) pose = load_pose(g);
      const float phi = tile.phi[li + 2][lj + 2];
      float pf[9], ph[9], ax, ay;
      collide_cell<true>(g, own, near, pose, tile, li + 2, lj + 2, li + 1, lj + 1, i, j, n, 1, pf, ph, ax, ay, load);
      g.a[n] = ax;
      g.a[N + n] = ay;
      pop_set<kMomentum>(g.fbuf, g, n, pf[0]);
      phase_store<0x1u>(g.hbuf, g, 0, n, phi, ph[0]);
#pragma unroll
      for (int q = 1; q < 9; ++q) {
        const int di = cxq(q), dj = cyq(q);
        if (tile.fluid[li + 2 + di][lj + 2 + dj]) {
          const int m = at(g, i + di, j + dj);
          pop_set<kMomentum>(g.fbuf, g, q * N + m, pf[q]);
          phase_store<0u>(g.hbuf, g, q, m, phase_relative(g) ? tile.phi[li + 2 + di][lj + 2 + dj] : 0.0f, ph[q]);
        } else {
          float ho = ph[q];
          if (tile.kind[li + 1 + di][lj + 1 + dj] == 1) {
            const float eta = cut_fraction(g, pose, i, j, i + di, j + dj);
            float ub[2];
            body_velocity(pose, (i + 0.5f) + eta * (float)di, (j + 0.5f) + eta * (float)dj, ub);
            ho -= 6.0f * wq(q) * phi * ((float)di * ub[0] + (float)dj * ub[1]);
          }
          const int o = oppq(q);
          pop_set<kMomentum>(g.fbuf, g, o * N + n, pf[q]);
          phase_store<0u>(g.hbuf, g, o, n, phi, ho);
        }
      }
    } else {
#pragma unroll
      for (int q = 0; q < 9; ++q) {
        pop_copy<kMomentum>(g.fbuf, g.f, g, q * N + n);
        pop_copy<kPhase>(g.hbuf, g.h, g, q * N + n);
      }
    }
  }
  block_partials<3>(load, g.partials, blk);
}
// simulator.py:3860-3897
__device__ __forceinline__ void k2_update_pressure(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk), N = cells(g);
  if (n >= N) return;
  const int i = n / g.ny, j = n - i * g.ny;
  if (fluid_at(g, i, j)) {
    const float phi = g.phi[n], rho = mixture(g, phi);
    const float ux = g.u[n] + 0.5f * g.a[n], uy = g.u[N + n] + 0.5f * g.a[N + n];
    float gx = 0.0f, gy = 0.0f;
#pragma unroll
    for (int q = 1; q < 9; ++q) {
      const float nb = phase_neighbor(g, i, j, cxq(q), cyq(q), 1, phi);
      if (cxq(q)) gx += 3.0f * wq(q) * (float)cxq(q) * (nb - phi);
      if (cyq(q)) gy += 3.0f * wq(q) * (float)cyq(q) * (nb - phi);
    }
    const float drho = g.rho_w - g.rho_a;
    const float s0 = -1.5f * wq(0) * (ux * ux + uy * uy);
    const float dynamic = 0.6f * (g.moving[n] + 0.5f * (ux * drho * gx + uy * drho * gy) + rho * s0);
    g.p[n] = g.p_ref[j] + dynamic;
  } else if (wall_at(g, i, j)) {
    g.p[n] = 0.0f;
  }
}
// simulator.py:3163-3236
__device__ __forceinline__ void k2_refill(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk), N = cells(g);
  if (n >= N) return;
  const int i = n / g.ny, j = n - i * g.ny;
  if (wall_at(g, i, j)) return;
  const bool became_solid = g.prev_solid[n] == 0 && g.solid[n] == 1;
  const bool became_fluid = g.prev_solid[n] == 1 && g.solid[n] == 0;
  if (!became_solid && !became_fluid) return;
  const Pose pose = load_pose(g);
  if (became_solid) {
    float v[2];
    body_velocity(pose, i + 0.5f, j + 0.5f, v);
    g.phi[n] = clamp01(g.phi[n]);
    g.u[n] = v[0];
    g.u[N + n] = v[1];
    g.a[n] = g.a[N + n] = 0.0f;
    g.p[n] = g.p[n] - g.p_ref[j];
    return;
  }
  float phi_sum = 0.0f, p_sum = 0.0f, vx = 0.0f, vy = 0.0f, count = 0.0f;
  for (int di = -1; di <= 1; ++di)
    for (int dj = -1; dj <= 1; ++dj) {
      const int ni = i + di, nj = j + dj;
      if ((di || dj) && inside(g, ni, nj) && fluid_at(g, ni, nj) && g.prev_solid[at(g, ni, nj)] == 0) {
        const int m = at(g, ni, nj);
        phi_sum += clamp01(g.phi[m]);
        p_sum += g.p[m] - g.p_ref[nj];
        vx += g.u[m];
        vy += g.u[N + m];
        count += 1.0f;
      }
    }
  float phi0 = clamp01(g.phi[n]), p0 = g.p[n], v[2];
  body_velocity(pose, i + 0.5f, j + 0.5f, v);
  if (count > 0.0f) {
    phi0 = phi_sum / count;
    p0 = p_sum / count;
    v[0] = vx / count;
    v[1] = vy / count;
  }
  p0 += g.p_ref[j];
  const float rho = mixture(g, phi0);
  g.phi[n] = phi0;
  g.u[n] = v[0];
  g.u[N + n] = v[1];
  g.a[n] = g.a[N + n] = 0.0f;
  g.p[n] = p0;
  const float pdyn = p0 - g.p_ref[j];
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    pop_set<kMomentum>(g.f, g, q * N + n, momentum_eq_rt(q, pdyn, rho, v[0], v[1]));
    phase_set(g.h, g, q, n, phi0, phase_eq_rt(q, phi0, v[0], v[1]));
  }
}
// simulator.py:2303-2338 (per-block maxima as partials)
__device__ __forceinline__ void k2_outflow_partials(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk), N = cells(g);
  double best = 0.0;
  if (n < N) {
    const int i = n / g.ny, j = n - i * g.ny;
    // Labels and phases of the cell and its neighbours in one go (nested in
    // the tests they cost a memory latency each: 145 us over the 64-case
    // ensemble, 84).
    const int off[5][2] = {{0, 0}, {1, 0}, {-1, 0}, {0, 1}, {0, -1}};
    int m[5];
    float phase[5];
    bool open[5];
    int label[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const int ni = i + off[k][0], nj = j + off[k][1];
      open[k] = !wall_at(g, ni, nj);  // and so inside
      m[k] = open[k] ? at(g, ni, nj) : n;
      label[k] = g.solid[m[k]];
      phase[k] = g.phi[m[k]];
    }
    bool wet[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) wet[k] = open[k] && label[k] == 0 && phase[k] > g.cutoff;
    if (wet[0]) {
      const float vx = g.u[n] + 0.5f * g.a[n], vy = g.u[N + n] + 0.5f * g.a[N + n];
      float outflow = 0.0f, wx[5], wy[5];
#pragma unroll
      for (int k = 1; k < 5; ++k) {
        const int w = wet[k] ? m[k] : n;
        wx[k] = g.u[w] + 0.5f * g.a[w];
        wy[k] = g.u[N + w] + 0.5f * g.a[N + w];
      }
#pragma unroll
      for (int k = 1; k < 5; ++k)
        if (wet[k])
          outflow += fmaxf(0.0f, (float)off[k][0] * (0.5f * (vx + wx[k])) + (float)off[k][1] * (0.5f * (vy + wy[k])));
      if (!isfinite(vx) || !isfinite(vy)) outflow = INFINITY;
      best = outflow;
    }
  }
  __shared__ double part[16];
  const double wave_best = wave_max(best);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = wave_best;
  __syncthreads();
  if (threadIdx.x == 0) {
    double r = part[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r = fmax(r, part[w]);
    g.partials[blk] = r;
  }
}
__device__ __forceinline__ void k2_store_outflow(const icy2d_grid& g, const int blk) {
  g.control->max_outflow = (float)g.partials[g.partials_capacity - 1];
}

// ----------------------------------------------------- volume projection
__device__ __forceinline__ void lift_phase(const icy2d_grid& g, int n, int j, float old_phase, float new_phase) {
  const int N = cells(g);
  const float ux = g.u[n], uy = g.u[N + n], pdyn = g.p[n] - g.p_ref[j];
  const float ro = mixture(g, old_phase), rn = mixture(g, new_phase), uu = ux * ux + uy * uy;
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const float poly = momentum_poly<false>(q, uu, ux, uy);
    pop_add<kMomentum>(g.f, g, q * N + n, momentum_eq_of(q, pdyn, rn, poly) - momentum_eq_of(q, pdyn, ro, poly));
  }
  const float stored = g.phi[n];
  float lifted[9], sum = 0.0f;
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const float poly = phase_poly<false, false>(q, uu, ux, uy);
    lifted[q] = fmaf(wq(q) * new_phase, poly, phase_decoded<true>(g, q, pop_get<kPhase>(g.h, g, q * N + n), stored));
    lifted[q] = fmaf(-(wq(q) * old_phase), poly, lifted[q]);
    sum += lifted[q];
  }
  lifted[0] += new_phase - sum;
#pragma unroll
  for (int q = 0; q < 9; ++q) phase_store<0x1u>(g.h, g, q, n, new_phase, lifted[q]);
  g.phi[n] = new_phase;
}
// simulator.py:4150-4229
__device__ __forceinline__ void k2_clip_phase(const icy2d_grid& g, const int blk, double max_bulk_l1) {
  const int n = cell_index(blk), N = cells(g);
  double v[1] = {0.0};
  if (n < N) {
    const int i = n / g.ny, j = n - i * g.ny;
    const float old_phase = g.phi[n];
    uint32_t own[9];  // loaded before the label is waited for
#pragma unroll
    for (int q = 0; q < 9; ++q) own[q] = pop_raw<kPhase>(g.h, g, q * N + n);
    if (fluid_at(g, i, j)) {
      float bounded = clamp01(old_phase);
      if (bounded <= g.cutoff) bounded = 0.0f;
      else if (bounded >= 1.0f - g.cutoff) bounded = 1.0f;
      if (bounded != old_phase) {
        const float ux = g.u[n], uy = g.u[N + n];
        const float pdyn = g.p[n] - g.p_ref[j];
        const float ro = mixture(g, old_phase), rn = mixture(g, bounded);
#pragma unroll
        for (int q = 0; q < 9; ++q) {
          const float poly = momentum_poly<false>(q, ux * ux + uy * uy, ux, uy);
          pop_add<kMomentum>(g.f, g, q * N + n, momentum_eq_of(q, pdyn, rn, poly) - momentum_eq_of(q, pdyn, ro, poly));
        }
      }
      float h[9], l1 = 0.0f;
#pragma unroll
      for (int q = 0; q < 9; ++q) {
        h[q] = phase_decoded<true>(g, q, pop_value<kPhase>(g, own[q]), old_phase);
        l1 += fabsf(h[q]);
      }
      const bool regularize = (bounded == 0.0f || bounded == 1.0f) && (double)l1 > max_bulk_l1;
      if (regularize || bounded != old_phase) {
        const float ux = g.u[n], uy = g.u[N + n];
        const float px = ux + 0.5f * g.a[n], py = uy + 0.5f * g.a[N + n];
        if (regularize) {
#pragma unroll
          for (int q = 0; q < 9; ++q) h[q] = wq(q) * bounded * phase_poly<true, false>(q, px * px + py * py, px, py);
        } else {
#pragma unroll
          for (int q = 0; q < 9; ++q) {
            const float poly = phase_poly<true, false>(q, ux * ux + uy * uy, ux, uy);
            h[q] = fmaf(-(wq(q) * old_phase), poly, fmaf(wq(q) * bounded, poly, h[q]));
          }
        }
        float sum = 0.0f;
#pragma unroll
        for (int q = 0; q < 9; ++q) sum += h[q];
        h[0] += bounded - sum;
#pragma unroll
        for (int q = 0; q < 9; ++q) phase_store<0u>(g.h, g, q, n, bounded, h[q]);
      }
      g.phi[n] = bounded;
      v[0] = (double)bounded;
    }
  }
  block_partials<1>(v, g.partials, blk);
}
// simulator.py:4231-4257; the two masks are hbuf planes 0 and 1
__device__ __forceinline__ void k2_seed_projection(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk), N = cells(g);
  if (n >= N) return;
  const int i = n / g.ny, j = n - i * g.ny;
  int seed = 0;
  if (fluid_at(g, i, j)) {
    const float phase = g.phi[n];
    if (g.cutoff < phase && phase < 1.0f - g.cutoff) {
      if (phase == 0.5f) seed = 1;
      for (int di = -1; di <= 1; ++di)
        for (int dj = -1; dj <= 1; ++dj) {
          const int ni = i + di, nj = j + dj;
          if ((di || dj) && inside(g, ni, nj) && fluid_at(g, ni, nj)) {
            const float nb = g.phi[at(g, ni, nj)];
            if ((phase < 0.5f && 0.5f <= nb) || (nb < 0.5f && 0.5f <= phase)) seed = 1;
          }
        }
    }
  }
  pop_set<kPhase>(g.hbuf, g, n, (float)seed);
  pop_set<kPhase>(g.hbuf, g, N + n, 0.0f);
}
// simulator.py:4259-4289
__device__ __forceinline__ void k2_dilate_projection(const icy2d_grid& g, const int blk, int primary_to_next) {
  const int n = cell_index(blk), N = cells(g);
  if (n >= N) return;
  const int src = primary_to_next ? 0 : N, dst = primary_to_next ? N : 0;
  const int i = n / g.ny, j = n - i * g.ny;
  int value = 0;
  const float phase = g.phi[n];
  if (fluid_at(g, i, j) && g.cutoff < phase && phase < 1.0f - g.cutoff) {
    value = (int)pop_get<kPhase>(g.hbuf, g, src + n);
    if (value == 0)
      for (int di = -1; di <= 1; ++di)
        for (int dj = -1; dj <= 1; ++dj) {
          const int ni = i + di, nj = j + dj;
          if ((di || dj) && inside(g, ni, nj) && pop_get<kPhase>(g.hbuf, g, src + at(g, ni, nj)) == 1.0f) value = 1;
        }
  }
  pop_set<kPhase>(g.hbuf, g, dst + n, (float)value);
}
// All R dilation sweeps of simulator.py:4259-4289 in one pass: a block stages
// a (16 + 2R) x (64 + 2R) window of the seed flags and the sweep mask
// (fluid, cutoff < phi < 1 - cutoff) in LDS, runs the R sweeps there
// (new = mask & (old | any of the 8 neighbours)), and writes the exact
// central 16 x 64 cells: after R sweeps a cell depends only on flags within
// R cells.  Blocks read the seeds from the primary plane and write the band
// to the second plane (no block reads what another writes); k2_copy_band then
// moves it to the primary plane, where the reference's ping-pong (R even)
// ends.
constexpr int kBandI = 16, kBandJ = 64, kMaxBand = 16;
constexpr int kBandRows = kBandI + 2 * kMaxBand, kBandWords = (kBandJ + 2 * kMaxBand + 31) / 32;
// Rows of the window are bit sets (bit b of word b / 32 = column b): one
// sweep is new = mask & dilate3x3(old), the 3x3 dilation a horizontal
// shift-or followed by an or of the row above and below.
__device__ __forceinline__ void k2_dilate_band(const icy2d_grid& g, const int blk, int radius) {
  __shared__ uint32_t flag[kBandRows][kBandWords], sweep[kBandRows][kBandWords], horiz[kBandRows][kBandWords];
  const int tiles_j = (g.ny + kBandJ - 1) / kBandJ;
  const int i0 = (blk / tiles_j) * kBandI - radius, j0 = (blk % tiles_j) * kBandJ - radius;
  const int H = kBandI + 2 * radius, W = kBandJ + 2 * radius, words = (W + 31) / 32;
  for (int e = threadIdx.x; e < kBandRows * kBandWords; e += blockDim.x) {
    (&flag[0][0])[e] = 0u;
    (&sweep[0][0])[e] = 0u;
  }
  __syncthreads();
  int any = 0;
  for (int e = threadIdx.x; e < H * W; e += blockDim.x) {
    const int a = e / W, b = e - a * W, i = i0 + a, j = j0 + b;
    if (inside(g, i, j) && fluid_at(g, i, j)) {
      const float phase = g.phi[at(g, i, j)];
      if (g.cutoff < phase && phase < 1.0f - g.cutoff) {
        const uint32_t bit = 1u << (b & 31);
        atomicOr(&sweep[a][b >> 5], bit);
        if (pop_get<kPhase>(g.hbuf, g, at(g, i, j)) == 1.0f) {
          atomicOr(&flag[a][b >> 5], bit);
          any = 1;
        }
      }
    }
  }
  // A window without seeds leaves no band: all of its central cells are 0.
  if (__syncthreads_or(any)) {
    for (int it = 0; it < radius; ++it) {
      for (int e = threadIdx.x; e < H * words; e += blockDim.x) {
        const int a = e / words, w = e - a * words;
        const uint32_t f = flag[a][w];
        const uint32_t left = (f << 1) | (w > 0 ? flag[a][w - 1] >> 31 : 0u);
        const uint32_t right = (f >> 1) | (w + 1 < words ? flag[a][w + 1] << 31 : 0u);
        horiz[a][w] = f | left | right;
      }
      __syncthreads();
      for (int e = threadIdx.x; e < H * words; e += blockDim.x) {
        const int a = e / words, w = e - a * words;
        uint32_t v = horiz[a][w];
        if (a > 0) v |= horiz[a - 1][w];
        if (a + 1 < H) v |= horiz[a + 1][w];
        flag[a][w] = v & sweep[a][w];
      }
      __syncthreads();
    }
  } else {
    for (int e = threadIdx.x; e < kBandRows * kBandWords; e += blockDim.x) (&flag[0][0])[e] = 0u;
    __syncthreads();
  }
  for (int e = threadIdx.x; e < kBandI * kBandJ; e += blockDim.x) {
    const int a = e / kBandJ, b = e - a * kBandJ, i = i0 + radius + a, j = j0 + radius + b;
    const int col = radius + b;
    if (i < g.nx && j < g.ny)
      pop_set<kPhase>(g.hbuf, g, cells(g) + at(g, i, j), (float)((flag[radius + a][col >> 5] >> (col & 31)) & 1u));
  }
}
__device__ __forceinline__ void k2_copy_band(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk), N = cells(g);
  if (n < N) pop_set<kPhase>(g.hbuf, g, n, pop_get<kPhase>(g.hbuf, g, N + n));
}
// simulator.py:4291-4351
__device__ __forceinline__ void k2_evaluate_projection(const icy2d_grid& g, const int blk, double lambda) {
  double v[kRun][2] = {};
#pragma unroll
  for (int r = 0; r < kRun; ++r) {
    const int first = (blk * kRun + r) * kBlock, n = first + (int)threadIdx.x;
    if (n >= cells(g)) continue;
    int i, j;
    row_col(g, first, n, i, j);
    const double phase = g.phi[n];
    const bool flagged = pop_get<kPhase>(g.hbuf, g, n) == 1.0f;
    if (fluid_at(g, i, j)) {
      double mapped = phase;
      const bool adjustable = flagged;
      if (adjustable) {
        const double e = exp(lambda);
        mapped = phase * e / (1.0 - phase + phase * e);
      }
      float m32 = (float)mapped;
      if (m32 <= g.cutoff) m32 = 0.0f;
      else if (m32 >= 1.0f - g.cutoff) m32 = 1.0f;
      v[r][0] = (double)m32;
      if (adjustable && g.cutoff < m32 && m32 < 1.0f - g.cutoff) v[r][1] = (double)m32 * (1.0 - (double)m32);
    }
  }
  run_partials<2>(g, v, blk);
}
// simulator.py:4353-4406
__device__ __forceinline__ void k2_apply_projection(const icy2d_grid& g, const int blk, double lambda) {
  const double e = exp(lambda);
  const int n = cell_index(blk);
  double v[1] = {0.0};
  if (n < cells(g)) {
    const int i = n / g.ny, j = n - i * g.ny;
    if (fluid_at(g, i, j)) {
      const float old_phase = g.phi[n];
      float new_phase = old_phase;
      if (pop_get<kPhase>(g.hbuf, g, n) == 1.0f) {
        const double p = old_phase;
        new_phase = (float)(p * e / (1.0 - p + p * e));
      }
      if (new_phase <= g.cutoff) new_phase = 0.0f;
      else if (new_phase >= 1.0f - g.cutoff) new_phase = 1.0f;
      if (new_phase != old_phase) lift_phase(g, n, j, old_phase, new_phase);
      v[0] = (double)new_phase;
    }
  }
  block_partials<1>(v, g.partials, blk);
}
__device__ __forceinline__ bool residual_free(const icy2d_grid& g, int n, double phase, double residual) {
  const double margin = 4.0 * 1.1920928955078125e-07;
  const double cutoff = g.cutoff;
  if (!(pop_get<kPhase>(g.hbuf, g, n) == 1.0f && cutoff < phase && phase < 1.0 - cutoff)) return false;
  const double magnitude = fabs(residual);
  if (residual > 0.0) return 1.0 - cutoff - phase > magnitude + margin;
  return phase - cutoff > magnitude + margin;
}
// simulator.py:4408-4431
__device__ __forceinline__ void k2_residual_weight(const icy2d_grid& g, const int blk, double residual) {
  const int n = cell_index(blk);
  double v[1] = {0.0};
  if (n < cells(g)) {
    const int i = n / g.ny, j = n - i * g.ny;
    const double phase = g.phi[n];
    if (fluid_at(g, i, j) && residual_free(g, n, phase, residual)) v[0] = phase * (1.0 - phase);
  }
  block_partials<1>(v, g.partials, blk);
}
// simulator.py:4433-4492
__device__ __forceinline__ void k2_apply_residual(const icy2d_grid& g, const int blk, double residual, double total_weight) {
  const int n = cell_index(blk);
  double v[1] = {0.0};
  if (n < cells(g)) {
    const int i = n / g.ny, j = n - i * g.ny;
    if (fluid_at(g, i, j)) {
      const float old_phase = g.phi[n];
      float new_phase = old_phase;
      const double p = old_phase;
      if (residual_free(g, n, p, residual) && total_weight > 0.0)
        new_phase = (float)(p + residual * (p * (1.0 - p)) / total_weight);
      if (new_phase != old_phase) lift_phase(g, n, j, old_phase, new_phase);
      v[0] = (double)new_phase;
    }
  }
  block_partials<1>(v, g.partials, blk);
}

// ------------------------------------------------------- mass properties
// simulator.py:3014-3044 over the material grid
__device__ __forceinline__ void k2_mass_partials(const icy2d_grid& g, const int blk) {
  const int k = cell_index(blk);
  double v[4] = {0.0, 0.0, 0.0, 0.0};
  if (k < g.body_nx * g.body_ny) {
    const int bi = k / g.body_ny, bj = k - bi * g.body_ny;
    const double mass = g.body_mass[k] * (1.0 / (g.rho_w_si * g.area));
    const double fraction = (double)body_fraction(g, bi, bj);
    const double lx = bi + 0.5 - 0.5 * g.body_nx, ly = bj + 0.5 - 0.5 * g.body_ny;
    v[0] = mass;
    v[1] = mass * lx;
    v[2] = mass * ly;
    v[3] = mass * (lx * lx + ly * ly + fraction / 6.0);
  }
  block_partials<4>(v, g.partials, blk);
}
// simulator.py:3046-3161
__device__ __forceinline__ void k2_apply_mass_properties(const icy2d_grid& g, const int blk, int initialize) {
  icy2d_control* ctl = g.control;
  const double reduced = ctl->reduced[0], old_mass = ctl->mass, initial = g.initial_mass;
  const double tol = 1.0e-12 * fmax(initial, 1.0);
  double new_mass = reduced;
  bool hold = false;
  if (!initialize && reduced > 0.0 && (fabs(reduced - old_mass) <= tol || reduced > old_mass)) {
    new_mass = old_mass;
    hold = true;
  }
  const double inactive_mass = fmax(1.0e-12, 1.0e-14 * fmax(initial, 1.0));
  const double inactive_inertia = 1.0e-14 * fmax(g.initial_inertia, 1.0);
  const bool resolved = new_mass > inactive_mass, was_active = ctl->inertia > 0.0;
  const double old_com[2] = {ctl->local_com[0], ctl->local_com[1]};
  double new_com[2] = {old_com[0], old_com[1]}, raw_inertia = 0.0;
  if (resolved) {
    if (hold) {
      raw_inertia = ctl->inertia;
    } else {
      new_com[0] = ctl->reduced[1] / new_mass;
      new_com[1] = ctl->reduced[2] / new_mass;
      raw_inertia = ctl->reduced[3] - new_mass * (new_com[0] * new_com[0] + new_com[1] * new_com[1]);
    }
    raw_inertia = fmax(raw_inertia, 0.0);
  }
  const bool mechanical = resolved && raw_inertia > inactive_inertia && (initialize || was_active);
  const double new_inertia = mechanical ? raw_inertia : 0.0;
  const Pose p = load_pose(g);
  const double c = p.c, s = p.s;
  const double ow[2] = {c * old_com[0] - s * old_com[1], s * old_com[0] + c * old_com[1]};
  const double nw[2] = {c * new_com[0] - s * new_com[1], s * new_com[0] + c * new_com[1]};
  const bool retiring = was_active && !mechanical;
  if (!initialize && (new_mass < old_mass || retiring)) {
    const double v0[2] = {ctl->velocity[0], ctl->velocity[1]}, omega = ctl->omega;
    double sv[2] = {0.0, 0.0};
    if (mechanical) {
      sv[0] = v0[0] - omega * (nw[1] - ow[1]);
      sv[1] = v0[1] + omega * (nw[0] - ow[0]);
    }
    const float sv32[2] = {(float)sv[0], (float)sv[1]};
    const double svs[2] = {sv32[0], sv32[1]};
    const double nc[2] = {(double)(float)((double)p.ox + nw[0]), (double)(float)((double)p.oy + nw[1])};
    const double oc[2] = {p.cx, p.cy};
    ctl->melted[0] += old_mass * v0[0] - new_mass * svs[0];
    ctl->melted[1] += old_mass * v0[1] - new_mass * svs[1];
    const double ob[2] = {old_mass * v0[0], old_mass * v0[1]}, nb[2] = {new_mass * svs[0], new_mass * svs[1]};
    const double old_l = oc[0] * ob[1] - oc[1] * ob[0] + ctl->inertia * omega;
    const double new_l = nc[0] * nb[1] - nc[1] * nb[0] + new_inertia * omega;
    ctl->melted[2] += old_l - new_l;
    ctl->velocity[0] = sv32[0];
    ctl->velocity[1] = sv32[1];
  }
  ctl->local_com[0] = new_com[0];
  ctl->local_com[1] = new_com[1];
  ctl->mass = new_mass;
  ctl->inertia = new_inertia;
  if (!mechanical) {
    ctl->velocity[0] = ctl->velocity[1] = 0.0f;
    ctl->omega = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) ctl->support[k] = 0.0f;
  }
}

// -------------------------------------------------------- melt momentum
// Fluid momentum (x, y, angular about the origin) of simulator.py:2735-2760.
__device__ __forceinline__ void k2_momentum_partials(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk), N = cells(g);
  double v[3] = {0.0, 0.0, 0.0};
  if (n < N) {
    const int i = n / g.ny, j = n - i * g.ny;
    if (fluid_at(g, i, j)) {
      double mx = 0.0, my = 0.0;
#pragma unroll
      for (int q = 0; q < 9; ++q) {
        const double fv = pop_get<kMomentum>(g.f, g, q * N + n);
        if (cxq(q)) mx += (double)cxq(q) * fv;
        if (cyq(q)) my += (double)cyq(q) * fv;
      }
      v[0] = mx;
      v[1] = my;
      v[2] = (i + 0.5) * my - (j + 0.5) * mx;
    }
  }
  block_partials<3>(v, g.partials, blk);
}
__device__ __forceinline__ void k2_snapshot_body(const icy2d_grid& g, const int blk) {
  icy2d_control* ctl = g.control;
  for (int k = 0; k < 3; ++k) ctl->body_before[k] = ctl->melted[k];
}
// simulator.py:2762-2797: wet weight and the min/max wet cell codes
__device__ __forceinline__ void k2_wet_partials(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk);
  double v[1] = {0.0};
  int lo = INT32_MAX, hi = -1;
  if (n < cells(g)) {
    const int i = n / g.ny, j = n - i * g.ny;
    const float phase = clamp01(g.phi[n]);
    if (fluid_at(g, i, j) && phase > g.cutoff) {
      v[0] = (double)phase;
      lo = hi = n;
    }
  }
  // The wet weight and the first and last wet cell as three block partials
  // (a sum, a minimum, a maximum; cell codes are exact in FP64), folded by
  // the finish like every other reduction.
  double w[3] = {v[0], lo >= 0 && lo < cells(g) ? (double)lo : 1.0e300, hi >= 0 ? (double)hi : -1.0e300};
  __shared__ double part[3][16];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const double r0 = wave_sum(w[0]), r1 = wave_min(w[1]), r2 = wave_max(w[2]);
  if (lane == 0) {
    part[0][wave] = r0;
    part[1][wave] = r1;
    part[2][wave] = r2;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const int k = threadIdx.x;
    double r = part[k][0];
    for (int q = 1; q < (int)(blockDim.x >> 6); ++q) r = k == 0 ? r + part[k][q] : k == 1 ? fmin(r, part[k][q]) : fmax(r, part[k][q]);
    g.partials[blk * 3 + k] = r;
  }
}
// The folded wet weight into wet[0] and the extreme wet cell codes into
// wet_target / wet_target_max (nx*ny and -1 without a wet cell), then the
// provisional momentum copy.
__device__ __forceinline__ void k2_store_wet(const icy2d_grid& g, const int blk) {
  icy2d_control* ctl = g.control;
  const double* t = g.partials + g.partials_capacity - 3;
  ctl->wet[0] = t[0];
  ctl->wet_target = t[1] < 1.0e299 ? (int)t[1] : g.nx * g.ny;
  ctl->wet_target_max = t[2] > -1.0e299 ? (int)t[2] : -1;
  for (int k = 0; k < 3; ++k) ctl->after[k] = ctl->provisional[k];  // as k2_copy_provisional
}
__device__ __forceinline__ void k2_reset_wet(const icy2d_grid& g, const int blk) {
  g.control->wet_target = g.nx * g.ny;
  g.control->wet_target_max = -1;
}
__device__ __forceinline__ void k2_copy_provisional(const icy2d_grid& g, const int blk) {
  icy2d_control* ctl = g.control;
  for (int k = 0; k < 3; ++k) ctl->after[k] = ctl->provisional[k];
}
__device__ __forceinline__ void melt_correction(const icy2d_control* ctl, double c[3]) {
  for (int k = 0; k < 3; ++k) c[k] = ctl->melted[k] - ctl->body_before[k] - (ctl->after[k] - ctl->before[k]);
}
// simulator.py:2799-2840: first and second moments of the wet weights
__device__ __forceinline__ void k2_weight_partials(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk);
  double v[3] = {0.0, 0.0, 0.0};
  if (n < cells(g)) {
    const int i = n / g.ny, j = n - i * g.ny;
    const float phase = clamp01(g.phi[n]);
    if (fluid_at(g, i, j) && phase > g.cutoff) {
      const double w = phase, px = i + 0.5, py = j + 0.5;
      v[0] = w * px;
      v[1] = w * py;
      v[2] = w * (px * px + py * py);
    }
  }
  block_partials<3>(v, g.partials, blk);
}
__device__ __forceinline__ void wet_geometry(const icy2d_control* ctl, double cen[2], double& polar) {
  cen[0] = cen[1] = 0.0;
  if (ctl->wet[0] > 1.0e-30) {
    cen[0] = ctl->wet[1] / ctl->wet[0];
    cen[1] = ctl->wet[2] / ctl->wet[0];
  }
  polar = fmax(0.0, ctl->wet[3] - ctl->wet[0] * (cen[0] * cen[0] + cen[1] * cen[1]));
}
__device__ __forceinline__ void k2_melt_status(const icy2d_grid& g, const int blk) {
  icy2d_control* ctl = g.control;
  double c[3], cen[2], polar;
  melt_correction(ctl, c);
  wet_geometry(ctl, cen, polar);
  const double norm = sqrt(c[0] * c[0] + c[1] * c[1]);
  int status = 0;
  if (ctl->wet[0] <= 1.0e-30) {
    if (norm > 1.0e-12 || fabs(c[2]) > 1.0e-12) status = -1;
  } else {
    const double couple = c[2] - (cen[0] * c[1] - cen[1] * c[0]);
    if (polar <= 1.0e-30 && fabs(couple) > 1.0e-12) status = -2;
    else if (norm > 1.0e-14 || fabs(c[2]) > 1.0e-14) status = 1;
  }
  ctl->melt_status = status;
}
__device__ __forceinline__ void add_momentum(const icy2d_grid& g, int n, double dmx, double dmy) {
  const int N = cells(g);
  const float mx = (float)dmx, my = (float)dmy;
  const float rho = fmaxf(mixture(g, clamp01(g.phi[n])), 1.0e-12f);
  g.u[n] += mx / rho;
  g.u[N + n] += my / rho;
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const float c_m = (float)cxq(q) * mx + (float)cyq(q) * my;
    pop_set<kMomentum>(g.f, g, q * N + n, fmaf(3.0f * wq(q), c_m, pop_get<kMomentum>(g.f, g, q * N + n)));
  }
}
// simulator.py:2842-2884
__device__ __forceinline__ void k2_apply_melt_correction(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk);
  if (n >= cells(g)) return;
  const icy2d_control* ctl = g.control;
  const int i = n / g.ny, j = n - i * g.ny;
  const float phase = clamp01(g.phi[n]);
  const double den = ctl->wet[0];
  if (!(fluid_at(g, i, j) && phase > g.cutoff) || !(den > 1.0e-30)) return;
  double c[3], cen[2], polar, scale = 0.0;
  melt_correction(ctl, c);
  wet_geometry(ctl, cen, polar);
  if (polar > 1.0e-30) scale = (c[2] - (cen[0] * c[1] - cen[1] * c[0])) / polar;
  const double w = phase, rx = i + 0.5 - cen[0], ry = j + 0.5 - cen[1];
  add_momentum(g, n, w * (c[0] / den - scale * ry), w * (c[1] / den + scale * rx));
}
// simulator.py:2905-2958
__device__ __forceinline__ void k2_local_melt_correction(const icy2d_grid& g, const int blk) {
  const icy2d_control* ctl = g.control;
  const int e1 = ctl->wet_target, e2 = ctl->wet_target_max, total = g.nx * g.ny;
  if (!(e1 >= 0 && e1 < total && e2 >= 0 && e2 < total && e1 != e2)) return;
  const int i1 = e1 / g.ny, j1 = e1 - i1 * g.ny, i2 = e2 / g.ny, j2 = e2 - i2 * g.ny;
  const double p1[2] = {i1 + 0.5, j1 + 0.5}, p2[2] = {i2 + 0.5, j2 + 0.5};
  double c[3];
  melt_correction(ctl, c);
  const double d[2] = {p1[0] - p2[0], p1[1] - p2[1]}, mid[2] = {0.5 * (p1[0] + p2[0]), 0.5 * (p1[1] + p2[1])};
  const double couple = c[2] - (mid[0] * c[1] - mid[1] * c[0]);
  const double dn = fmax(d[0] * d[0] + d[1] * d[1], 1.0e-30);
  const double qx = couple * -d[1] / dn, qy = couple * d[0] / dn;
  add_momentum(g, e1, 0.5 * c[0] + qx, 0.5 * c[1] + qy);
  add_momentum(g, e2, 0.5 * c[0] - qx, 0.5 * c[1] - qy);
}
// simulator.py:2960-2986
__device__ __forceinline__ void k2_finish_melt_momentum(const icy2d_grid& g, const int blk) {
  icy2d_control* ctl = g.control;
  for (int k = 0; k < 3; ++k) {
    ctl->carrier[k] += ctl->provisional[k] - ctl->before[k];
    ctl->correction[k] += ctl->after[k] - ctl->provisional[k];
  }
}

// ------------------------------------------------------------- thermal
__device__ __forceinline__ bool water_cell(const icy2d_grid& g, int i, int j) {
  const int n = at(g, i, j);
  return !wall_at(g, i, j) && g.solid[n] == 0 && g.phi[n] > g.cutoff;
}
// simulator.py:579-588
__device__ __forceinline__ void k2_initialize_body_state(const icy2d_grid& g, const int blk, double ice_temperature) {
  const int k = cell_index(blk);
  if (k >= g.body_nx * g.body_ny) return;
  g.body_mass[k] = g.cell_mass;
  g.body_energy[k] = g.cell_mass * (g.cp_i * (ice_temperature - g.t_melt));
}
// simulator.py:589-617
__device__ __forceinline__ void k2_initialize_water_state(const icy2d_grid& g, const int blk, double water_temperature_c) {
  const int n = cell_index(blk);
  if (n >= cells(g)) return;
  const int i = n / g.ny, j = n - i * g.ny;
  const float phase = clamp01(g.phi[n]);
  double v = 0.0;
  if (!wall_at(g, i, j) && g.solid[n] == 0 && phase > g.cutoff) v = g.area * (double)phase;
  g.water_v[n] = v;
  g.water_e[n] = (g.rho_w_si * g.cp_w) * v * (water_temperature_c - g.t_melt);
}
__device__ __forceinline__ void k2_reset_thermal_diagnostics(const icy2d_grid& g, const int blk) {
  icy2d_control* ctl = g.control;
  ctl->boundary_power = ctl->boundary_heat_input = ctl->correction_abs = 0.0;
}
// simulator.py:633-714 in control order: volume, energy, base and full
// capacity (sums), specific energy min, max.
__device__ __forceinline__ void k2_aperture_partials(const icy2d_grid& g, const int blk) {
  double v[kRun][6];
#pragma unroll
  for (int r = 0; r < kRun; ++r) {
    const int first = (blk * kRun + r) * kBlock, n = first + (int)threadIdx.x;
    v[r][0] = v[r][1] = v[r][2] = v[r][3] = 0.0;
    v[r][4] = 1.0e30;
    v[r][5] = -1.0e30;
    if (n >= cells(g)) continue;
    int i, j;
    row_col(g, first, n, i, j);
    const double vol = g.water_v[n];
    const double energy = g.water_e[n];
    v[r][0] = vol;
    v[r][1] = energy;
    if (vol > 1.0e-30) v[r][4] = v[r][5] = energy / vol;
    const float phase = clamp01(g.phi[n]);
    if (!wall_at(g, i, j) && g.solid[n] == 0 && phase > g.cutoff) {
      v[r][2] = g.area * (double)phase;
      v[r][3] = g.area;
    }
  }
  run_partials<6, 0x10u, 0x20u>(g, v, blk);
}
// simulator.py:522-540: the thermal volume must stay within [0, capacity].
__device__ __forceinline__ void k2_check_aperture(const icy2d_grid& g, const int blk) {
  icy2d_control* ctl = g.control;
  const double total = ctl->aperture[0], full = ctl->aperture[3];
  const double tol = 1.0e-12 * fmax(g.area, fmax(fabs(total), fabs(full)));
  int flags = 0;
  if (total < -tol) flags |= 1;
  if (total > full + tol) flags |= 2;
  if (flags && !ctl->error_flags) {
    ctl->error_values[0] = total;
    ctl->error_values[1] = full;
  }
  ctl->error_flags |= flags;
}
__device__ __forceinline__ void aperture_scales(const icy2d_control* ctl, double& base_scale, double& spare_scale) {
  const double total = fmax(0.0, ctl->aperture[0]), base = ctl->aperture[2], full = ctl->aperture[3];
  base_scale = spare_scale = 0.0;
  if (total <= base && base > 1.0e-30) {
    base_scale = total / base;
  } else if (total > base) {
    base_scale = 1.0;
    if (full > base + 1.0e-30) spare_scale = fmin(1.0, (total - base) / (full - base));
  }
}
// simulator.py:1629-1658
__device__ __forceinline__ double aperture_target(const icy2d_grid& g, int i, int j, double bs, double ss) {
  const int n = at(g, i, j);
  const float phase = clamp01(g.phi[n]);
  double target = 0.0;
  if (!wall_at(g, i, j) && g.solid[n] == 0 && phase > g.cutoff) {
    const double p = phase;
    target = g.area * (bs * p + ss * (1.0 - p));
  }
  return fmin(g.area, fmax(0.0, target));
}
// simulator.py:716-827 (control aperture = {volume, energy, base, full, min, max})
__device__ __forceinline__ void k2_build_aperture_targets(const icy2d_grid& g, const int blk) {
  const icy2d_control* ctl = g.control;
  double v[kRun][3] = {}, bs, ss;
  aperture_scales(ctl, bs, ss);
  const double low = ctl->aperture[4], high = ctl->aperture[5], total = fmax(0.0, ctl->aperture[0]);
#pragma unroll
  for (int run = 0; run < kRun; ++run) {
    const int first = (blk * kRun + run) * kBlock, n = first + (int)threadIdx.x;
    if (n >= cells(g)) continue;
    int i, j;
    row_col(g, first, n, i, j);
    const double target = aperture_target(g, i, j, bs, ss), vol = g.water_v[n];
    double energy = 0.0;
    if (target > 0.0) {
      double sp = 0.0;
      if (vol > 1.0e-30) {
        sp = g.water_e[n] / vol;
      } else {
        double weight = 0.0;
        for (int r = 1; r <= 3 && weight <= 1.0e-30; ++r)
          for (int di = -r; di <= r; ++di)
            for (int dj = -r; dj <= r; ++dj) {
              const int ni = i + di, nj = j + dj;
              if ((abs(di) > abs(dj) ? abs(di) : abs(dj)) != r || !inside(g, ni, nj) || wall_at(g, ni, nj)) continue;
              const int m = at(g, ni, nj);
              const double nv = g.water_v[m];
              if (nv > 1.0e-30) {
                const double d2 = (double)(di * di + dj * dj);
                sp += g.water_e[m] / d2;
                weight += nv / d2;
              }
            }
        if (weight > 1.0e-30) sp /= weight;
        else if (total > 1.0e-30) sp = ctl->aperture[1] / total;
      }
      sp = fmin(high, fmax(low, sp));
      energy = target * sp;
      v[run][1] = target * (sp - low);
      v[run][2] = target * (high - sp);
    }
    g.target_e[n] = energy;
    v[run][0] = energy;
  }
  run_partials<3>(g, v, blk);
}
// simulator.py:829-859
// with the new water in v (left alone past the grid) for the totals of its block.
__device__ __forceinline__ void aperture_transfer_cell(const icy2d_grid& g, int first, int n, double bs, double ss,
                                                       double (&v)[2]) {
  if (n >= cells(g)) return;
  const icy2d_control* ctl = g.control;
  int i, j;
  row_col(g, first, n, i, j);
  const double correction = ctl->aperture[1] - ctl->targets[0];
  const double low = ctl->aperture[4], high = ctl->aperture[5], cool = ctl->targets[1], heat = ctl->targets[2];
  const double target = aperture_target(g, i, j, bs, ss);
  double energy = g.target_e[n];
  if (target > 0.0) {
    if (correction < 0.0 && cool > 1.0e-30) energy += fmax(-1.0, correction / cool) * fmax(0.0, energy - low * target);
    else if (correction > 0.0 && heat > 1.0e-30) energy += fmin(1.0, correction / heat) * fmax(0.0, high * target - energy);
  }
  g.water_v[n] = target;
  g.water_e[n] = energy;
  v[0] = target;
  v[1] = energy;
}
__device__ __forceinline__ void k2_apply_aperture_transfer(const icy2d_grid& g, const int blk) {
  double v[2] = {0.0, 0.0}, bs, ss;
  aperture_scales(g.control, bs, ss);
  aperture_transfer_cell(g, blk * (int)blockDim.x, cell_index(blk), bs, ss, v);
}
// The transfer and the block sums of what it wrote (k2_water_totals_partials),
// without reading the water planes again: 13 us at 1024x2048 instead of 12 + 11.
__device__ __forceinline__ void k2_transfer_partials(const icy2d_grid& g, const int blk) {
  double v[kRun][2] = {}, bs, ss;
  aperture_scales(g.control, bs, ss);
#pragma unroll
  for (int r = 0; r < kRun; ++r) {
    const int first = (blk * kRun + r) * kBlock;
    aperture_transfer_cell(g, first, first + (int)threadIdx.x, bs, ss, v[r]);
  }
  run_partials<2>(g, v, blk);
}
__device__ __forceinline__ void k2_add_correction_abs(const icy2d_grid& g, const int blk) {
  icy2d_control* ctl = g.control;
  ctl->correction_abs += fabs(ctl->aperture[1] - ctl->targets[0]);
}
// simulator.py:861-877
__device__ __forceinline__ void k2_water_totals_partials(const icy2d_grid& g, const int blk) {
  double v[kRun][2] = {};
#pragma unroll
  for (int r = 0; r < kRun; ++r) {
    const int n = (blk * kRun + r) * kBlock + (int)threadIdx.x;
    if (n >= cells(g)) continue;
    v[r][0] = g.water_v[n];
    v[r][1] = g.water_e[n];
  }
  run_partials<2>(g, v, blk);
}
// simulator.py:879-907
__device__ __forceinline__ void k2_body_conduction(const icy2d_grid& g, const int blk, double dt) {
  const int k = cell_index(blk);
  if (k == 0) g.control->unassigned[0] = g.control->unassigned[1] = 0.0;
  if (k >= g.body_nx * g.body_ny) return;
  const int bi = k / g.body_ny, bj = k - bi * g.body_ny;
  g.melt_target[k] = -1;
  const float fr = body_fraction(g, bi, bj);
  const double t = body_temperature(g, k);
  double rate = 0.0;
  const int off[4][2] = {{1, 0}, {-1, 0}, {0, 1}, {0, -1}};
#pragma unroll
  for (int o = 0; o < 4; ++o) {
    const int ni = bi + off[o][0], nj = bj + off[o][1];
    if (ni >= 0 && ni < g.body_nx && nj >= 0 && nj < g.body_ny) {
      const double face = (double)fminf(fr, body_fraction(g, ni, nj));
      rate += g.k_i * face * (t - body_temperature(g, ni * g.body_ny + nj));
    }
  }
  g.body_heat[k] = heat_to_fixed(g, -dt * rate);
}
__device__ __forceinline__ double cell_aperture(const icy2d_grid& g, int n) { return fmin(1.0, fmax(0.0, g.water_v[n] / g.area)); }
// simulator.py:909-1010 (axis 0) and :1063-1164 (axis 1); boundary power as partials
__device__ __forceinline__ void k2_conduction_flux(const icy2d_grid& g, const int blk, int axis) {
  const int t = cell_index(blk);
  const int fx = axis == 0 ? g.nx + 1 : g.nx, fy = axis == 0 ? g.ny : g.ny + 1, limit = axis == 0 ? g.nx : g.ny;
  double inward[1] = {0.0};
  if (t < fx * fy) {
    const int a = t / fy, b = t - a * fy, face = axis == 0 ? a : b;
    const int lo_kind = axis == 0 ? g.left_kind : g.bottom_kind, hi_kind = axis == 0 ? g.right_kind : g.top_kind;
    const double lo_value = axis == 0 ? g.left_value : g.bottom_value, hi_value = axis == 0 ? g.right_value : g.top_value;
    double out = 0.0;
    if (face > 0 && face < limit) {
      const int li = axis == 0 ? a - 1 : a, lj = axis == 0 ? b : b - 1;
      const int l = at(g, li, lj), r = at(g, a, b);
      const bool la = water_cell(g, li, lj), ra = water_cell(g, a, b);
      if (la && ra) {
        if (g.water_v[l] > 1.0e-30 && g.water_v[r] > 1.0e-30)
          out = -g.k_w * fmin(cell_aperture(g, l), cell_aperture(g, r)) * (water_temperature(g, r) - water_temperature(g, l));
      } else if (wall_at(g, li, lj) && ra && g.water_v[r] > 1.0e-30) {
        if (lo_kind == 1) out = 2.0 * g.k_w * cell_aperture(g, r) * (lo_value - water_temperature(g, r));
        inward[0] = out;
      } else if (la && g.water_v[l] > 1.0e-30 && wall_at(g, a, b)) {
        if (hi_kind == 1) out = 2.0 * g.k_w * cell_aperture(g, l) * (water_temperature(g, l) - hi_value);
        inward[0] = -out;
      }
    }
    (axis == 0 ? g.flux_ex : g.flux_ey)[t] = out;
  }
  block_partials<1>(inward, g.partials, blk);
}
// simulator.py:1012-1061 (axis 0) and :1166-1215 (axis 1)
__device__ __forceinline__ void k2_advection_flux(const icy2d_grid& g, const int blk, int axis) {
  const int t = cell_index(blk), N = cells(g);
  const int fx = axis == 0 ? g.nx + 1 : g.nx, fy = axis == 0 ? g.ny : g.ny + 1, limit = axis == 0 ? g.nx : g.ny;
  if (t >= fx * fy) return;
  const int a = t / fy, b = t - a * fy, face = axis == 0 ? a : b;
  double e = 0.0, v = 0.0;
  if (g.advection && face > 0 && face < limit) {
    const int li = axis == 0 ? a - 1 : a, lj = axis == 0 ? b : b - 1;
    if (water_cell(g, li, lj) && water_cell(g, a, b)) {
      const int l = at(g, li, lj), r = at(g, a, b);
      const float ul = g.u[axis * N + l] + 0.5f * g.a[axis * N + l];
      const float ur = g.u[axis * N + r] + 0.5f * g.a[axis * N + r];
      const double speed = 0.5 * (double)(ul + ur) * g.velocity_scale;
      const int up = speed >= 0.0 ? l : r;
      const double uv = g.water_v[up], frac = fmin(1.0, fmax(0.0, uv / g.area));
      v = speed * frac * (double)g.dx;
      e = v * (g.water_e[up] / fmax(uv, 1.0e-30));
    }
  }
  (axis == 0 ? g.flux_ex : g.flux_ey)[t] = e;
  (axis == 0 ? g.flux_vx : g.flux_vy)[t] = v;
}
// simulator.py:1217-1246
__device__ __forceinline__ void k2_update_water(const icy2d_grid& g, const int blk, double dt, int volume) {
  const int n = cell_index(blk);
  if (n >= cells(g)) return;
  const int i = n / g.ny, j = n - i * g.ny, ny = g.ny;
  if (wall_at(g, i, j)) return;
  const double de = g.flux_ex[(i + 1) * ny + j] - g.flux_ex[i * ny + j] + g.flux_ey[i * (ny + 1) + j + 1] -
                    g.flux_ey[i * (ny + 1) + j];
  g.water_e[n] -= dt * de;
  if (volume) {
    const double dv = g.flux_vx[(i + 1) * ny + j] - g.flux_vx[i * ny + j] + g.flux_vy[i * (ny + 1) + j + 1] -
                      g.flux_vy[i * (ny + 1) + j];
    g.water_v[n] -= dt * dv;
  }
}
// simulator.py:624-627
__device__ __forceinline__ void k2_reset_interval_sources(const icy2d_grid& g, const int blk) { g.control->interval[0] = g.control->interval[1] = 0.0; }
__device__ __forceinline__ void k2_accumulate_boundary_heat(const icy2d_grid& g, const int blk, double dt) {
  g.control->boundary_heat_input += dt * g.control->boundary_power;
}
// simulator.py:1252-1372
__device__ __forceinline__ void k2_exchange_heat(const icy2d_grid& g, const int blk, double dt) {
  const int n = cell_index(blk);
  if (n >= cells(g)) return;
  const int i = n / g.ny, j = n - i * g.ny;
  if (!(water_cell(g, i, j) && g.water_v[n] > 1.0e-30)) return;
  const double k = 2.0 * g.k_w * g.k_i / (g.k_w + g.k_i);
  bool touches = false;
  for (int di = -1; di <= 1; ++di)
    for (int dj = -1; dj <= 1; ++dj)
      if ((di == 0 || dj == 0) && inside(g, i + di, j + dj)) touches = touches || g.coverage[at(g, i + di, j + dj)] > 0.0f;
  if (!touches) return;  // nothing requested: the energy stays as it is
  const Pose pose = load_pose(g);
  double req[20];
  int tgt[20];
#pragma unroll
  for (int s = 0; s < 20; ++s) {
    req[s] = 0.0;
    tgt[s] = 0;
  }
  double requested = 0.0;
  const double ap = fmin(1.0, g.water_v[n] / g.area), tw = water_temperature(g, n);
  const int off[5][2] = {{0, 0}, {1, 0}, {-1, 0}, {0, 1}, {0, -1}};
#pragma unroll
  for (int f = 0; f < 5; ++f) {
    const int wi = i + off[f][0], wj = j + off[f][1];
    if (!inside(g, wi, wj)) continue;
    const double coverage = g.coverage[at(g, wi, wj)];
    if (!(coverage > 0.0)) continue;
    const double contact = fmin(ap, fmin(1.0, coverage / (double)g.threshold));
    // simulator.py:1615-1627, stored as FP32 grid coordinates
    const double rx = (wi + 0.5) - pose.ox, ry = (wj + 0.5) - pose.oy;
    const float gx = (float)(pose.c * rx + pose.s * ry + 0.5 * g.body_nx - 0.5);
    const float gy = (float)(-pose.s * rx + pose.c * ry + 0.5 * g.body_ny - 0.5);
    const int bi0 = (int)floorf(gx), bj0 = (int)floorf(gy);
    const double fx = (double)(gx - (float)bi0), fy = (double)(gy - (float)bj0);
#pragma unroll
    for (int oi = 0; oi < 2; ++oi)
#pragma unroll
      for (int oj = 0; oj < 2; ++oj) {
        const int bi = bi0 + oi, bj = bj0 + oj;
        if (!(bi >= 0 && bi < g.body_nx && bj >= 0 && bj < g.body_ny)) continue;
        const int kb = bi * g.body_ny + bj;
        if (!(g.body_mass[kb] > 0.0)) continue;
        const double wx = oi ? fx : 1.0 - fx, wy = oj ? fy : 1.0 - fy;
        const double share = wx * wy * (double)body_fraction(g, bi, bj) / coverage;
        const double heat = dt * k * contact * share * fmax(0.0, tw - body_temperature(g, kb));
        const int slot = f * 4 + oi * 2 + oj;
        req[slot] = heat;
        tgt[slot] = kb;
        requested += heat;
      }
  }
  double scale = 0.0;
  if (requested > 0.0) scale = fmin(1.0, fmax(0.0, g.water_e[n]) / requested);
  double transferred = 0.0;
#pragma unroll
  for (int s = 0; s < 20; ++s) {
    const double heat = scale * req[s];
    if (heat > 0.0) {
      add_fixed(g.body_heat + tgt[s], heat_to_fixed(g, heat));
      atomicMax(&g.melt_target[tgt[s]], n);
      transferred += heat;
    }
  }
  g.water_e[n] -= transferred;
}
// simulator.py:1374-1406 (interval melt as partials)
__device__ __forceinline__ void k2_phase_change(const icy2d_grid& g, const int blk) {
  const int k = cell_index(blk);
  double v[1] = {0.0};
  if (k < g.body_nx * g.body_ny) {
    const double heat = (double)g.body_heat[k] / heat_fixed_scale(g);
    double solid = g.body_mass[k], sensible = g.body_energy[k], melt = 0.0, melt_sensible = 0.0;
    if (heat <= 0.0) {
      if (solid > 0.0) sensible += heat;
    } else {
      const double gain = fmin(heat, fmax(-sensible, 0.0));
      sensible += gain;
      const double remaining = heat - gain;
      melt = fmin(solid, remaining / g.latent);
      solid -= melt;
      melt_sensible = fmax(0.0, remaining - melt * g.latent);
    }
    if (solid <= 0.0) {
      solid = 0.0;
      sensible = 0.0;
    }
    g.body_mass[k] = solid;
    g.body_energy[k] = sensible;
    g.melt_mass[k] = melt;
    g.melt_sensible[k] = melt_sensible;
    if (melt > 0.0) v[0] = melt;
  }
  block_partials<1>(v, g.partials, blk);
}
// simulator.py:1408-1422
__device__ __forceinline__ void k2_freeze_eligibility(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk);
  if (n >= cells(g)) return;
  const int i = n / g.ny, j = n - i * g.ny;
  g.eligible[n] = (int8_t)(water_cell(g, i, j) && g.water_v[n] > 1.0e-30);
}
// simulator.py:1424-1475 (assigned melt mass and the unassigned pool as partials)
__device__ __forceinline__ void k2_inject_melt(const icy2d_grid& g, const int blk) {
  const int k = cell_index(blk);
  double v[3] = {0.0, 0.0, 0.0};
  if (k < g.body_nx * g.body_ny && g.melt_mass[k] > 0.0) {
    const icy2d_control* ctl = g.control;
    const float c = cosf(ctl->angle), s = sinf(ctl->angle);
    const int bi = k / g.body_ny, bj = k - bi * g.body_ny;
    const double melt = g.melt_mass[k];
    const double lx = bi + 0.5 - 0.5 * g.body_nx, ly = bj + 0.5 - 0.5 * g.body_ny;
    const double wx = ctl->origin[0] + (double)c * lx - (double)s * ly;
    const double wy = ctl->origin[1] + (double)s * lx + (double)c * ly;
    const int enc = g.melt_target[k];
    int ti = -1, tj = -1;
    if (enc >= 0) {
      ti = enc / g.ny;
      tj = enc - ti * g.ny;
    } else {
      const int bi0 = (int)floor(wx), bj0 = (int)floor(wy);
      float best = 1.0e30f;
      for (int di = -2; di <= 2; ++di)
        for (int dj = -2; dj <= 2; ++dj) {
          const int xi = bi0 + di, xj = bj0 + dj;
          if (inside(g, xi, xj) && g.eligible[at(g, xi, xj)]) {
            const float d = (float)(di * di + dj * dj);
            if (d < best) {
              best = d;
              ti = xi;
              tj = xj;
            }
          }
        }
    }
    const double volume = melt / g.rho_w_si, energy = g.melt_sensible[k];
    if (ti >= 0 && tj >= 0) {
      const int t = at(g, ti, tj);
      add_fixed(g.inject_acc + t, to_fixed(g, volume, volume_fixed_scale(g)));
      add_fixed(g.inject_acc + cells(g) + t, to_fixed(g, energy, energy_fixed_scale(g)));
      g.melt_target[k] = t;
      v[0] = melt;
    } else {
      g.melt_target[k] = -1;
      v[1] = melt;
      v[2] = energy;
    }
  }
  block_partials<3>(v, g.partials, blk);
}
// Adds the injection's fixed-point sums to the water cells they feed and
// clears them: of the body cells feeding one water cell, whichever swaps a
// sum out first applies it, so each sum is added once and its value does not
// depend on which cell that is.
__device__ __forceinline__ void k2_fold_injection(const icy2d_grid& g, const int blk) {
  const int k = cell_index(blk);
  if (k >= g.body_nx * g.body_ny || !(g.melt_mass[k] > 0.0)) return;
  const int t = g.melt_target[k];
  if (t < 0) return;
  unsigned long long* acc = reinterpret_cast<unsigned long long*>(g.inject_acc);
  const long long volume = (long long)atomicExch(acc + t, 0ull);
  const long long energy = (long long)atomicExch(acc + cells(g) + t, 0ull);
  if (volume) g.water_v[t] += (double)volume / volume_fixed_scale(g);
  if (energy) g.water_e[t] += (double)energy / energy_fixed_scale(g);
}
__device__ __forceinline__ void k2_store_injection(const icy2d_grid& g, const int blk) {
  const double* t = g.partials + g.partials_capacity - 3;
  icy2d_control* ctl = g.control;
  ctl->interval[1] += t[0];
  ctl->unassigned[0] += t[1];
  ctl->unassigned[1] += t[2];
}
// simulator.py:1477-1502
__device__ __forceinline__ void k2_fallback_partials(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk);
  double v[2] = {0.0, 0.0};
  if (n < cells(g)) {
    const int i = n / g.ny, j = n - i * g.ny;
    if (water_cell(g, i, j) && g.water_v[n] > 1.0e-30) {
      v[0] = fmax(g.area - g.water_v[n], 0.0);
      v[1] = g.water_v[n];
    }
  }
  block_partials<2>(v, g.partials, blk);
}
// simulator.py:1504-1540
__device__ __forceinline__ void k2_apply_fallback(const icy2d_grid& g, const int blk, int use_free) {
  const int n = cell_index(blk);
  if (n >= cells(g)) return;
  const icy2d_control* ctl = g.control;
  const double den = use_free ? ctl->fallback[0] : ctl->fallback[1];
  const double mass = ctl->unassigned[0], volume = mass / g.rho_w_si, energy = ctl->unassigned[1];
  const int i = n / g.ny, j = n - i * g.ny;
  double w = 0.0;
  if (water_cell(g, i, j) && g.water_v[n] > 1.0e-30) w = use_free ? fmax(g.area - g.water_v[n], 0.0) : g.water_v[n];
  if (w > 0.0 && den > 1.0e-30) {
    const double fr = w / den;
    g.water_v[n] += fr * volume;
    g.water_e[n] += fr * energy;
  }
}
__device__ __forceinline__ void k2_count_fallback(const icy2d_grid& g, const int blk, int use_free) {
  icy2d_control* ctl = g.control;
  const double den = use_free ? ctl->fallback[0] : ctl->fallback[1];
  if (den > 1.0e-30 && ctl->unassigned[0] > 0.0) ctl->interval[1] += ctl->unassigned[0];
}
// simulator.py:1565-1583
__device__ __forceinline__ void k2_totals_partials(const icy2d_grid& g, const int blk) {
  const int n = cell_index(blk);
  double v[4] = {0.0, 0.0, 0.0, 0.0};
  if (n < g.body_nx * g.body_ny) {
    v[0] = g.body_mass[n];
    v[2] = g.body_energy[n];
  }
  if (n < cells(g)) {
    v[1] = g.rho_w_si * g.water_v[n];
    v[3] = g.water_e[n];
  }
  block_partials<4>(v, g.partials, blk);
}

// ---------------------------------------------------------------- host
// Index spaces a kernel covers per case, and the launch wrappers.  Every
// kernel body above takes (grid, block index within its case); one_case
// runs it for one grid passed by value, many_cases for the case that owns
// the block in a batch's prefix table.
enum Shape : int {
  kCells = 0, kBody, kFaceX, kFaceY, kOne, kTotals, kCells128, kCells512, kBandTiles,
  kTiles128, kTiles256, kTiles512, kRuns, kShapes
};
static_assert(kShapes == ICY2D_SHAPES, "shape count");

long shape_count(const icy2d_grid& g, int shape) {
  const long cells = (long)g.nx * g.ny, body = (long)g.body_nx * g.body_ny;
  switch (shape) {
    case kBody: return body;
    case kFaceX: return (long)(g.nx + 1) * g.ny;
    case kFaceY: return (long)g.nx * (g.ny + 1);
    case kOne: return 1;
    case kTotals: return cells > body ? cells : body;
    case kRuns: return (cells + kRun - 1) / kRun;
    case kBandTiles:  // one block of kBlock threads per 16 x 64 band tile
      return (long)((g.nx + kBandI - 1) / kBandI) * ((g.ny + kBandJ - 1) / kBandJ) * kBlock;
    case kTiles128:  // one block per (threads / 64) x 64 collision tile
    case kTiles256:
    case kTiles512: {
      const int threads = shape == kTiles128 ? 128 : shape == kTiles512 ? 512 : 256, rows = threads / kTileCols;
      return (long)((g.nx + rows - 1) / rows) * ((g.ny + kTileCols - 1) / kTileCols) * threads;
    }
    default: return cells;
  }
}
int shape_threads(int shape) {
  if (shape == kOne) return 1;
  if (shape == kCells128 || shape == kTiles128) return 128;
  if (shape == kCells512 || shape == kTiles512) return 512;
  return kBlock;
}
unsigned shape_blocks(const icy2d_grid& g, int shape) {
  const long t = shape_threads(shape);
  return (unsigned)((shape_count(g, shape) + t - 1) / t);
}
int cells_shape(int threads) { return threads == 128 ? kCells128 : threads == 512 ? kCells512 : kCells; }
int tiles_shape(int threads) { return threads == 128 ? kTiles128 : threads == 512 ? kTiles512 : kTiles256; }

struct PerCase {
  const double* v;
};
__device__ __forceinline__ double resolve(PerCase a, int c) { return a.v[c]; }
template <class T>
__device__ __forceinline__ T resolve(T a, int) {
  return a;
}

// Storage >= 0: every case stores its populations that way, so a kernel body
// has no branch around each of a cell's 18 loads and stores (an FP16 load that
// is converted in its own branch is waited for there, one after the other).
// Compiled for FP32 and the two stochastic FP16 forms; any other runs with
// the branches.
constexpr int kAnyStorage = -1, kHalfMomentum = 5, kHalfRelative = 15;
// Waves a SIMD that a kernel's registers have to leave room for: the collision
// takes 126 to 129 by itself, and four waves fit up to 128 (over the 64-case
// ensemble with FP16 deviations 862 us at three waves, 748 at four).
template <auto F>
constexpr int kWaves = 1;
template <>
constexpr int kWaves<k2_collide_push> = 4;
template <int T, auto F, int Storage = kAnyStorage, class... A>
__global__ void __launch_bounds__(T, kWaves<F>) one_case(icy2d_grid g, A... a) {
  if (Storage != kAnyStorage) g.half_populations = Storage;
  F(g, (int)blockIdx.x, a...);
}
// Largest c with first[c] <= x (first is non-decreasing, first[0] = 0).
__device__ __forceinline__ int owner(const int32_t* first, int ncases, int x) {
  int lo = 0, hi = ncases;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (first[mid] <= x) lo = mid;
    else hi = mid;
  }
  return lo;
}
// A case's grid, its pointers known to the compiler as global memory: read
// from memory they could be LDS too, and each access would be a flat one, which
// counts as an LDS access as well and is waited for as such.
template <class T>
__device__ __forceinline__ void as_global(T*& p) {
  p = (T*)(__attribute__((address_space(1))) T*)(uintptr_t)p;
}
__device__ __forceinline__ icy2d_grid case_grid(const icy2d_batch& b, int c) {
  icy2d_grid g = b.grids[c];
  as_global(g.f), as_global(g.fbuf), as_global(g.h), as_global(g.hbuf);
  as_global(g.phi), as_global(g.u), as_global(g.a), as_global(g.p), as_global(g.moving);
  as_global(g.p_ref), as_global(g.rho_ref);
  as_global(g.solid), as_global(g.prev_solid), as_global(g.eligible);
  as_global(g.coverage), as_global(g.phase_ref);
  as_global(g.body_mass), as_global(g.body_energy), as_global(g.body_heat);
  as_global(g.melt_mass), as_global(g.melt_sensible), as_global(g.melt_target);
  as_global(g.water_v), as_global(g.water_e), as_global(g.target_e);
  as_global(g.flux_ex), as_global(g.flux_vx), as_global(g.flux_ey), as_global(g.flux_vy);
  as_global(g.inject_acc), as_global(g.partials), as_global(g.control);
  return g;
}
template <int T, auto F, int Storage = kAnyStorage, class... A>
__global__ void __launch_bounds__(T, kWaves<F>) many_cases(icy2d_batch b, int shape, A... a) {
  const int32_t* first = b.first_block + shape * (b.ncases + 1);
  const int c = owner(first, b.ncases, (int)blockIdx.x);
  if (b.active && !b.active[c]) return;
  icy2d_grid g = case_grid(b, c);
  if (Storage != kAnyStorage) {
    // The batch's word is not taken for it: at the wrong width the accesses
    // would leave the case's buffers.  check_storage reports it, as a store
    // here would keep the grid's fields from being loaded as scalars (143
    // registers for 128, and 848 us for 702 over the 64-case ensemble).
    if (g.half_populations != Storage) return;
    g.half_populations = Storage;
  }
  F(g, (int)blockIdx.x - first[c], resolve(a, c)...);
}
// Of a batch that states a storage, the cases that have another.
__device__ __forceinline__ void check_storage(const icy2d_batch& b, const icy2d_grid& g) {
  if (b.storage != 0 && b.storage != 1 + g.half_populations && threadIdx.x == 0) atomicOr(&g.control->error_flags, 8);
}
// Destination of a finished reduction: a byte offset into the control block,
// or the last `tail` slots of the case's partials.
struct Dest {
  long control_offset;
  int tail;
};
__host__ __device__ inline double* dest_ptr(const icy2d_grid& g, Dest d) {
  return d.tail ? g.partials + g.partials_capacity - d.tail : (double*)((char*)g.control + d.control_offset);
}
#define CTL(field, k) (Dest{(long)offsetof(icy2d_control, field) + 8 * (k), 0})
#define TAIL(k) (Dest{0, (k)})

__global__ void __launch_bounds__(kFinishThreads) k2_finish_many(icy2d_batch b, int shape, int K, Dest d,
                                                                 unsigned min_mask, unsigned max_mask,
                                                                 unsigned add_mask) {
  const int c = (int)blockIdx.x / K, k = (int)blockIdx.x - c * K;
  if (b.active && !b.active[c]) return;
  const icy2d_grid g = case_grid(b, c);
  check_storage(b, g);
  const int32_t* first = b.first_block + shape * (b.ncases + 1);
  finish_fold(g.partials, first[c + 1] - first[c], K, k, dest_ptr(g, d), min_mask, max_mask, add_mask);
}

// A fold followed by a one-thread step that reads its results, in one
// launch: each of the K blocks folds its column, and the last block to get
// there (a device-scope ticket in the control block, which that block puts
// back to 0) runs Tail(g, 0, a...).  Saves the launch of the one-thread
// kernel that would otherwise follow the fold.
__device__ __forceinline__ bool last_finisher(icy2d_control* ctl, int K) {
  __shared__ bool last;
  if (threadIdx.x == 0) {
    __threadfence();
    last = atomicAdd(&ctl->finish_ticket, 1) == K - 1;
    if (last) {
      __threadfence();
      ctl->finish_ticket = 0;
    }
  }
  __syncthreads();
  return last;
}
template <auto Tail, class... A>
__global__ void __launch_bounds__(kFinishThreads) k2_finish_tail(icy2d_grid g, int blocks, int K, Dest d,
                                                                 unsigned min_mask, unsigned max_mask,
                                                                 unsigned add_mask, A... a) {
  finish_fold(g.partials, blocks, K, (int)blockIdx.x, dest_ptr(g, d), min_mask, max_mask, add_mask);
  if (last_finisher(g.control, K) && threadIdx.x == 0) Tail(g, 0, a...);
}
template <auto Tail, class... A>
__global__ void __launch_bounds__(kFinishThreads) k2_finish_many_tail(icy2d_batch b, int shape, int K, Dest d,
                                                                      unsigned min_mask, unsigned max_mask,
                                                                      unsigned add_mask, A... a) {
  const int c = (int)blockIdx.x / K, k = (int)blockIdx.x - c * K;
  if (b.active && !b.active[c]) return;
  const icy2d_grid g = case_grid(b, c);
  check_storage(b, g);
  const int32_t* first = b.first_block + shape * (b.ncases + 1);
  finish_fold(g.partials, first[c + 1] - first[c], K, k, dest_ptr(g, d), min_mask, max_mask, add_mask);
  if (last_finisher(g.control, K) && threadIdx.x == 0) Tail(g, 0, resolve(a, c)...);
}

int launch_status() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? 0 : (int)e;
}

// One case (the single-case C ABI).
struct One {
  const icy2d_grid& g;
  hipStream_t s;
  using Real = double;
  bool fits(int shape, int K) const { return (long)shape_blocks(g, shape) * K + 8 <= (long)g.partials_capacity; }
  int tuned_shape(int which) const { return which == 0 ? kTiles256 : kCells; }
  template <auto F, class... A>
  int launch(int shape, A... a) const {
    one_case<kBlock, F><<<shape_blocks(g, shape), shape_threads(shape), 0, s>>>(g, a...);
    return launch_status();
  }
  // A kernel that moves populations, compiled for the grid's storage: for the
  // three that the single run, the ensembles and the smallest footprint take by
  // default (each costs its own code); the others run the general kernel.
  template <auto F, class... A>
  int launch_stored(int shape, A... a) const {
    const unsigned blocks = shape_blocks(g, shape);
    const int threads = shape_threads(shape);
    auto kernel = one_case<kBlock, F, kAnyStorage, A...>;
    if (g.half_populations == 0) kernel = one_case<kBlock, F, 0, A...>;
    if (g.half_populations == kHalfMomentum) kernel = one_case<kBlock, F, kHalfMomentum, A...>;
    if (g.half_populations == kHalfRelative) kernel = one_case<kBlock, F, kHalfRelative, A...>;
    kernel<<<blocks, threads, 0, s>>>(g, a...);
    return launch_status();
  }
  template <auto F, class... A>
  int launch_tuned(int shape, A... a) const {
    return launch_stored<F>(shape, a...);
  }
  int finish(int shape, int K, Dest d, unsigned mn, unsigned mx, unsigned add) const {
    k2_finish<<<K, kFinishThreads, 0, s>>>(g.partials, (int)shape_blocks(g, shape), K, dest_ptr(g, d), mn, mx, add);
    return launch_status();
  }
  template <auto Tail, class... A>
  int finish_tail(int shape, int K, Dest d, unsigned mn, unsigned mx, unsigned add, A... a) const {
    k2_finish_tail<Tail><<<K, kFinishThreads, 0, s>>>(g, (int)shape_blocks(g, shape), K, d, mn, mx, add, a...);
    return launch_status();
  }
};
// Every case of a batch (capacities are checked once by icy2d_batch_plan).
struct Many {
  const icy2d_batch& b;
  hipStream_t s;
  using Real = PerCase;
  bool fits(int, int) const { return true; }
  int tuned_shape(int which) const {
    return which == 0 ? tiles_shape(b.collide_threads) : cells_shape(b.stream_threads);
  }
  template <auto F, class... A>
  int launch(int shape, A... a) const {
    many_cases<kBlock, F><<<b.total_blocks[shape], shape_threads(shape), 0, s>>>(b, shape, a...);
    return launch_status();
  }
  // A kernel that moves populations, compiled for the cases' common storage.
  template <auto F, class... A>
  int launch_stored(int shape, A... a) const {
    auto kernel = many_cases<kBlock, F, kAnyStorage, A...>;
    if (b.storage == 1) kernel = many_cases<kBlock, F, 0, A...>;
    if (b.storage == 1 + kHalfMomentum) kernel = many_cases<kBlock, F, kHalfMomentum, A...>;
    if (b.storage == 1 + kHalfRelative) kernel = many_cases<kBlock, F, kHalfRelative, A...>;
    kernel<<<b.total_blocks[shape], kBlock, 0, s>>>(b, shape, a...);
    return launch_status();
  }
  template <auto F, class... A>
  int launch_tuned(int shape, A... a) const {
    const unsigned blocks = b.total_blocks[shape];
    if (shape_threads(shape) == 128) many_cases<128, F><<<blocks, 128, 0, s>>>(b, shape, a...);
    else if (shape_threads(shape) == 512) many_cases<512, F><<<blocks, 512, 0, s>>>(b, shape, a...);
    else return launch_stored<F>(shape, a...);
    return launch_status();
  }
  int finish(int shape, int K, Dest d, unsigned mn, unsigned mx, unsigned add) const {
    k2_finish_many<<<b.ncases * K, kFinishThreads, 0, s>>>(b, shape, K, d, mn, mx, add);
    return launch_status();
  }
  template <auto Tail, class... A>
  int finish_tail(int shape, int K, Dest d, unsigned mn, unsigned mx, unsigned add, A... a) const {
    k2_finish_many_tail<Tail><<<b.ncases * K, kFinishThreads, 0, s>>>(b, shape, K, d, mn, mx, add, a...);
    return launch_status();
  }
};

#define TRY(expr)                \
  do {                           \
    if (int rc_ = (expr)) return rc_; \
  } while (0)
#define NEED(d, shape, K)                              \
  do {                                                 \
    if (!(d).fits((shape), (K))) return ICY2D_ERR_ARGUMENT; \
  } while (0)

// ------------------------------------------------------------ operations
template <class D> int op_body_fraction(const D& d, int only_if_projected) {
  return d.template launch<k2_body_fraction>(kCells, only_if_projected);
}
template <class D> int op_commit_raster(const D& d) { return d.template launch<k2_commit_raster>(kCells); }
template <class D> int op_contact_support(const D& d, int reduce, int only_if_projected) {
  NEED(d, kCells, 4);
  if (reduce) {
    TRY(d.template launch<k2_support_partials>(kRuns, only_if_projected));
    // min x, max x, min y, max y into the last four partials slots
    return d.template finish_tail<k2_support_store>(kRuns, 4, TAIL(4), 0x5u, 0xAu, 0u, reduce, only_if_projected);
  }
  return d.template launch<k2_support_store>(kOne, reduce, only_if_projected);
}
template <class D> int op_integrate_rigid(const D& d) { return d.template launch<k2_integrate_rigid>(kOne); }
template <class D> int op_project_inside(const D& d) { return d.template launch<k2_project_inside>(kOne); }
template <class D> int op_update_solid_mask(const D& d, int init) {
  return d.template launch<k2_update_solid_mask>(kCells, init);
}
template <class D> int op_reduce_mass_properties(const D& d) {
  NEED(d, kBody, 4);
  TRY(d.template launch<k2_mass_partials>(kBody));
  return d.finish(kBody, 4, CTL(reduced, 0), 0u, 0u, 0u);
}
template <class D> int op_apply_mass_properties(const D& d, int initialize) {
  return d.template launch<k2_apply_mass_properties>(kOne, initialize);
}
template <class D> int op_collide(const D& d, int with_momentum) {
  const int shape = d.tuned_shape(0);
  NEED(d, shape, 3);
  TRY(d.template launch_tuned<k2_collide>(shape, with_momentum));
  if (!with_momentum) return 0;
  return d.finish(shape, 3, CTL(impulse, 0), 0u, 0u, 0x7u);
}
template <class D> int op_collide_stream(const D& d) {
  const int shape = d.tuned_shape(0);
  NEED(d, shape, 3);
  TRY(d.template launch_tuned<k2_collide_push>(shape));
  return d.finish(shape, 3, CTL(impulse, 0), 0u, 0u, 0x7u);
}
template <class D> int op_prepare_cut_links(const D& d) {
  NEED(d, kCells, 3);
  TRY(d.template launch<k2_prepare_cut_links>(kCells));
  return d.finish(kCells, 3, CTL(impulse, 0), 0u, 0u, 0x7u);
}
template <class D> int op_stream(const D& d, int phase_only, int mode) {
  if (mode < 1 || mode > 3) return ICY2D_ERR_ARGUMENT;
  const int shape = d.tuned_shape(1);
  if (mode == kStreamPull) return d.template launch_tuned<k2_stream<kStreamPull>>(shape, phase_only);
  if (mode == kStreamUpdate) return d.template launch_tuned<k2_stream<kStreamUpdate>>(shape, phase_only);
  return d.template launch_tuned<k2_stream<kStreamPull | kStreamUpdate>>(shape, phase_only);
}
template <class D> int op_update_pressure(const D& d) { return d.template launch<k2_update_pressure>(kCells); }
template <class D> int op_refill(const D& d) { return d.template launch<k2_refill>(kCells); }
template <class D> int op_measure_outflow(const D& d) {
  NEED(d, kCells, 1);
  TRY(d.template launch<k2_outflow_partials>(kCells));
  return d.template finish_tail<k2_store_outflow>(kCells, 1, TAIL(1), 0u, 0x1u, 0u);
}
template <class D> int op_clip_phase(const D& d, double max_bulk_l1) {
  NEED(d, kCells, 1);
  TRY(d.template launch_stored<k2_clip_phase>(kCells, max_bulk_l1));
  return d.finish(kCells, 1, CTL(water, 1), 0u, 0u, 0u);
}
template <class D> int op_seed_projection(const D& d) { return d.template launch<k2_seed_projection>(kCells); }
template <class D> int op_dilate_projection(const D& d, int primary_to_next) {
  return d.template launch<k2_dilate_projection>(kCells, primary_to_next);
}
template <class D> int op_dilate_band(const D& d, int radius) {
  if (radius < 0 || radius > kMaxBand || radius % 2) return ICY2D_ERR_ARGUMENT;
  if (radius == 0) return 0;
  TRY(d.template launch<k2_dilate_band>(kBandTiles, radius));
  return d.template launch<k2_copy_band>(kCells);
}
template <class D> int op_evaluate_projection(const D& d, typename D::Real lambda) {
  NEED(d, kCells, 2);
  TRY(d.template launch<k2_evaluate_projection>(kRuns, lambda));
  return d.finish(kCells, 2, CTL(water, 1), 0u, 0u, 0u);
}
template <class D> int op_apply_projection(const D& d, typename D::Real lambda) {
  NEED(d, kCells, 1);
  TRY(d.template launch_stored<k2_apply_projection>(kCells, lambda));
  return d.finish(kCells, 1, CTL(water, 1), 0u, 0u, 0u);
}
template <class D> int op_projection_residual_weight(const D& d, typename D::Real residual) {
  NEED(d, kCells, 1);
  TRY(d.template launch<k2_residual_weight>(kCells, residual));
  return d.finish(kCells, 1, CTL(water, 2), 0u, 0u, 0u);
}
template <class D>
int op_apply_projection_residual(const D& d, typename D::Real residual, typename D::Real weight) {
  NEED(d, kCells, 1);
  TRY(d.template launch<k2_apply_residual>(kCells, residual, weight));
  return d.finish(kCells, 1, CTL(water, 1), 0u, 0u, 0u);
}
template <class D> int fluid_momentum(const D& d, Dest out) {
  NEED(d, kCells, 3);
  TRY(d.template launch<k2_momentum_partials>(kCells));
  return d.finish(kCells, 3, out, 0u, 0u, 0u);
}
template <class D> int op_snapshot_melt_momentum(const D& d) {
  TRY(d.template launch<k2_snapshot_body>(kOne));
  return fluid_momentum(d, CTL(before, 0));
}
template <class D> int op_reduce_provisional_momentum(const D& d) {
  TRY(fluid_momentum(d, CTL(provisional, 0)));
  NEED(d, kCells, 3);
  TRY(d.template launch<k2_wet_partials>(kCells));
  return d.template finish_tail<k2_store_wet>(kCells, 3, TAIL(3), 0x2u, 0x4u, 0u);
}
template <class D> int op_melt_weight_geometry(const D& d) {
  NEED(d, kCells, 3);
  TRY(d.template launch<k2_weight_partials>(kCells));
  return d.template finish_tail<k2_melt_status>(kCells, 3, CTL(wet, 1), 0u, 0u, 0u);
}
template <class D> int op_apply_melt_correction(const D& d) {
  return d.template launch_stored<k2_apply_melt_correction>(kCells);
}
template <class D> int op_reduce_final_momentum(const D& d) { return fluid_momentum(d, CTL(after, 0)); }
template <class D> int op_local_melt_correction(const D& d) {
  return d.template launch<k2_local_melt_correction>(kOne);
}
template <class D> int op_finish_melt_momentum(const D& d) {
  return d.template launch<k2_finish_melt_momentum>(kOne);
}
template <class D> int op_measure_aperture(const D& d) {
  NEED(d, kCells, 6);
  TRY(d.template launch<k2_aperture_partials>(kRuns));
  return d.template finish_tail<k2_check_aperture>(kCells, 6, CTL(aperture, 0), 0x10u, 0x20u, 0u);
}
template <class D> int op_build_aperture_targets(const D& d) {
  NEED(d, kCells, 3);
  TRY(d.template launch<k2_build_aperture_targets>(kRuns));
  // the transfer's |energy correction| (simulator.py:829-859) is added as
  // soon as the targets are folded
  return d.template finish_tail<k2_add_correction_abs>(kCells, 3, CTL(targets, 0), 0u, 0u, 0u);
}
template <class D> int op_apply_aperture_transfer(const D& d) {
  return d.template launch<k2_apply_aperture_transfer>(kCells);
}
template <class D> int op_finish_aperture_transfer(const D& d) {
  NEED(d, kCells, 2);
  TRY(d.template launch<k2_water_totals_partials>(kRuns));
  return d.finish(kCells, 2, CTL(transfer, 0), 0u, 0u, 0u);
}
template <class D> int op_transfer_aperture(const D& d) {
  NEED(d, kCells, 2);
  TRY(d.template launch<k2_transfer_partials>(kRuns));
  return d.finish(kCells, 2, CTL(transfer, 0), 0u, 0u, 0u);
}
// measure, build, transfer: the whole of simulator.py:511-548.
template <class D> int op_synchronize_aperture(const D& d) {
  TRY(op_measure_aperture(d));
  TRY(op_build_aperture_targets(d));
  return op_transfer_aperture(d);
}
// The fixed launches of a step after its populations have streamed
// (simulator.py:2203-2210 and the outflow measurement of :2233-2247).
template <class D> int op_after_stream(const D& d) {
  TRY(op_stream(d, 0, kStreamUpdate));
  TRY(op_update_pressure(d));
  TRY(op_integrate_rigid(d));
  TRY(op_body_fraction(d, 0));
  TRY(op_contact_support(d, 1, 0));
  TRY(op_project_inside(d));
  TRY(op_body_fraction(d, 1));
  TRY(op_contact_support(d, 1, 1));
  TRY(op_commit_raster(d));
  TRY(op_update_solid_mask(d, 0));
  TRY(op_refill(d));
  return op_measure_outflow(d);
}
template <class D> int op_body_conduction(const D& d, typename D::Real dt) {
  return d.template launch<k2_body_conduction>(kBody, dt);
}
template <class D> int op_conduction_flux(const D& d, int axis) {
  if (axis != 0 && axis != 1) return ICY2D_ERR_ARGUMENT;
  const int shape = axis == 0 ? kFaceX : kFaceY;
  NEED(d, shape, 1);
  TRY(d.template launch<k2_conduction_flux>(shape, axis));
  // simulator.py:630-631: the power is reset before the x faces and summed over both passes
  return d.finish(shape, 1, CTL(boundary_power, 0), 0u, 0u, axis == 0 ? 0u : 0x1u);
}
template <class D> int op_advection_flux(const D& d, int axis) {
  if (axis != 0 && axis != 1) return ICY2D_ERR_ARGUMENT;
  return d.template launch<k2_advection_flux>(axis == 0 ? kFaceX : kFaceY, axis);
}
template <class D> int op_update_water(const D& d, typename D::Real dt, int volume) {
  return d.template launch<k2_update_water>(kCells, dt, volume);
}
template <class D> int op_reset_interval_sources(const D& d) {
  return d.template launch<k2_reset_interval_sources>(kOne);
}
template <class D> int op_accumulate_boundary_heat(const D& d, typename D::Real dt) {
  return d.template launch<k2_accumulate_boundary_heat>(kOne, dt);
}
template <class D> int op_exchange_heat(const D& d, typename D::Real dt) {
  return d.template launch<k2_exchange_heat>(kCells, dt);
}
template <class D> int op_phase_change(const D& d) {
  NEED(d, kBody, 1);
  TRY(d.template launch<k2_phase_change>(kBody));
  return d.finish(kBody, 1, CTL(interval, 0), 0u, 0u, 0x1u);
}
template <class D> int op_freeze_eligibility(const D& d) {
  return d.template launch<k2_freeze_eligibility>(kCells);
}
template <class D> int op_inject_melt(const D& d) {
  NEED(d, kBody, 3);
  TRY(d.template launch<k2_inject_melt>(kBody));
  TRY(d.template launch<k2_fold_injection>(kBody));
  // partial columns: assigned melt, unassigned mass, unassigned energy
  return d.template finish_tail<k2_store_injection>(kBody, 3, TAIL(3), 0u, 0u, 0u);
}
template <class D> int op_measure_fallback(const D& d) {
  NEED(d, kCells, 2);
  TRY(d.template launch<k2_fallback_partials>(kCells));
  return d.finish(kCells, 2, CTL(fallback, 0), 0u, 0u, 0u);
}
template <class D> int op_apply_fallback(const D& d, int use_free) {
  TRY(d.template launch<k2_count_fallback>(kOne, use_free));
  return d.template launch<k2_apply_fallback>(kCells, use_free);
}
template <class D> int op_reduce_totals(const D& d) {
  NEED(d, kTotals, 4);
  TRY(d.template launch<k2_totals_partials>(kTotals));
  return d.finish(kTotals, 4, CTL(totals, 0), 0u, 0u, 0u);
}

bool valid(const icy2d_grid* g) {
  return g && g->nx > 0 && g->ny > 0 && g->body_nx > 0 && g->body_ny > 0 && g->control && g->partials &&
         g->partials_capacity >= 8;
}
bool valid_batch(const icy2d_batch* b) {
  if (!b || b->ncases <= 0 || !b->grids || !b->first_block) return false;
  for (int t : {b->collide_threads, b->stream_threads})
    if (t != 128 && t != 256 && t != 512) return false;
  return true;
}
// Partials a case needs for its largest reduction (K columns per block plus
// the eight tail slots).
long partials_needed(const icy2d_grid& g) {
  long need = 0;
  auto take = [&](int shape, int K) {
    const long v = (long)shape_blocks(g, shape) * K;
    if (v > need) need = v;
  };
  take(kCells, 6);
  take(kCells128, 3);
  take(kCells512, 3);
  take(kTiles128, 3);
  take(kTiles256, 3);
  take(kTiles512, 3);
  take(kBody, 4);
  take(kFaceX, 1);
  take(kFaceY, 1);
  take(kTotals, 4);
  return need + 8;
}

}  // namespace icy2

using namespace icy2;

#define S(stream) ((hipStream_t)(stream))
#define SINGLE(name, params, ...)                                 \
  int icy2d_##name(const icy2d_grid* g ICY2D_EXPAND params, void* stream) { \
    if (!valid(g)) return ICY2D_ERR_ARGUMENT;                      \
    return op_##name(One{*g, S(stream)} __VA_ARGS__);              \
  }
#define BATCH(name, params, ...)                                         \
  int icy2d_batch_##name(const icy2d_batch* b ICY2D_EXPAND params, void* stream) { \
    if (!valid_batch(b)) return ICY2D_ERR_ARGUMENT;                       \
    return op_##name(Many{*b, S(stream)} __VA_ARGS__);                    \
  }
#define ICY2D_EXPAND(...) __VA_ARGS__
#define BOTH(name, params, ...) SINGLE(name, params, __VA_ARGS__) BATCH(name, params, __VA_ARGS__)
#define PC(x) PerCase{x}

// The population stores' stochastic rounding applied `steps` times to each
// value (icy2d_probe_rounding).
__global__ void k2_probe_rounding(const float* __restrict__ values, int count, float lift, int steps,
                                  uint32_t first_step, float scale, float* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  __half stored = __float2half(values[i] * scale);
  for (int s = 0; s < steps; ++s)
    stored = half_stochastic(__half2float(stored) + lift * scale, (uint32_t)i * 2u, first_step + (uint32_t)s);
  out[i] = __half2float(stored) / scale;
}

// The batch counterpart of the host's plane swap after a fused collide-stream.
__global__ void k2_swap_flow_planes(icy2d_batch b) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= b.ncases) return;
  icy2d_grid* g = const_cast<icy2d_grid*>(b.grids) + c;
  float* t = g->f;
  g->f = g->fbuf;
  g->fbuf = t;
  t = g->h;
  g->h = g->hbuf;
  g->hbuf = t;
}

extern "C" {

BOTH(body_fraction, (, int only_if_projected), , only_if_projected)
BOTH(commit_raster, ())
BOTH(contact_support, (, int reduce, int only_if_projected), , reduce, only_if_projected)
BOTH(integrate_rigid, ())
BOTH(project_inside, ())
BOTH(update_solid_mask, (, int init), , init)
BOTH(reduce_mass_properties, ())
BOTH(apply_mass_properties, (, int initialize), , initialize)
BOTH(collide, (, int with_momentum), , with_momentum)
BOTH(stream, (, int phase_only, int mode), , phase_only, mode)
BOTH(collide_stream, ())
BOTH(update_pressure, ())
BOTH(refill, ())
BOTH(measure_outflow, ())
BOTH(clip_phase, (, double max_bulk_l1), , max_bulk_l1)
BOTH(seed_projection, ())
BOTH(dilate_projection, (, int primary_to_next), , primary_to_next)
BOTH(dilate_band, (, int radius), , radius)
BOTH(snapshot_melt_momentum, ())
BOTH(reduce_provisional_momentum, ())
BOTH(melt_weight_geometry, ())
BOTH(apply_melt_correction, ())
BOTH(reduce_final_momentum, ())
BOTH(local_melt_correction, ())
BOTH(finish_melt_momentum, ())
BOTH(measure_aperture, ())
BOTH(build_aperture_targets, ())
BOTH(apply_aperture_transfer, ())
BOTH(finish_aperture_transfer, ())
BOTH(transfer_aperture, ())
SINGLE(synchronize_aperture, ())
SINGLE(after_stream, ())
BOTH(conduction_flux, (, int axis), , axis)
BOTH(advection_flux, (, int axis), , axis)
BOTH(reset_interval_sources, ())
BOTH(phase_change, ())
BOTH(freeze_eligibility, ())
BOTH(inject_melt, ())
BOTH(measure_fallback, ())
BOTH(apply_fallback, (, int use_free), , use_free)
BOTH(reduce_totals, ())
SINGLE(prepare_cut_links, ())
int icy2d_batch_swap_flow_planes(const icy2d_batch* b, void* stream) {
  if (!valid_batch(b)) return ICY2D_ERR_ARGUMENT;
  k2_swap_flow_planes<<<(b->ncases + 63) / 64, 64, 0, S(stream)>>>(*b);
  return launch_status();
}

// Entry points whose double arguments are one value per case in a batch.
SINGLE(evaluate_projection, (, double lambda), , lambda)
BATCH(evaluate_projection, (, const double* lambda), , PC(lambda))
SINGLE(apply_projection, (, double lambda), , lambda)
BATCH(apply_projection, (, const double* lambda), , PC(lambda))
SINGLE(projection_residual_weight, (, double residual), , residual)
BATCH(projection_residual_weight, (, const double* residual), , PC(residual))
SINGLE(apply_projection_residual, (, double residual, double weight), , residual, weight)
BATCH(apply_projection_residual, (, const double* residual, const double* weight), , PC(residual), PC(weight))
SINGLE(body_conduction, (, double dt), , dt)
BATCH(body_conduction, (, const double* dt), , PC(dt))
SINGLE(update_water, (, double dt, int volume), , dt, volume)
BATCH(update_water, (, const double* dt, int volume), , PC(dt), volume)
SINGLE(accumulate_boundary_heat, (, double dt), , dt)
BATCH(accumulate_boundary_heat, (, const double* dt), , PC(dt))
SINGLE(exchange_heat, (, double dt), , dt)
BATCH(exchange_heat, (, const double* dt), , PC(dt))

// Initialisation (single case).
int icy2d_initialize_fluid(const icy2d_grid* g, int water_width, int water_height, void* stream) {
  if (!valid(g)) return ICY2D_ERR_ARGUMENT;
  return One{*g, S(stream)}.launch<k2_initialize_fluid>(kCells, water_width, water_height);
}
int icy2d_hydrostatic_equilibrium(const icy2d_grid* g, void* stream) {
  if (!valid(g)) return ICY2D_ERR_ARGUMENT;
  return One{*g, S(stream)}.launch<k2_hydrostatic_equilibrium>(kCells);
}
int icy2d_initialize_water_volume(const icy2d_grid* g, void* stream) {
  if (!valid(g)) return ICY2D_ERR_ARGUMENT;
  const One d{*g, S(stream)};
  NEED(d, kCells, 1);
  TRY(d.launch<k2_water_volume_partials>(kCells));
  return d.template finish_tail<k2_copy_initial_volume>(kCells, 1, CTL(water, 0), 0u, 0u, 0u);
}
int icy2d_recover_initial_moments(const icy2d_grid* g, void* stream) {
  if (!valid(g)) return ICY2D_ERR_ARGUMENT;
  return One{*g, S(stream)}.launch<k2_recover_initial_moments>(kCells);
}
int icy2d_initialize_body_state(const icy2d_grid* g, double ice_temperature, void* stream) {
  if (!valid(g)) return ICY2D_ERR_ARGUMENT;
  return One{*g, S(stream)}.launch<k2_initialize_body_state>(kBody, ice_temperature);
}
int icy2d_initialize_water_state(const icy2d_grid* g, double water_temperature_c, void* stream) {
  if (!valid(g)) return ICY2D_ERR_ARGUMENT;
  const One d{*g, S(stream)};
  TRY(d.launch<k2_initialize_water_state>(kCells, water_temperature_c));
  return d.launch<k2_reset_thermal_diagnostics>(kOne);
}

int icy2d_batch_plan(const icy2d_grid* grids, int32_t ncases, int32_t* first_block, int32_t* total_blocks) {
  if (!grids || ncases <= 0 || !first_block || !total_blocks) return ICY2D_ERR_ARGUMENT;
  for (int c = 0; c < ncases; ++c)
    if (!valid(&grids[c]) || partials_needed(grids[c]) > (long)grids[c].partials_capacity) return ICY2D_ERR_ARGUMENT;
  for (int shape = 0; shape < kShapes; ++shape) {
    int32_t* first = first_block + shape * (ncases + 1);
    long total = 0;
    for (int c = 0; c < ncases; ++c) {
      first[c] = (int32_t)total;
      total += shape_blocks(grids[c], shape);
    }
    if (total > 0x7fffffffL) return ICY2D_ERR_ARGUMENT;
    first[ncases] = (int32_t)total;
    total_blocks[shape] = (int32_t)total;
  }
  return 0;
}
void icy2d_batch_abi_size(int32_t* batch) {
  if (batch) *batch = (int32_t)sizeof(icy2d_batch);
}

int icy2d_graph_begin(void* stream) {
  return (int)hipStreamBeginCapture(S(stream), hipStreamCaptureModeThreadLocal);
}
int icy2d_graph_end(void* stream, void** graph) {
  if (!graph) return ICY2D_ERR_ARGUMENT;
  *graph = nullptr;
  hipGraph_t captured = nullptr;
  if (hipError_t e = hipStreamEndCapture(S(stream), &captured)) return (int)e;
  hipGraphExec_t exec = nullptr;
  const hipError_t e = hipGraphInstantiate(&exec, captured, nullptr, nullptr, 0);
  (void)hipGraphDestroy(captured);
  if (e != hipSuccess) return (int)e;
  *graph = (void*)exec;
  return 0;
}
int icy2d_graph_launch(void* graph, void* stream) {
  if (!graph) return ICY2D_ERR_ARGUMENT;
  return (int)hipGraphLaunch((hipGraphExec_t)graph, S(stream));
}
int icy2d_graph_destroy(void* graph) {
  if (!graph) return 0;
  return (int)hipGraphExecDestroy((hipGraphExec_t)graph);
}
int icy2d_copy_async(void* dst, const void* src, size_t bytes, void* stream) {
  if (!bytes) return 0;
  if (!dst || !src) return ICY2D_ERR_ARGUMENT;
  return (int)hipMemcpyAsync(dst, src, bytes, hipMemcpyDefault, S(stream));
}

// A blocking copy: asynchronous and followed by a synchronisation of the
// stream it took the 24x20x16 tank's eight steps from 1760 to 1950 us.
int icy2d_read_control(const icy2d_grid* g, icy2d_control* host, void* stream) {
  if (!valid(g) || !host) return ICY2D_ERR_ARGUMENT;
  return (int)hipMemcpyWithStream(host, g->control, sizeof(*host), hipMemcpyDeviceToHost, S(stream));
}

int icy2d_probe_rounding(const float* values, int count, float lift, int steps, uint32_t first_step, float scale,
                         float* out, void* stream) {
  if (count < 0 || steps < 0 || (count && (!values || !out)) || !(scale > 0.0f)) return ICY2D_ERR_ARGUMENT;
  if (!count) return 0;
  k2_probe_rounding<<<(count + kBlock - 1) / kBlock, kBlock, 0, S(stream)>>>(values, count, lift, steps, first_step,
                                                                             scale, out);
  return (int)hipGetLastError();
}

void icy2d_abi_sizes(int32_t* grid, int32_t* control) {
  if (grid) *grid = (int32_t)sizeof(icy2d_grid);
  if (control) *control = (int32_t)sizeof(icy2d_control);
}

}  // extern "C"

#ifndef ICY_SOURCE_HASH
#define ICY_SOURCE_HASH "unrecorded"
#endif
extern "C" const char* icy2d_source_hash(void) { return ICY_SOURCE_HASH; }
