// Finite-volume heat transport and disappearing ice (iceflow3d/thermal.py),
// material-grid mass reductions (simulator.py:738-776) and initialisation.
//
// Water stores volume [m^3] and sensible energy [J] per world cell; ice
// stores mass [kg] and sensible energy [J] per material cell.  Scalar sums
// (remap energy, discarded heat) are reduced per wave64 before one atomic.
#include "icy3d_device.h"

namespace icy {

__device__ __forceinline__ float water_target(const icy3d_grid& g, int n) {
  return (g.id[n] == -1 && g.phi[n] > 1e-3f) ? g.phi[n] * g.cell_volume : 0.0f;
}

// thermal.py:98-118: the energy a cell holds after the remap (its volume is
// water_target): the cell's own specific energy, or for a newly wet cell the
// mean over its wet 3x3x3 neighbourhood.
__device__ __forceinline__ float remapped_energy(const icy3d_grid& g, int n, float target) {
  float specific = 0.0f;
  if (target > 0.0f) {
    const float v = g.water_volume[n];
    if (v > 1e-30f) {
      specific = g.water_energy[n] / v;
    } else {
      const Cell c = cell_of(g, n);
      float total = 0.0f;
      for (int a = -1; a <= 1; ++a)
        for (int b = -1; b <= 1; ++b)
          for (int d = -1; d <= 1; ++d) {
            int i = c.i + a, j = c.j + b, k = c.k + d;
            if (!inside(g, i, j, k)) continue;
            int m = lin(g, i, j, k);
            if (g.water_volume[m] > 1e-30f) {
              specific += g.water_energy[m];
              total += g.water_volume[m];
            }
          }
      if (total > 1e-30f) specific /= total;
    }
  }
  // rounded here as the two-kernel remap rounds it into target_energy: with
  // contraction off the product cannot fuse into a caller's subtraction
  // (__fmul_rn is a plain contractable multiply in this HIP)
  {
#pragma clang fp contract(off)
    return target * specific;
  }
}
// thermal.py:98-127 in one pass: the remapped volume and energy go to
// volume_out / energy_out (the caller swaps them with the water planes) and
// the remap energy is summed per block as k_commit_water_targets does.
__global__ void k_synchronize_water_into(icy3d_grid g, float* __restrict__ volume_out,
                                         float* __restrict__ energy_out) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  float delta = 0.0f;
  if (n < (int)cells(g)) {
    const float target = water_target(g, n);
    const float e = remapped_energy(g, n, target);
    delta = e - g.water_energy[n];
    volume_out[n] = target;
    energy_out[n] = e;
  }
  const float total = block_sum(delta);
  if (threadIdx.x == 0) g.partials[blockIdx.x] = total;
}
// thermal.py:98-118
__global__ void k_build_water_targets(icy3d_grid g) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (int)cells(g)) return;
  const float target = water_target(g, n);
  float specific = 0.0f;
  if (target > 0.0f) {
    const float v = g.water_volume[n];
    if (v > 1e-30f) {
      specific = g.water_energy[n] / v;
    } else {
      const Cell c = cell_of(g, n);
      float total = 0.0f;
      for (int a = -1; a <= 1; ++a)
        for (int b = -1; b <= 1; ++b)
          for (int d = -1; d <= 1; ++d) {
            int i = c.i + a, j = c.j + b, k = c.k + d;
            if (!inside(g, i, j, k)) continue;
            int m = lin(g, i, j, k);
            if (g.water_volume[m] > 1e-30f) {
              specific += g.water_energy[m];
              total += g.water_volume[m];
            }
          }
      if (total > 1e-30f) specific /= total;
    }
  }
  g.target_energy[n] = target * specific;
}
// thermal.py:120-127 (remap energy as a deterministic two-stage sum)
__global__ void k_commit_water_targets(icy3d_grid g) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  float delta = 0.0f;
  if (n < (int)cells(g)) {
    const float e = g.target_energy[n];
    delta = e - g.water_energy[n];
    g.water_volume[n] = water_target(g, n);
    g.water_energy[n] = e;
  }
  const float total = block_sum(delta);
  if (threadIdx.x == 0) g.partials[blockIdx.x] = total;
}
// thermal.py:88-96
__global__ void k_initialize_water_heat(icy3d_grid g) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (int)cells(g)) return;
  const float v = water_target(g, n);
  g.water_volume[n] = v;
  g.water_energy[n] = v * g.rho_cp * (g.water_t0 - g.tm);
}

// The advection flux through the +a face of cell p into q (thermal.py:133-169,
// advect branch): volume and energy carried upwind, zero unless p is fluid,
// q is a fluid cell and both hold water.
__device__ __forceinline__ void advect_face(const icy3d_grid& g, const float* __restrict__ volume,
                                            const float* __restrict__ energy, int p, int q, int a, float& vf,
                                            float& ef) {
  const size_t N = cells(g);
  vf = 0.0f;
  ef = 0.0f;
  const float vi = volume[p], vj = volume[q];
  if (!(vi > 1e-30f && vj > 1e-30f)) return;
  const float speed = 0.5f * (g.u[a * N + p] + g.u[a * N + q]) * g.velocity_m_s;
  float V = vi, E = energy[p];
  if (speed < 0.0f) {
    V = vj;
    E = energy[q];
  }
  vf = speed * fminf(1.0f, V / g.cell_volume) * (g.dx * g.dx);
  ef = vf * E / V;
}
// thermal.py:133-169
__global__ void k_thermal_fluxes(icy3d_grid g, int advect) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t N = cells(g);
  if (n >= (int)N) return;
  const Cell c = cell_of(g, n);
  float ef[3] = {0.0f, 0.0f, 0.0f}, vf[3] = {0.0f, 0.0f, 0.0f};
  if (g.id[n] == -1) {
    const float vi = g.water_volume[n];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      int i = c.i + (a == 0), j = c.j + (a == 1), k = c.k + (a == 2);
      if (!fluid_at(g, i, j, k)) continue;
      const int m = lin(g, i, j, k);
      const float vj = g.water_volume[m];
      if (!(vi > 1e-30f && vj > 1e-30f)) continue;
      if (advect) {
        advect_face(g, g.water_volume, g.water_energy, n, m, a, vf[a], ef[a]);
      } else {
        const float aperture = fminf(vi, vj) / g.cell_volume;
        ef[a] = g.k_water * g.dx * aperture * (water_temperature(g, n) - water_temperature(g, m));
      }
    }
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    g.energy_flux[a * N + n] = ef[a];
    g.volume_flux[a * N + n] = vf[a];
  }
}
// The conduction flux through the +a face of cell p into its neighbour q
// (thermal.py:133-169, conduct branch), exactly as k_thermal_fluxes forms it
// for p: zero unless p and q are fluid and both hold water.
__device__ __forceinline__ float conduction_face(const icy3d_grid& g, int p, int pi, int pj, int pk, int a) {
  if (g.id[p] != -1) return 0.0f;
  const int i = pi + (a == 0), j = pj + (a == 1), k = pk + (a == 2);
  if (!fluid_at(g, i, j, k)) return 0.0f;
  const int q = lin(g, i, j, k);
  const float vi = g.water_volume[p], vj = g.water_volume[q];
  if (!(vi > 1e-30f && vj > 1e-30f)) return 0.0f;
  const float aperture = fminf(vi, vj) / g.cell_volume;
  return g.k_water * g.dx * aperture * (water_temperature(g, p) - water_temperature(g, q));
}
// thermal.py:133-184 with advect = 0 in one pass: each cell forms the
// conduction fluxes of its six faces (each face identically by its two
// cells, in the order k_apply_thermal_fluxes adds them) and writes its
// updated energy to energy_out; no flux plane is stored.
__global__ void k_conduct_water(icy3d_grid g, float dt, float* __restrict__ energy_out) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (int)cells(g)) return;
  const Cell c = cell_of(g, n);
  float de = 0.0f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    de += conduction_face(g, n, c.i, c.j, c.k, a);
    const int i = c.i - (a == 0), j = c.j - (a == 1), k = c.k - (a == 2);
    if (inside(g, i, j, k)) de -= conduction_face(g, lin(g, i, j, k), i, j, k, a);
  }
  energy_out[n] = g.water_energy[n] - dt * de;
}
// thermal.py:171-184
__global__ void k_apply_thermal_fluxes(icy3d_grid g, float dt, int advect) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t N = cells(g);
  if (n >= (int)N) return;
  const Cell c = cell_of(g, n);
  float de = 0.0f, dv = 0.0f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    de += g.energy_flux[a * N + n];
    dv += g.volume_flux[a * N + n];
    int i = c.i - (a == 0), j = c.j - (a == 1), k = c.k - (a == 2);
    if (inside(g, i, j, k)) {
      const int m = lin(g, i, j, k);
      de -= g.energy_flux[a * N + m];
      dv -= g.volume_flux[a * N + m];
    }
  }
  g.water_energy[n] -= dt * de;
  if (advect) g.water_volume[n] -= dt * dv;
}
// thermal.py:133-184, advection in one pass: each cell forms the fluxes of
// its six faces from the current water volume and energy (every face is
// formed identically by its two cells) and writes its updated values to
// volume_out / energy_out, so no flux plane is stored.  The caller swaps the
// output planes with the grid's water planes.
__global__ void k_advect_water(icy3d_grid g, float dt, float* __restrict__ volume_out,
                               float* __restrict__ energy_out) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (int)cells(g)) return;
  const Cell c = cell_of(g, n);
  const bool own_fluid = g.id[n] == -1;
  float de = 0.0f, dv = 0.0f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    float vf = 0.0f, ef = 0.0f;
    int i = c.i + (a == 0), j = c.j + (a == 1), k = c.k + (a == 2);
    if (own_fluid && fluid_at(g, i, j, k)) advect_face(g, g.water_volume, g.water_energy, n, lin(g, i, j, k), a, vf, ef);
    de += ef;
    dv += vf;
    i = c.i - (a == 0);
    j = c.j - (a == 1);
    k = c.k - (a == 2);
    if (inside(g, i, j, k)) {
      const int m = lin(g, i, j, k);
      float vb = 0.0f, eb = 0.0f;
      if (own_fluid && g.id[m] == -1) advect_face(g, g.water_volume, g.water_energy, m, n, a, vb, eb);
      de -= eb;
      dv -= vb;
    }
  }
  energy_out[n] = g.water_energy[n] - dt * de;
  volume_out[n] = g.water_volume[n] - dt * dv;
}
// The step's water update in one pass: remap to the phase field
// (thermal.py:98-127), one advection substep (:133-184) and the remap again,
// as k_synchronize_water_into, k_advect_water and k_synchronize_water_into
// form them, face by face and in their order of adds.  A row sweep
// (k_stream_rows): each cell is remapped once on load, z neighbours come from
// the neighbour lanes, y neighbours through LDS, x neighbours from the slab
// before; a cell that the advection empties takes the mean of its advected
// neighbours, formed again from the planes (such cells are rare).  Bound by
// memory: 37 bytes a cell are needed, and 55 move at 256x128x128 at 85% of the
// copy rate (VALUs 32% busy), where the three passes needed 60 and divided seven
// times a cell: 115 us there with their two sums' folds, 60 here.
struct Water {
  float volume, energy;
};
__device__ __forceinline__ Water remapped_cell(const icy3d_grid& g, int n) {
  const float target = water_target(g, n);
  return {target, remapped_energy(g, n, target)};
}
// The flux through the face from cell p to cell q along one axis (advect_face
// on remapped cells; a dry or non-fluid cell has no volume).
__device__ __forceinline__ Water face_of(const icy3d_grid& g, Water p, Water q, float up, float uq) {
  Water f = {0.0f, 0.0f};
  if (!(p.volume > 1e-30f && q.volume > 1e-30f)) return f;
  const float speed = 0.5f * (up + uq) * g.velocity_m_s;
  const Water donor = speed < 0.0f ? q : p;
  f.volume = speed * fminf(1.0f, donor.volume / g.cell_volume) * (g.dx * g.dx);
  f.energy = f.volume * donor.energy / donor.volume;
  return f;
}
__device__ __forceinline__ Water advected_cell(const icy3d_grid& g, int i, int j, int k, float dt) {
  const size_t N = cells(g);
  const int n = lin(g, i, j, k);
  const Water own = remapped_cell(g, n);
  float de = 0.0f, dv = 0.0f;
#pragma unroll 1
  for (int face = 0; face < 6; ++face) {  // +x, -x, +y, -y, +z, -z
    const int a = face >> 1, d = (face & 1) ? -1 : 1;
    const int mi = i + (a == 0 ? d : 0), mj = j + (a == 1 ? d : 0), mk = k + (a == 2 ? d : 0);
    if (!inside(g, mi, mj, mk)) continue;
    const int m = lin(g, mi, mj, mk);
    const Water other = remapped_cell(g, m);
    const float u_own = g.u[a * N + n], u_other = g.u[a * N + m];
    const Water f = d > 0 ? face_of(g, own, other, u_own, u_other) : face_of(g, other, own, u_other, u_own);
    de += (float)d * f.energy;
    dv += (float)d * f.volume;
  }
  return {own.volume - dt * dv, own.energy - dt * de};
}
__device__ __forceinline__ float advected_mean(const icy3d_grid& g, int i, int j, int k, float dt) {
  float specific = 0.0f, total = 0.0f;
#pragma unroll 1
  for (int q = 0; q < 27; ++q) {
    const int ni = i + cx(q), nj = j + cy(q), nk = k + cz(q);
    if (!inside(g, ni, nj, nk)) continue;
    const Water w = advected_cell(g, ni, nj, nk, dt);
    if (w.volume > 1e-30f) {
      specific += w.energy;
      total += w.volume;
    }
  }
  return total > 1e-30f ? specific / total : specific;
}
__global__ void __launch_bounds__(kWaterThreads)
    k_water_rows(icy3d_grid g, StreamTiles T, float dt, float* __restrict__ volume_out,
                 float* __restrict__ energy_out) {
  __shared__ float row_v[2][sweep_cells(kWaterThreads)], row_e[2][sweep_cells(kWaterThreads)],
      row_u[2][sweep_cells(kWaterThreads)];
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
  int label = -2;
  float phi = 0.0f, volume = 0.0f, energy = 0.0f, u[3] = {0.0f, 0.0f, 0.0f};
  auto fetch = [&](int s) __attribute__((always_inline)) {
    label = -2;
    phi = volume = energy = 0.0f;
    if (present && s >= 0 && s < g.nx) {
      const unsigned n = (unsigned)s * plane + in_plane, o = 4u * n;
      label = g.id[n];
      phi = plane_get(g.phi, o);
      volume = plane_get(g.water_volume, o);
      energy = plane_get(g.water_energy, o);
#pragma unroll
      for (int e = 0; e < 3; ++e) u[e] = plane_get(g.u + e * N, o);
    }
  };
  fetch(x0 - 1);
  // The last slab's cell: its remapped water, x velocity, the flux through
  // its lower x face and those through its y and z faces (upper, lower).
  Water last = {0.0f, 0.0f}, x_in = {0.0f, 0.0f}, y_up = {0.0f, 0.0f}, y_lo = {0.0f, 0.0f}, z_up = {0.0f, 0.0f},
        z_lo = {0.0f, 0.0f};
  float last_u = 0.0f, first_change = 0.0f, second_change = 0.0f;
  for (int s = x0 - 1; s <= x1; ++s) {
    const int buffer = s & 1;
    // The first remap, as water_target and remapped_energy.
    Water now = {label == -1 && phi > 1e-3f ? phi * g.cell_volume : 0.0f, 0.0f};
    if (now.volume > 0.0f) {
      if (volume > 1e-30f) {
#pragma clang fp contract(off)
        now.energy = now.volume * (energy / volume);
      } else {
        now.energy = remapped_energy(g, s * (int)plane + (int)in_plane, now.volume);
      }
    }
    if (owned && s >= x0 && s < x1) first_change += now.energy - energy;
    const float ux = u[0], uy = u[1], uz = u[2];
    if (s < x1) fetch(s + 1);
    const Water below = {from_below(now.volume), from_below(now.energy)};
    const Water above = {from_above(now.volume), from_above(now.energy)};
    const Water z_lo_s = face_of(g, below, now, from_below(uz), uz), z_up_s = face_of(g, now, above, uz, from_above(uz));
    if (sends) {
      row_v[buffer][t] = now.volume;
      row_e[buffer][t] = now.energy;
      row_u[buffer][t] = uy;
    }
    __syncthreads();
    if (owned) {
      const Water y_lo_s = face_of(g, Water{row_v[buffer][t - L], row_e[buffer][t - L]}, now, row_u[buffer][t - L], uy);
      const Water y_up_s = face_of(g, now, Water{row_v[buffer][t + L], row_e[buffer][t + L]}, uy, row_u[buffer][t + L]);
      const Water x_face = face_of(g, last, now, last_u, ux);  // between the slabs s - 1 and s
      if (s > x0) {
        const float de = ((((x_face.energy - x_in.energy) + y_up.energy) - y_lo.energy) + z_up.energy) - z_lo.energy;
        const float dv = ((((x_face.volume - x_in.volume) + y_up.volume) - y_lo.volume) + z_up.volume) - z_lo.volume;
        const float e2 = last.energy - dt * de, v2 = last.volume - dt * dv, target = last.volume;
        float out = 0.0f;
        if (target > 0.0f) {
#pragma clang fp contract(off)
          out = target * (v2 > 1e-30f ? e2 / v2 : advected_mean(g, s - 1, j, k, dt));
        }
        second_change += out - e2;
        const unsigned o = 4u * ((unsigned)(s - 1) * plane + in_plane);
        plane_set(volume_out, o, target);
        plane_set(energy_out, o, out);
      }
      x_in = x_face;
      y_up = y_up_s;
      y_lo = y_lo_s;
      z_up = z_up_s;
      z_lo = z_lo_s;
    }
    last = now;
    last_u = ux;
  }
  const float first = block_sum(first_change), second = block_sum(second_change);
  if (threadIdx.x == 0) {
    g.partials[blockIdx.x] = first;
    g.partials[gridDim.x + blockIdx.x] = second;
  }
}
// Adds both remaps' sums to the remap energy, the first remap's first.
__global__ void __launch_bounds__(kFinishThreads) k_fold_remaps(icy3d_grid g, int blocks) {
  const float first = finish_total(g.partials, blocks), second = finish_total(g.partials + blocks, blocks);
  if (threadIdx.x == 0) {
    g.control->remap_energy += first;
    g.control->remap_energy += second;
  }
}
// thermal.py:186-206
__global__ void k_measure_outflow(icy3d_grid g) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t N = cells(g);
  float rate = 0.0f;
  if (n < (int)N && g.id[n] == -1 && g.water_volume[n] > 1e-30f) {
    const Cell c = cell_of(g, n);
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int sign = 0; sign < 2; ++sign) {
        const int d = 2 * sign - 1;
        int i = c.i + (a == 0) * d, j = c.j + (a == 1) * d, k = c.k + (a == 2) * d;
        if (!fluid_at(g, i, j, k)) continue;
        const int m = lin(g, i, j, k);
        if (g.water_volume[m] > 1e-30f) rate += fmaxf(0.0f, (float)d * 0.5f * (g.u[a * N + n] + g.u[a * N + m]));
      }
  }
  if (isnan(rate)) rate = 0.0f;
  rate = wave_max(rate);
  if (wave_leader() && rate > 0.0f) atomic_max_nonneg(&g.control->max_outflow, rate);
}
__global__ void k_reset_outflow(icy3d_grid g) { g.control->max_outflow = 0.0f; }

// thermal.py:53-62
__global__ void k_initialize_material(icy3d_grid g) {
  size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t total = (size_t)g.bodies * g.mx * g.my * g.mz;
  if (t >= total) return;
  int k = t % g.mz, j = (t / g.mz) % g.my, i = (t / ((size_t)g.mz * g.my)) % g.mx;
  int b = t / ((size_t)g.mz * g.my * g.mx);
  if (!mat_inside(g, b, i, j, k)) return;
  g.material_mass[t] = g.initial_cell_mass;
  g.material_energy[t] = g.initial_cell_mass * g.cp_ice * (g.body_t0[b] - g.tm);
}
// thermal.py:260-281
__global__ void k_body_conduction(icy3d_grid g, float dt) {
  size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t total = (size_t)g.bodies * g.mx * g.my * g.mz;
  if (t >= total) return;
  int k = t % g.mz, j = (t / g.mz) % g.my, i = (t / ((size_t)g.mz * g.my)) % g.mx;
  int b = t / ((size_t)g.mz * g.my * g.mx);
  const float mass = g.material_mass[t];
  float heat = 0.0f;
  if (mass > 0.0f) {
    const float temp = ice_temperature(g, b, i, j, k);
    const int faces[6][3] = {{1, 0, 0}, {-1, 0, 0}, {0, 1, 0}, {0, -1, 0}, {0, 0, 1}, {0, 0, -1}};
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      int fi = i + faces[f][0], fj = j + faces[f][1], fk = k + faces[f][2];
      if (!mat_inside(g, b, fi, fj, fk)) continue;
      const float other = g.material_mass[mat_index(g, b, fi, fj, fk)];
      if (other > 0.0f) {
        const float aperture = fminf(mass, other) / g.initial_cell_mass;
        heat += dt * g.k_ice * g.dx * aperture * (ice_temperature(g, b, fi, fj, fk) - temp);
      }
    }
  }
  g.material_heat[t] = heat;
}


// The exchange scatters its heat in fixed point: units of 2^-46 of the
// latent heat of one full material cell.
__device__ __forceinline__ double exchange_fixed_scale(const icy3d_grid& g) {
  return 0x1p46 / ((double)g.latent * (double)g.initial_cell_mass);
}

// thermal.py:308-392: seven world samples x eight trilinear material donors.
__device__ void exchange_heat_cell(const icy3d_grid& g, const Cell& c, float dt) {
  const int n = c.n;
  if (!(g.water_volume[n] > 1e-30f && g.id[n] == -1)) return;
  const int offs[7][3] = {{1, 0, 0}, {-1, 0, 0}, {0, 1, 0}, {0, -1, 0}, {0, 0, 1}, {0, 0, -1}, {0, 0, 0}};
  // The seven samples' coverage labels and fractions, loaded together: they
  // decide whether the cell touches thermal ice (thermal.py:283-293) and
  // each sample's body.
  int face_b[7];
  float face_fraction[7];
  bool touches = false;
#pragma unroll
  for (int f = 0; f < 7; ++f) {
    const int ji = c.i + offs[f][0], jj = c.j + offs[f][1], jk = c.k + offs[f][2];
    face_b[f] = -1;
    face_fraction[f] = 0.0f;
    if (inside(g, ji, jj, jk)) {
      const int m = lin(g, ji, jj, jk);
      face_b[f] = g.cov_id[m];
      face_fraction[f] = g.coverage[m];
    }
  }
#pragma unroll
  for (int f = 0; f < 7; ++f) touches = touches || (face_b[f] >= 0 && face_fraction[f] > 1e-8f);
  if (!touches) return;
  float heat[56];
  int body[7], base[7][3];
  float requested = 0.0f;
  const float tw = water_temperature(g, n);
  const float aperture = g.water_volume[n] / g.cell_volume;
  const float gain = g.exchange_gain ? g.exchange_gain[n] : 1.0f;
  const float kh = 2.0f * g.k_water * g.k_ice / (g.k_water + g.k_ice);
  for (int f = 0; f < 7; ++f) {
    body[f] = 0;
    base[f][0] = base[f][1] = base[f][2] = 0;
    for (int s = 0; s < 8; ++s) heat[8 * f + s] = 0.0f;
    const int ji = c.i + offs[f][0], jj = c.j + offs[f][1], jk = c.k + offs[f][2];
    const int b = face_b[f];
    const float fraction = face_fraction[f];
    if (!(b >= 0 && fraction > 1e-8f)) continue;
    float grid[3], part[3];
    material_grid(g, ji + 0.5f, jj + 0.5f, jk + 0.5f, b, grid);
    for (int a = 0; a < 3; ++a) {
      base[f][a] = (int)floorf(grid[a]);
      part[a] = grid[a] - (float)base[f][a];
    }
    body[f] = b;
    const float contact = fminf(aperture, fminf(1.0f, fraction / g.threshold));
    // The eight donors' mass and energy are loaded together (a donor outside
    // the material grid reads as massless), then used in order.
    float donor_mass[8], donor_energy[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int ki = base[f][0] + (s >> 2), kj = base[f][1] + ((s >> 1) & 1), kk = base[f][2] + (s & 1);
      donor_mass[s] = donor_energy[s] = 0.0f;
      if (mat_inside(g, b, ki, kj, kk)) {
        const size_t m = mat_index(g, b, ki, kj, kk);
        donor_mass[s] = g.material_mass[m];
        donor_energy[s] = g.material_energy[m];
      }
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      int a = s >> 2, cc = (s >> 1) & 1, d = s & 1;
      const float mass = donor_mass[s];
      if (!(mass > 0.0f)) continue;
      const float w = (a ? part[0] : 1.0f - part[0]) * (cc ? part[1] : 1.0f - part[1]) * (d ? part[2] : 1.0f - part[2]);
      const float share = w * mass / (g.initial_cell_mass * fraction);
      float t_ice = g.tm;  // ice_temperature of the donor
      if (mass > 1e-30f) t_ice += donor_energy[s] / (g.cp_ice * mass);
      const float value = gain * dt * kh * g.dx * contact * share * fmaxf(0.0f, tw - t_ice);
      heat[8 * f + s] = value;
      requested += value;
    }
  }
  const float scale = fminf(1.0f, fmaxf(0.0f, g.water_energy[n]) / fmaxf(requested, 1e-30f));
  const double fixed = exchange_fixed_scale(g);
  for (int f = 0; f < 7; ++f)
    for (int s = 0; s < 8; ++s) {
      const float value = scale * heat[8 * f + s];
      if (value > 0.0f) {
        int a = s >> 2, cc = (s >> 1) & 1, d = s & 1;
        const size_t m = mat_index(g, body[f], base[f][0] + a, base[f][1] + cc, base[f][2] + d);
        if ((double)value * fixed <= kFixedTermLimit)
          add_fixed(reinterpret_cast<long long*>(g.heat_acc) + m, to_fixed(value, fixed));
        else
          g.material_heat[m] = __builtin_inff();  // flagged by the heat check after melting
      }
    }
  g.water_energy[n] -= scale * requested;
  if (g.exchange_heat_out) g.exchange_heat_out[n] += scale * requested;
}

__global__ void k_exchange_heat(icy3d_grid g, int lo0, int lo1, int lo2, int ex, int ey, int ez, float dt) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ex * ey * ez) return;
  Cell c;
  c.k = lo2 + t % ez;
  c.j = lo1 + (t / ez) % ey;
  c.i = lo0 + t / (ez * ey);
  c.n = lin(g, c.i, c.j, c.k);
  exchange_heat_cell(g, c, dt);
}

// Adds the exchange's fixed-point heat to material_heat and clears the
// accumulator for the next exchange.
__global__ void k_fold_exchange_heat(icy3d_grid g) {
  size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)g.bodies * g.mx * g.my * g.mz) return;
  const long long q = reinterpret_cast<long long*>(g.heat_acc)[t];
  if (q == 0) return;
  g.material_heat[t] += (float)((double)q / exchange_fixed_scale(g));
  g.heat_acc[t] = 0;
}

// thermal.py:401-415
__global__ void k_apply_melting(icy3d_grid g) {
  size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t total = (size_t)g.bodies * g.mx * g.my * g.mz;
  float discarded = 0.0f;
  if (t < total) {
    float mass = g.material_mass[t];
    float energy = g.material_energy[t] + g.material_heat[t];
    if (energy > 0.0f) {
      const float melted = fminf(mass, energy / g.latent);
      discarded += energy - melted * g.latent;
      mass -= melted;
      energy = 0.0f;
    }
    if (mass <= 1e-6f * g.initial_cell_mass) {
      discarded += energy - mass * g.latent;
      mass = 0.0f;
      energy = 0.0f;
    }
    g.material_mass[t] = mass;
    g.material_energy[t] = energy;
  }
  const float block_total = block_sum(discarded);
  if (threadIdx.x == 0) g.partials[blockIdx.x] = block_total;
}

// simulator.py:738-776 in two deterministic stages.  Stage one: block
// (body, chunk) gives each thread one material column (FP32 sums along z),
// folds the block's 19 values (mass, first and second moments, lower and
// upper bounds) in a fixed tree in LDS and writes them as a partial.  Stage
// two folds a body's chunks in order into control->reduced.  A body with no
// mass keeps zero moments and the bounds +-1e9.
constexpr int kReduceThreads = 256;
__global__ void __launch_bounds__(kReduceThreads) k_reduce_mass(icy3d_grid g, int chunks) {
  __shared__ float part[ICY3D_REDUCED_STRIDE][kReduceThreads];
  const int b = blockIdx.x / chunks, chunk = blockIdx.x - b * chunks;
  const int column = chunk * kReduceThreads + threadIdx.x;
  const int* size = g.material_size + 3 * b;
  float total = 0.0f, first[3] = {0, 0, 0}, second[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  float lower[3] = {1e9f, 1e9f, 1e9f}, upper[3] = {-1e9f, -1e9f, -1e9f};
  if (column < g.mx * g.my) {
    const int i = column / g.my, j = column - i * g.my;
    for (int k = 0; k < g.mz; ++k) {
      const float mass = g.material_mass[mat_index(g, b, i, j, k)] / g.mass_kg;
      if (!(mass > 0.0f)) continue;
      const float p[3] = {(i + 0.5f) - 0.5f * size[0], (j + 0.5f) - 0.5f * size[1], (k + 0.5f) - 0.5f * size[2]};
      const float pp = p[0] * p[0] + p[1] * p[1] + p[2] * p[2];
      total += mass;
#pragma unroll
      for (int a = 0; a < 3; ++a) first[a] += mass * p[a];
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int c = 0; c < 3; ++c) second[3 * a + c] += mass * ((a == c ? pp + 1.0f / 6.0f : 0.0f) - p[a] * p[c]);
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        lower[a] = fminf(lower[a], p[a] - 0.5f);
        upper[a] = fmaxf(upper[a], p[a] + 0.5f);
      }
    }
  }
  const int t = threadIdx.x;
  part[0][t] = total;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    part[1 + a][t] = first[a];
    part[13 + a][t] = lower[a];
    part[16 + a][t] = upper[a];
  }
#pragma unroll
  for (int e = 0; e < 9; ++e) part[4 + e][t] = second[e];
  __syncthreads();
  for (int stride = kReduceThreads / 2; stride > 0; stride >>= 1) {
    if (t < stride) {
#pragma unroll
      for (int e = 0; e < 13; ++e) part[e][t] += part[e][t + stride];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        part[13 + a][t] = fminf(part[13 + a][t], part[13 + a][t + stride]);
        part[16 + a][t] = fmaxf(part[16 + a][t], part[16 + a][t + stride]);
      }
    }
    __syncthreads();
  }
  if (t < ICY3D_REDUCED_STRIDE) g.partials[(size_t)blockIdx.x * ICY3D_REDUCED_STRIDE + t] = part[t][0];
}
__global__ void k_finish_reduced(icy3d_grid g, int chunks) {
  const int b = blockIdx.x, e = threadIdx.x;
  if (e >= ICY3D_REDUCED_STRIDE) return;
  const float* p = g.partials + (size_t)b * chunks * ICY3D_REDUCED_STRIDE + e;
  float v = p[0];
  for (int c = 1; c < chunks; ++c) {
    const float x = p[(size_t)c * ICY3D_REDUCED_STRIDE];
    v = e < 13 ? v + x : (e < 16 ? fminf(v, x) : fmaxf(v, x));
  }
  g.control->reduced[b][e] = v;
}

// thermal.py:417-428
__global__ void k_sample_ice_temperature(icy3d_grid g) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (int)cells(g)) return;
  float t = g.tm;
  const int b = g.id[n];
  if (b >= 0) {
    const Cell c = cell_of(g, n);
    float grid[3];
    material_grid(g, c.i + 0.5f, c.j + 0.5f, c.k + 0.5f, b, grid);
    const int* size = g.material_size + 3 * b;
    int J[3];
    for (int a = 0; a < 3; ++a) J[a] = min(size[a] - 1, max(0, (int)floorf(grid[a] + 0.5f)));
    t = ice_temperature(g, b, J[0], J[1], J[2]);
  }
  g.sampled_ice_t[n] = t;
}
// thermal.py:430-440
__global__ void k_check_heat(icy3d_grid g) {
  size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t N = cells(g);
  const size_t M = (size_t)g.bodies * g.mx * g.my * g.mz;
  int bad = 0;
  if (t < N) {
    const float e = g.water_energy[t], v = g.water_volume[t];
    bad += (!isfinite(e) || e < -1e-10f || v < -1e-20f) ? 1 : 0;
  }
  if (t < M) {
    const float m = g.material_mass[t], e = g.material_energy[t];
    bad += (isnan(m) || !isfinite(e) || m < 0.0f) ? 1 : 0;
  }
  bad = wave_sum_int(bad);
  if (wave_leader() && bad) atomicAdd(&g.control->thermal_invalid, bad);
}
__global__ void k_reset_thermal_invalid(icy3d_grid g) { g.control->thermal_invalid = 0; }

// simulator.py:325-347
__global__ void k_initialize_phase(icy3d_grid g) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  const size_t N = cells(g);
  if (n >= (int)N) return;
  float phi = 0.0f;
  if (g.id[n] == -1) {
    const Cell c = cell_of(g, n);
    float column = fminf((float)g.water_width - c.i - 0.5f, (float)g.water_height - c.j - 0.5f);
    float distance = column;
    if (g.floor_depth > 0) distance = fmaxf(column, (float)(g.boundary + g.floor_depth) - c.j - 0.5f);
    phi = 0.5f + 0.5f * tanhf(2.0f * distance / g.width);
  }
  g.phi[n] = phi;
#pragma unroll
  for (int q = 0; q < 7; ++q) g.h[(size_t)q * N + n] = phase_equilibrium7(q, phi, 0.0f, 0.0f, 0.0f);
}

}  // namespace icy

using namespace icy;

namespace {
bool ok_grid(const icy3d_grid* g) {
  return g && g->nx > 0 && g->ny > 0 && g->nz > 0 && g->bodies >= 0 && g->bodies <= ICY3D_MAX_BODIES && g->control &&
         (size_t)g->nx * g->ny * g->nz < (size_t)INT32_MAX / 16;
}
size_t n_cells(const icy3d_grid& g) { return (size_t)g.nx * g.ny * g.nz; }
size_t n_material(const icy3d_grid& g) { return (size_t)g.bodies * g.mx * g.my * g.mz; }
}  // namespace

extern "C" {

int icy3d_synchronize_water(const icy3d_grid* g, void* stream) {
  if (!ok_grid(g)) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  const unsigned blocks = icy_blocks(n_cells(*g));
  if ((int)blocks > g->partials_capacity) return ICY3D_ERR_ARGUMENT;
  k_build_water_targets<<<blocks, kBlock, 0, s>>>(*g);
  k_commit_water_targets<<<blocks, kBlock, 0, s>>>(*g);
  k_finish_sum<<<1, kFinishThreads, 0, s>>>(g->partials, (int)blocks, &g->control->remap_energy);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_synchronize_water_into(const icy3d_grid* g, float* volume_out, float* energy_out, void* stream) {
  if (!ok_grid(g) || !volume_out || !energy_out) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  const unsigned blocks = icy_blocks(n_cells(*g));
  if ((int)blocks > g->partials_capacity) return ICY3D_ERR_ARGUMENT;
  k_synchronize_water_into<<<blocks, kBlock, 0, s>>>(*g, volume_out, energy_out);
  k_finish_sum<<<1, kFinishThreads, 0, s>>>(g->partials, (int)blocks, &g->control->remap_energy);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_initialize_water_heat(const icy3d_grid* g, void* stream) {
  if (!ok_grid(g)) return ICY3D_ERR_ARGUMENT;
  k_initialize_water_heat<<<icy_blocks(n_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_thermal_fluxes(const icy3d_grid* g, int advect, void* stream) {
  if (!ok_grid(g)) return ICY3D_ERR_ARGUMENT;
  k_thermal_fluxes<<<icy_blocks(n_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g, advect);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_apply_thermal_fluxes(const icy3d_grid* g, float dt, int advect, void* stream) {
  if (!ok_grid(g)) return ICY3D_ERR_ARGUMENT;
  k_apply_thermal_fluxes<<<icy_blocks(n_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g, dt, advect);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_advect_water(const icy3d_grid* g, float dt, float* volume_out, float* energy_out, void* stream) {
  if (!ok_grid(g) || !volume_out || !energy_out) return ICY3D_ERR_ARGUMENT;
  k_advect_water<<<icy_blocks(n_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g, dt, volume_out, energy_out);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_remap_advect_remap(const icy3d_grid* g, float dt, float* volume_out, float* energy_out, void* stream) {
  if (!ok_grid(g) || !volume_out || !energy_out) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  const StreamTiles T = stream_tiles(*g, kWaterThreads);
  const unsigned blocks = stream_blocks(*g, T);
  if ((size_t)2 * blocks > (size_t)g->partials_capacity) return ICY3D_ERR_ARGUMENT;
  k_water_rows<<<blocks, stream_threads(T), 0, s>>>(*g, T, dt, volume_out, energy_out);
  k_fold_remaps<<<1, kFinishThreads, 0, s>>>(*g, (int)blocks);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_conduct_water(const icy3d_grid* g, float dt, float* energy_out, void* stream) {
  if (!ok_grid(g) || !energy_out) return ICY3D_ERR_ARGUMENT;
  k_conduct_water<<<icy_blocks(n_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g, dt, energy_out);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_measure_outflow(const icy3d_grid* g, void* stream) {
  if (!ok_grid(g)) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  k_reset_outflow<<<1, 1, 0, s>>>(*g);
  k_measure_outflow<<<icy_blocks(n_cells(*g)), kBlock, 0, s>>>(*g);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_initialize_material(const icy3d_grid* g, void* stream) {
  if (!ok_grid(g)) return ICY3D_ERR_ARGUMENT;
  size_t n = n_material(*g);
  if (n) k_initialize_material<<<icy_blocks(n), kBlock, 0, (hipStream_t)stream>>>(*g);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_body_conduction(const icy3d_grid* g, float dt, void* stream) {
  if (!ok_grid(g)) return ICY3D_ERR_ARGUMENT;
  size_t n = n_material(*g);
  if (n) k_body_conduction<<<icy_blocks(n), kBlock, 0, (hipStream_t)stream>>>(*g, dt);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_exchange_heat(const icy3d_grid* g, float dt, const int32_t lo[3], const int32_t hi[3], void* stream) {
  if (!ok_grid(g)) return ICY3D_ERR_ARGUMENT;
  const int shape[3] = {g->nx, g->ny, g->nz};
  for (int a = 0; a < 3; ++a)
    if (lo[a] < 0 || hi[a] > shape[a]) return ICY3D_ERR_ARGUMENT;
  int ex = hi[0] - lo[0], ey = hi[1] - lo[1], ez = hi[2] - lo[2];
  if (ex <= 0 || ey <= 0 || ez <= 0) return 0;
  if (n_material(*g) && !g->heat_acc) return ICY3D_ERR_ARGUMENT;
  k_exchange_heat<<<icy_blocks((size_t)ex * ey * ez), kBlock, 0, (hipStream_t)stream>>>(*g, lo[0], lo[1], lo[2], ex,
                                                                                        ey, ez, dt);
  if (const size_t m = n_material(*g)) k_fold_exchange_heat<<<icy_blocks(m), kBlock, 0, (hipStream_t)stream>>>(*g);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_apply_melting(const icy3d_grid* g, void* stream) {
  if (!ok_grid(g)) return ICY3D_ERR_ARGUMENT;
  size_t n = n_material(*g);
  if (!n) return 0;
  const unsigned blocks = icy_blocks(n);
  if ((int)blocks > g->partials_capacity) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  k_apply_melting<<<blocks, kBlock, 0, s>>>(*g);
  k_finish_sum<<<1, kFinishThreads, 0, s>>>(g->partials, (int)blocks, &g->control->discarded_heat);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_reduce_mass(const icy3d_grid* g, void* stream) {
  if (!ok_grid(g)) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  const size_t columns = (size_t)g->mx * g->my;
  if (!g->bodies || !columns) return 0;
  const int chunks = (int)((columns + kReduceThreads - 1) / kReduceThreads);
  if ((size_t)g->bodies * chunks * ICY3D_REDUCED_STRIDE > (size_t)g->partials_capacity) return ICY3D_ERR_ARGUMENT;
  k_reduce_mass<<<(unsigned)(g->bodies * chunks), kReduceThreads, 0, s>>>(*g, chunks);
  k_finish_reduced<<<(unsigned)g->bodies, 64, 0, s>>>(*g, chunks);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_sample_ice_temperature(const icy3d_grid* g, void* stream) {
  if (!ok_grid(g)) return ICY3D_ERR_ARGUMENT;
  k_sample_ice_temperature<<<icy_blocks(n_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_check_heat(const icy3d_grid* g, void* stream) {
  if (!ok_grid(g)) return ICY3D_ERR_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  size_t n = n_cells(*g) > n_material(*g) ? n_cells(*g) : n_material(*g);
  k_reset_thermal_invalid<<<1, 1, 0, s>>>(*g);
  k_check_heat<<<icy_blocks(n), kBlock, 0, s>>>(*g);
  ICY_LAUNCH_CHECK();
  return 0;
}
int icy3d_initialize_phase(const icy3d_grid* g, void* stream) {
  if (!ok_grid(g)) return ICY3D_ERR_ARGUMENT;
  k_initialize_phase<<<icy_blocks(n_cells(*g)), kBlock, 0, (hipStream_t)stream>>>(*g);
  ICY_LAUNCH_CHECK();
  return 0;
}

}  // extern "C"
