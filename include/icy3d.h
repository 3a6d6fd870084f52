/* icy3d — C ABI of the MI355X (gfx950) 3D ice/water coupled solver step.
 *
 * Drop-in boundary for the reference's Python solver class
 * ``iceflow3d.simulator.IceFlow3D`` (iceflow3d/simulator.py:40-947).  The
 * reference has no native FFI: its operator API is the Python class, whose
 * methods each launch one or more Taichi kernels.  Every entry point below
 * replaces one such method (cited per function) and is enqueued on the
 * caller's HIP stream.  The Python host (``projecticy_amd.iceflow3d``) owns
 * every device buffer (PyTorch-ROCm tensors); this library never allocates
 * persistent memory and keeps no global state.
 *
 * Conventions
 *   - Every device array is a plain pointer in ``icy3d_grid``.  Grid fields
 *     are structure-of-arrays planes: component c of cell n lives at
 *     ``ptr[c * N + n]`` with ``n = (i * ny + j) * nz + k`` (z fastest).
 *   - Return codes: 0 = success, >0 = hipError_t of a failed launch,
 *     <0 = ICY3D_ERR_* below.
 *   - ``stream`` is a ``hipStream_t`` passed as ``void*`` (null = default).
 */
#ifndef ICY3D_H
#define ICY3D_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define ICY3D_MAX_BODIES 32
#define ICY3D_STATE_STRIDE 21   /* origin[3], rotation[9] row-major, centre[3], v[3], omega[3] */
#define ICY3D_REDUCED_STRIDE 19 /* mass, first[3], second[9], lower[3], upper[3] */

enum {
  ICY3D_OK = 0,
  ICY3D_ERR_ARGUMENT = -1,
  ICY3D_ERR_LAUNCH = -2,
  ICY3D_ERR_TRAVEL = -4,   /* rigid displacement exceeds half a cell */
  ICY3D_ERR_CONTACT = -5,  /* contact projection did not converge */
  ICY3D_ERR_MANIFOLD = -6, /* wall contact manifold infeasible */
  ICY3D_ERR_SCRATCH = -7   /* grid larger than icy3d_flow_step_static's scratch */
};

/* Result of icy3d_rigid_step_device: status 0 or the first failing stage's
 * ICY3D_ERR_* code, the body that failed the travel check (-1 if none), the
 * contact residual (penetration, closing speed) and each body's coverage box
 * of the packed rows (as icy3d_rigid_coverage_boxes). */
typedef struct icy3d_rigid_result {
  int32_t status, failed_body;
  int32_t box_lo[ICY3D_MAX_BODIES][3], box_hi[ICY3D_MAX_BODIES][3];
  double residual[2];
} icy3d_rigid_result;

/* Device control block: every scalar the reference keeps in 0-d Taichi
 * fields plus the per-body loads and mass reductions, laid out so that one
 * small device-to-host copy returns all of them. */
typedef struct icy3d_control {
  int32_t invalid_index;   /* simulator.py:133 */
  int32_t thermal_invalid; /* thermal.py:51 */
  int32_t openings;        /* simulator.py:113 */
  int32_t covered;
  int32_t remaining;       /* simulator.py:114 */
  int32_t repair_count;
  int32_t refill_lower[3], refill_upper[3];
  int32_t geometry_lower[3], geometry_upper[3];
  /* Cells labelled unresolved (-3) after the last refill commit or before
   * it; a refresh of part of the grid must relabel them (lower > upper: none). */
  int32_t cavity_lower[3], cavity_upper[3];
  int32_t tank_count, ice_count; /* lengths of the boundary-cell lists */
  float maximum_speed, peak_speed, phase_clip_volume;
  float remap_energy, discarded_heat, max_outflow;
  float loads[ICY3D_MAX_BODIES][6];                     /* hydrodynamic force, torque */
  float reduced[ICY3D_MAX_BODIES][ICY3D_REDUCED_STRIDE]; /* simulator.py:738-776 */
  icy3d_rigid_result rigid;                             /* icy3d_rigid_step_device */
} icy3d_control;

typedef struct icy3d_grid {
  int32_t nx, ny, nz, boundary, bodies, mx, my, mz;
  int32_t water_width, water_height, floor_depth, check_stability;
  /* lattice-unit physics */
  float rho_air, gravity_y, sigma, width, mobility, normal_eps, bulk_rate;
  float threshold, max_velocity, expansion, water_t0, air_t, flux_limit;
  float rho_water_si, rho_air_si, mu_air, nu_scale;
  /* SI thermal constants */
  float tm, rho_cp, cp_ice, k_water, k_ice, latent, cell_volume, dx;
  float velocity_m_s, initial_cell_mass, mass_kg;
  /* grid fields */
  float *home, *home_post;             /* [10][N] HOME moments */
  float* h;                            /* [7][N] D3Q7 AA slots */
  float *phi, *pressure, *old_pressure, *coverage; /* [N] */
  float *u, *old_u, *force, *accel, *grad, *flux;  /* [3][N] */
  int8_t *id, *prev_id, *cov_id, *flag;            /* [N] */
  float *refill_state, *refill_next;               /* [5][N] */
  int8_t *refill_valid, *refill_next_valid;        /* [N] */
  float *ref_density, *ref_pressure;               /* [ny] */
  float* body;                                     /* [bodies][ICY3D_STATE_STRIDE] */
  int32_t* material_size;                          /* [bodies][3] */
  float* body_t0;                                  /* [bodies] */
  float *material_mass, *material_energy, *material_heat; /* [bodies][mx][my][mz] */
  float *water_volume, *water_energy, *target_energy, *sampled_ice_t; /* [N] */
  float *energy_flux, *volume_flux;                /* [3][N] */
  int32_t *tank_cells, *ice_cells;                 /* [N] flag-1 / flag-2 cell lists */
  float* partials;                                 /* [partials_capacity] block partial sums */
  /* [bodies][mx][my][mz] the exchange's heat in fixed point while
   * icy3d_exchange_heat runs (so the sum does not depend on the order of the
   * scatter); all zero between calls. */
  int64_t* heat_acc;
  /* Learned interface closure (no reference counterpart; both may be NULL):
   * exchange_gain[n] multiplies the heat a water cell requests from the ice
   * in the exchange (thermal.py:308-392); exchange_heat_out[n] accumulates
   * the heat the cell hands to the ice. */
  float *exchange_gain, *exchange_heat_out;        /* [N] */
  int32_t partials_capacity;
  /* Nonzero only on a call of icy3d_refresh_begin_boxes that is queued
   * before the host reads the flow step's stability scan: with
   * check_stability, that refresh's kernels then do nothing when the scan
   * found an invalid cell, so the caller can still raise with the geometry
   * untouched, as the reference checks before it advances the bodies
   * (simulator.py:835-839).  Every other call leaves it 0, and the scan
   * result it reads is only meaningful right after a recovery with the
   * scan on. */
  int32_t refresh_guard;
  icy3d_control* control;
} icy3d_grid;

/* Host rigid-body arrays (FP64, row-major, length body_count). */
typedef struct icy3d_rigid_arrays {
  int32_t body_count;
  double *origin, *q, *velocity, *omega, *com, *mass, *inertia, *lower, *upper;
} icy3d_rigid_arrays;

/* ---- initialisation (simulator.py:143-167) ---------------------------- */
int icy3d_initialize_material(const icy3d_grid* g, void* stream);       /* thermal.py:53-62 */
int icy3d_initialize_phase(const icy3d_grid* g, void* stream);          /* simulator.py:325-347 */
int icy3d_initialize_water_heat(const icy3d_grid* g, void* stream);     /* thermal.py:88-96 */
int icy3d_seed_populations(const icy3d_grid* g, void* stream);          /* simulator.py:385-395 */
/* Equilibrium from the current phase/velocity (optionally a constant
 * pressure) at every fluid cell: the reference tests' seed kernels
 * (test_numerics.py:37-46, test_mirror_gradient.py:49-55). */
int icy3d_set_equilibrium_all(const icy3d_grid* g, int parity, int with_phase, int use_constant_pressure,
                              float pressure, void* stream);
int icy3d_phase_warmup(const icy3d_grid* g, int steps, int* parity, void* stream); /* simulator.py:149-152 */

/* ---- flow step (simulator.py:823-842) ----------------------------------- */
int icy3d_classify(const icy3d_grid* g, const int32_t lo[3], const int32_t hi[3], void* stream); /* home.py:280-284 */
int icy3d_gradients(const icy3d_grid* g, const int32_t lo[3], const int32_t hi[3], void* stream); /* gradients.py:352-386 */
int icy3d_refill_gradients(const icy3d_grid* g, const int32_t lo[3], const int32_t hi[3], void* stream); /* gradients.py:402-431 */
/* icy3d_refill_gradients of the box [ref_lo, ref_hi) when every changed
 * cell lies in one of `count` boxes (lo/hi: [count][3], at most
 * ICY3D_MAX_BODIES + 1): classification within one cell and gradients within
 * the dependency radius (6, gradients.py:15-20) of those boxes, inside the
 * reference box, where the reference's pass can change them; the boundary
 * lists rebuilt once. */
int icy3d_refill_gradients_boxes(const icy3d_grid* g, int count, const int32_t* lo, const int32_t* hi,
                                 const int32_t ref_lo[3], const int32_t ref_hi[3], void* stream);
int icy3d_collide_phase(const icy3d_grid* g, int parity, int moving_walls, void* stream); /* phase.py:90-127 */
int icy3d_recover_phase(const icy3d_grid* g, int parity, int recover_flow, void* stream); /* phase.py:129-161 */
int icy3d_recover_pressure(const icy3d_grid* g, void* stream);          /* home.py:347-353 */
int icy3d_scan_stability(const icy3d_grid* g, void* stream);            /* simulator.py:796-805 */
int icy3d_forces(const icy3d_grid* g, int with_flux, int moment_pressure, void* stream); /* simulator.py:521-557 */
int icy3d_collide_momentum(const icy3d_grid* g, void* stream);          /* home.py:199-211 */
int icy3d_stream_home(const icy3d_grid* g, void* stream);               /* home.py:256-345 */
/* icy3d_collide_momentum then icy3d_stream_home in one pass (home.py:199-211,
 * :256-345): each cell is collided as the stream stages it, so the
 * post-collision moments never reach memory.  Reads home, writes the
 * streamed moments to home_post: on return the caller swaps the home and
 * home_post pointers of its grid (home then holds the values of the two
 * separate calls, up to FMA contraction; old_velocity and old_pressure, which
 * the reference writes but reads only inside this pass, are not written;
 * home_post then holds the pre-stream moments). */
int icy3d_collide_stream_home(const icy3d_grid* g, void* stream);
/* Device part of IceFlow3D.step up to the stability check
 * (simulator.py:826-838): [gradients] collide_phase, forces, fused HOME
 * collide-stream with the loads zeroed, recover+scan, gradients.  The
 * collide-stream leaves the new moments in home_post, and the launches
 * after it in the same call use them there: on return the caller swaps the
 * home and home_post pointers of its grid, as after
 * icy3d_collide_stream_home. */
/* classify != 0 recomputes the link classes and boundary lists first
 * (needed after any external edit of the labels). */
int icy3d_flow_step(const icy3d_grid* g, int parity, int refresh_gradients, int classify, void* stream);
/* icy3d_flow_step in two parts (same launches, same results): _begin runs up
 * to the HOME collide-stream, after which the body loads in the control
 * block are final; the caller then swaps home and home_post, and _end runs
 * recovery, the stability scan and the gradients.  A host that copies the
 * loads out between the two can integrate the rigid bodies while _end
 * runs. */
int icy3d_flow_step_begin(const icy3d_grid* g, int parity, int refresh_gradients, int classify, void* stream);
int icy3d_flow_step_end(const icy3d_grid* g, int parity, void* stream);
/* _end without the gradient pass, for a caller that refreshes the geometry
 * next and runs that pass after it (icy3d_refresh_end_boxes with
 * full_gradients): outside the reference's refresh box nothing within the
 * gradients' dependency radius changes in between, so one pass after the
 * refresh gives the field the reference has after its refresh. */
int icy3d_flow_step_recover(const icy3d_grid* g, int parity, void* stream);
/* icy3d_flow_step with no device memory of the caller's beyond the grid's
 * fields: no counterpart in the reference; for callers that cannot allocate
 * (code under HIP graph capture, serving loops).  The block partial sums
 * that the step's kernels keep in g->partials go instead to a static
 * device array of the library (768 KiB per GPU, held until the process
 * ends); g->partials and g->partials_capacity are not used.  Grids of more
 * than icy3d_flow_step_static_max_cells() cells (2^24) return
 * ICY3D_ERR_SCRATCH.  No allocation, free or allocating library call is
 * made.  The array is shared by every call on one GPU and keeps the last
 * call's contents (each kernel writes the slots it reads first), so calls
 * that overlap on one GPU, on different streams, race. */
int icy3d_flow_step_static(const icy3d_grid* g, int parity, int refresh_gradients, int classify, void* stream);
int64_t icy3d_flow_step_static_max_cells(void);

/* Kernel-group timing of the fused flow step with HIP events on the same
 * stream (no reference counterpart; the reference measures with Taichi's
 * kernel profiler, iceflow3d/benchmarks/profile_complete_step.py:63-69).
 * Groups: 0 phase collide, 1 classify+forces, 2 HOME collide-stream,
 * 3 phase recovery+stability, 4 gradients. */
#define ICY3D_PROFILE_GROUPS 5
typedef struct icy3d_profile icy3d_profile;
int icy3d_profile_create(icy3d_profile** out);
int icy3d_profile_destroy(icy3d_profile* profile);
int icy3d_flow_step_profiled(const icy3d_grid* g, int parity, int refresh_gradients, int classify,
                             icy3d_profile* profile, void* stream);
int icy3d_profile_collect(icy3d_profile* profile); /* waits for the last step; accumulates */
int icy3d_profile_read(const icy3d_profile* profile, double* total_ms, int64_t* count);
int icy3d_repair_phase_layout(const icy3d_grid* g, int parity, const int32_t lo[3], const int32_t hi[3],
                              void* stream); /* phase.py:163-184 */
/* icy3d_repair_phase_layout over `count` disjoint boxes ([count][3]). */
int icy3d_repair_phase_layout_boxes(const icy3d_grid* g, int parity, int count, const int32_t* lo, const int32_t* hi,
                                    void* stream);
int icy3d_export_phase(const icy3d_grid* g, int parity, float* out, void* stream); /* phase.py:186-191 */

/* ---- geometry and refill (simulator.py:288-323, 589-736) ---------------- */
/* Box arguments (lo inclusive, hi exclusive) restrict a geometry pass to the
 * region where ice can have moved; NULL means the whole grid. */
int icy3d_rasterize(const icy3d_grid* g, const int32_t lo[3], const int32_t hi[3], void* stream);
int icy3d_find_refill_changes(const icy3d_grid* g, const int32_t lo[3], const int32_t hi[3], void* stream);
int icy3d_seed_refill_region(const icy3d_grid* g, const int32_t lo[3], const int32_t hi[3], void* stream);
int icy3d_propagate_refill(const icy3d_grid* g, const int32_t lo[3], const int32_t hi[3], void* stream);
int icy3d_accept_refill(const icy3d_grid* g, const int32_t lo[3], const int32_t hi[3], void* stream);
int icy3d_commit_refill(const icy3d_grid* g, const int32_t lo[3], const int32_t hi[3], void* stream);
/* The same passes over `count` disjoint boxes (lo/hi: [count][3], at most
 * ICY3D_MAX_BODIES + 1; simulator.py:708-736 runs them over the whole grid,
 * and only cells inside the boxes can change).  A box list lets a refresh
 * cover each body's region instead of one box spanning every body.
 * commit_refill also writes cavity_lower/cavity_upper. */
int icy3d_rasterize_boxes(const icy3d_grid* g, int count, const int32_t* lo, const int32_t* hi, void* stream);
int icy3d_find_refill_changes_boxes(const icy3d_grid* g, int count, const int32_t* lo, const int32_t* hi,
                                    void* stream);
int icy3d_commit_refill_boxes(const icy3d_grid* g, int count, const int32_t* lo, const int32_t* hi, void* stream);
/* simulator.py:708-736 over such boxes in two calls around the host's refill
 * loop.  _begin: one reset of the geometry and refill bounds, the refill
 * counters and the cavity bounds, then rasterize, the phase-layout repair
 * (parity odd; boxes extended one cell down) and find_refill_changes.
 * _end: commit_refill (its cavity bounds reset by _begin), then
 * icy3d_refill_gradients_boxes of [ref_lo, ref_hi) unless ref_lo is NULL;
 * with full_gradients, the same class refresh and one gradient pass over the
 * whole grid (after icy3d_flow_step_recover). */
int icy3d_refresh_begin_boxes(const icy3d_grid* g, int parity, int count, const int32_t* lo, const int32_t* hi,
                              void* stream);
int icy3d_refresh_end_boxes(const icy3d_grid* g, int count, const int32_t* lo, const int32_t* hi,
                            const int32_t ref_lo[3], const int32_t ref_hi[3], int full_gradients, void* stream);
/* Rebuild the tank (flag 1) and ice (flag 2) cell lists from the flags. */
int icy3d_build_boundary_lists(const icy3d_grid* g, void* stream);
int icy3d_project_refill(const icy3d_grid* g, int parity, const int32_t lo[3], const int32_t hi[3], void* stream);

/* ---- thermal (thermal.py:98-440) ---------------------------------------- */
int icy3d_synchronize_water(const icy3d_grid* g, void* stream);
/* icy3d_synchronize_water (thermal.py:98-127) in one pass: the remapped water
 * volume and energy go to volume_out / energy_out ([N] each, distinct from
 * the grid's planes); on return the caller swaps them with water_volume /
 * water_energy.  target_energy is not written. */
int icy3d_synchronize_water_into(const icy3d_grid* g, float* volume_out, float* energy_out, void* stream);
int icy3d_thermal_fluxes(const icy3d_grid* g, int advect, void* stream);
int icy3d_apply_thermal_fluxes(const icy3d_grid* g, float dt, int advect, void* stream);
/* icy3d_thermal_fluxes then icy3d_apply_thermal_fluxes with advect = 1
 * (thermal.py:133-184) in one pass that stores no flux planes: the updated
 * water volume and energy go to volume_out / energy_out ([N] each, distinct
 * from the grid's planes); on return the caller swaps them with
 * water_volume / water_energy.  energy_flux and volume_flux are not written. */
int icy3d_advect_water(const icy3d_grid* g, float dt, float* volume_out, float* energy_out, void* stream);
/* icy3d_synchronize_water, one advection substep of dt (icy3d_thermal_fluxes
 * and icy3d_apply_thermal_fluxes with advect = 1) and icy3d_synchronize_water
 * again (thermal.py:98-184) in one pass: the remapped water goes to
 * volume_out / energy_out ([N] each, distinct from the grid's planes), which
 * the caller swaps with water_volume / water_energy on return; the remap
 * energy takes both remaps' sums.  No intermediate plane is written. */
int icy3d_remap_advect_remap(const icy3d_grid* g, float dt, float* volume_out, float* energy_out, void* stream);
/* icy3d_thermal_fluxes then icy3d_apply_thermal_fluxes with advect = 0
 * (thermal.py:133-184, the conduction update) in one pass: the updated water
 * energy goes to energy_out ([N], distinct from water_energy), which the
 * caller swaps with water_energy on return; no flux plane is written. */
int icy3d_conduct_water(const icy3d_grid* g, float dt, float* energy_out, void* stream);
int icy3d_measure_outflow(const icy3d_grid* g, void* stream);
int icy3d_body_conduction(const icy3d_grid* g, float dt, void* stream);
int icy3d_exchange_heat(const icy3d_grid* g, float dt, const int32_t lo[3], const int32_t hi[3], void* stream);
int icy3d_apply_melting(const icy3d_grid* g, void* stream);
int icy3d_reduce_mass(const icy3d_grid* g, void* stream);              /* simulator.py:738-776 */
int icy3d_sample_ice_temperature(const icy3d_grid* g, void* stream);
int icy3d_check_heat(const icy3d_grid* g, void* stream);

/* ---- diagnostics and probes (the reference tests' probe kernels) -------- */
int icy3d_capillary_stress(const icy3d_grid* g, float* out, void* stream);  /* [9][N], gradients.py:147-158 */
int icy3d_generic_forces(const icy3d_grid* g, float* out, void* stream);    /* [6][N], test_home_phase.py:69-78 */
int icy3d_write_gradient_all(const icy3d_grid* g, void* stream);            /* test_home_phase.py:81-84 */
int icy3d_probe_home(const float* data, int rows, float* populations, float* collided, void* stream);
int icy3d_probe_phase(const float* data, int rows, float mobility, float width, float* out, void* stream);
int icy3d_probe_viscosity(const float* phi, int n_phi, const float* temps, int n_t, float rho_w, float rho_a,
                          float mu_air, float* out, void* stream);
int icy3d_probe_stress_velocity(const icy3d_grid* g, const int32_t cell[3], const int32_t c[3], float* out,
                                void* stream); /* simulator.py:559-587 */
int icy3d_probe_mirror(const icy3d_grid* g, const int32_t cell[3], const int32_t c[3], float* out,
                       void* stream); /* gradients.py:60-113 */

/* ---- host rigid bodies (rigid.py:121-404), FP64 ------------------------- */
int icy3d_rigid_integrate(const icy3d_rigid_arrays* s, const float* loads, const double gravity[3],
                          double linear_damping, double angular_damping, int* failed_body);
int icy3d_rigid_resolve_contacts(const icy3d_rigid_arrays* s, const int shape[3], int boundary, int iterations,
                                 double residual[2]);
int icy3d_rigid_contact_residuals(const icy3d_rigid_arrays* s, const int shape[3], int boundary,
                                  double residual[2]);
int icy3d_rigid_update_mass(const icy3d_rigid_arrays* s, const float* reduced);
int icy3d_rigid_pack_state(const icy3d_rigid_arrays* s, float* out);
/* Cells whose coverage can be nonzero for packed rows `state` (simulator.py:
 * 288-323's bounding box: the rotated material box plus its trilinear
 * support, a margin of one cell below and two above), clamped to the grid;
 * sizes: [body_count][3] material cells.  lo = shape, hi = 0 without bodies. */
int icy3d_rigid_coverage_box(const float* state, int body_count, const int32_t* sizes, const int shape[3],
                             int32_t lo[3], int32_t hi[3]);
/* The same box for each body separately (lo/hi: [body_count][3]). */
int icy3d_rigid_coverage_boxes(const float* state, int body_count, const int32_t* sizes, const int shape[3],
                               int32_t* lo, int32_t* hi);
/* Merge `count` boxes ([count][3], lo inclusive, hi exclusive; empty boxes
 * dropped) into disjoint ones: any two whose copies extended one cell down
 * on every axis overlap are replaced by their bounding box, until none do.
 * Writes at most `capacity` boxes to out_lo/out_hi and their number to
 * *out_count (no reference counterpart: the reference refreshes the whole
 * grid, simulator.py:708-736). */
int icy3d_merge_boxes(int count, const int32_t* lo, const int32_t* hi, int capacity, int32_t* out_lo,
                      int32_t* out_hi, int* out_count);
/* One rigid update of the flow loop in a single host call (rigid.py:178-347
 * then simulator.py:259-286): icy3d_rigid_integrate, _resolve_contacts,
 * _pack_state into `state` and _coverage_box of the packed rows.  Returns the
 * first failing stage's code (failed_body / residual as those stages set). */
int icy3d_rigid_step(const icy3d_rigid_arrays* s, const float* loads, const double gravity[3], double linear_damping,
                     double angular_damping, const int shape[3], int boundary, int iterations, const int32_t* sizes,
                     float* state, int32_t box_lo[3], int32_t box_hi[3], int* failed_body, double residual[2]);

/* icy3d_rigid_step on the device (rigid.py:178-347 then simulator.py:259-286;
 * the reference keeps this on the host in NumPy FP64): the same FP64
 * integration, contact projection, packing and per-body coverage boxes, run
 * by one lane of one wavefront on `stream`, so the loads and the state never
 * cross PCIe.  Every pointer except `s` itself, `gravity` and `shape` is
 * device memory: the arrays of *s, loads [body_count][6], sizes
 * [body_count][3], state [body_count][ICY3D_STATE_STRIDE] and `result`
 * (for instance &control->rigid, so the control block's copy carries it).
 * Returns a launch error; the solver's own status is result->status. */
int icy3d_rigid_step_device(const icy3d_rigid_arrays* s, const float* loads, const double gravity[3],
                            double linear_damping, double angular_damping, const int shape[3], int boundary,
                            int iterations, const int32_t* sizes, float* state, icy3d_rigid_result* result,
                            void* stream);

/* Stream-ordered copy between any two of device, pinned host and host
 * memory (hipMemcpyAsync); no reference counterpart: the host's per-step
 * upload of body rows without a framework tensor copy. */
int icy3d_copy_async(void* dst, const void* src, size_t bytes, void* stream);

/* The control block into host memory (pinned, or the copy blocks), complete
 * on return. */
int icy3d_read_control(const icy3d_grid* g, icy3d_control* host, void* stream);
/* Size of the structs this library was built with (ABI check). */
int icy3d_abi_sizes(int32_t* grid_bytes, int32_t* control_bytes);

/* The hash of the sources, headers and compiler flags the library was built
 * from (no reference counterpart): the Python loaders refuse a library whose
 * hash is not the current sources'. */
const char* icy3d_source_hash(void);

#ifdef __cplusplus
}
#endif

#endif /* ICY3D_H */
