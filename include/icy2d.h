/* icy2d — C ABI of the MI355X (gfx950) 2D falling-and-melting ice step.
 *
 * Drop-in boundary for the reference's Python solver class
 * ``iceflow2d.simulator.IceFlow2D`` (iceflow2d/simulator.py:1826-4939) and
 * its thermal component ``MovingBodyThermal2D`` (:126-1823).  The reference
 * has no native FFI: its operator API is the Python class whose methods
 * each launch Taichi kernels.  Every entry point below replaces one such
 * kernel (cited per function) and is enqueued on the caller's HIP stream.
 * The Python host (``projecticy_amd.iceflow2d``) owns every device buffer;
 * this library never allocates memory and keeps no global state.
 *
 * Conventions
 *   - Cells n = i * ny + j (j fastest).  Populations are q-plane major:
 *     population q of cell n is ``f[q * N + n]`` (D2Q9 order of
 *     iceflow2d/lattice.py:8-62), FP32 or scaled FP16 elements (see
 *     half_populations).  Vectors are planes: ``u[c * N + n]``.
 *   - x-face fields have (nx + 1) * ny entries (face (i, j) at i * ny + j);
 *     y-face fields nx * (ny + 1) (face (i, j) at i * (ny + 1) + j).
 *   - Body fields are body_nx * body_ny, index bi * body_ny + bj.
 *   - Return codes: 0 success, >0 hipError_t of a failed launch,
 *     <0 ICY2D_ERR_*.  ``stream`` is a hipStream_t passed as void*.
 *   - Scalars the reference keeps in 0-d fields live in the device control
 *     block ``icy2d_control``; one device-to-host copy returns all of them.
 */
#ifndef ICY2D_H
#define ICY2D_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

enum { ICY2D_OK = 0, ICY2D_ERR_ARGUMENT = -1 };

/* Device control block: rigid state, reduction results and diagnostics.
 * Triples are (x, y, angular). */
typedef struct icy2d_control {
  float velocity[2], angle, omega, origin[2], support[4]; /* simulator.py:1950-2089 */
  int32_t projected, melt_status, wet_target, wet_target_max;
  float max_outflow;
  int32_t error_flags;        /* bit 0: negative water volume, bit 1: volume above the aperture capacity,
                               * bit 2: a heat or melt term outside the fixed-point range of the
                               * thermal scatters (body_heat, inject_acc), bit 3: a batch stated a
                               * population storage that is not this case's */
  double mass, inertia, local_com[2];
  double impulse[3];          /* hydrodynamic impulse x, y and torque */
  double melted[3];           /* cumulative melted body momentum */
  double carrier[3], correction[3];
  double before[3], provisional[3], after[3], body_before[3];
  double wet[4];              /* weight, first moment x, y, second moment */
  double water[3];            /* initial volume, current volume, projection derivative */
  double aperture[6];         /* volume, energy, base and full capacity, specific min, max */
  double targets[3];          /* reconstructed energy, cooling, heating capacity */
  double transfer[2];         /* volume and energy after the transfer */
  double correction_abs, boundary_power, boundary_heat_input;
  double unassigned[2], fallback[2], interval[2];
  double reduced[4];          /* mass, first moment x, y, origin inertia */
  double totals[4];           /* solid mass, water mass, body and water sensible energy */
  double error_values[2];     /* volume and capacity when error_flags was first set */
  /* LBM steps taken (advanced by the rigid integration, once per step); it
   * salts the stochastic FP16 rounding so that an unchanged value is not
   * rounded the same way every step.  No reference counterpart. */
  uint32_t rounding_step;
  /* Blocks of a fold with a one-thread tail that have finished; the last
   * one runs the tail and puts this back to 0.  No reference counterpart. */
  int32_t finish_ticket;
} icy2d_control;

typedef struct icy2d_grid {
  int32_t nx, ny, boundary, body_nx, body_ny, advection;
  int32_t left_kind, right_kind, bottom_kind, top_kind;
  /* lattice-unit constants */
  float rho_w, rho_a, nu_w, nu_a, gx, gy, sigma, width, mobility, smagorinsky, interface_tau;
  float cutoff, threshold, dx, expansion, t_ref, linear_damping, angular_damping;
  double initial_mass, initial_inertia;
  /* SI thermal constants */
  double t_melt, cp_w, cp_i, k_w, k_i, latent, rho_w_si, area, velocity_scale, cell_mass, t_air;
  double left_value, right_value, bottom_value, top_value;
  /* flow fields (FP32) */
  float *f, *fbuf, *h, *hbuf;     /* [9][N] */
  float *phi, *u, *a, *p, *moving; /* u, a: [2][N]; moving: sum of f_q, q != 0 */
  float *p_ref, *rho_ref;         /* [ny] */
  int8_t *solid, *prev_solid, *eligible;
  float* coverage;                /* world body solid fraction [N] */
  float* phase_ref;               /* phase each cell's hbuf is stored against [N] (bit 3 below) */
  /* thermal fields (FP64) */
  double *body_mass, *body_energy;
  /* The step's heat per body cell in fixed point (units of 2^-54 of
   * latent * cell_mass), so the exchange's scatter sums the same whatever
   * order its atomics land in. */
  int64_t* body_heat;
  double *melt_mass, *melt_sensible;
  int32_t* melt_target;           /* contributing water cell; after the injection, the cell fed */
  double *water_v, *water_e, *target_e;
  double *flux_ex, *flux_vx, *flux_ey, *flux_vy;
  /* [2][N] injected melt volume and energy in fixed point while the
   * injection runs (units of 2^-52 of area and of latent * cell_mass);
   * all zero between calls. */
  int64_t* inject_acc;
  double* partials;               /* reduction scratch: partials_capacity doubles */
  int32_t partials_capacity;
  /* Population storage, a bit mask: bit 0 set = f and fbuf hold FP16
   * population * population_scale, bit 1 set = h and hbuf do (a power-of-two
   * scale; FP32 arithmetic in registers); clear bits mean FP32; bit 2 rounds
   * FP16 stores stochastically (hash of value and index) instead of to
   * nearest; bit 3 stores each phase population as its deviation from
   * w_q * phi (h against phi, hbuf against phase_ref, the phase at the
   * collision).  No reference counterpart. */
  int32_t half_populations;
  float population_scale, population_inverse_scale;
  icy2d_control* control;
} icy2d_grid;

/* Geometry and rigid body ------------------------------------------------ */
int icy2d_body_fraction(const icy2d_grid* g, int only_if_projected, void* stream); /* simulator.py:2532-2537 */
int icy2d_commit_raster(const icy2d_grid* g, void* stream);                         /* :2539-2544 */
int icy2d_contact_support(const icy2d_grid* g, int reduce, int only_if_projected,
                          void* stream);                                              /* :3914-3971 */
int icy2d_integrate_rigid(const icy2d_grid* g, void* stream);                       /* :3973-4017 */
int icy2d_project_inside(const icy2d_grid* g, void* stream);                        /* :4019-4080 */
int icy2d_update_solid_mask(const icy2d_grid* g, int init, void* stream);           /* :2699-2727 */
int icy2d_reduce_mass_properties(const icy2d_grid* g, void* stream);                /* :3014-3044 */
int icy2d_apply_mass_properties(const icy2d_grid* g, int initialize, void* stream); /* :3046-3161 */

/* Initialisation ---------------------------------------------------------- */
int icy2d_initialize_fluid(const icy2d_grid* g, int water_width, int water_height, void* stream); /* :2595-2624 */
int icy2d_hydrostatic_equilibrium(const icy2d_grid* g, void* stream);                            /* :2664-2697 */
int icy2d_initialize_water_volume(const icy2d_grid* g, void* stream);                            /* :4125-4133 */
int icy2d_recover_initial_moments(const icy2d_grid* g, void* stream);                            /* :3833-3858 */
int icy2d_initialize_body_state(const icy2d_grid* g, double ice_temperature, void* stream);       /* :579-588 */
int icy2d_initialize_water_state(const icy2d_grid* g, double water_temperature, void* stream);    /* :589-617 */

/* Flow -------------------------------------------------------------------- */
/* Momentum collision with forces and Tao cut-link preparation (:3241-3552,
 * :4798-4866) fused with the phase collision (:3554-3697) of the same cell;
 * with_momentum = 0 runs the phase collision alone (the warm-up). */
int icy2d_collide(const icy2d_grid* g, int with_momentum, void* stream);
/* Cut-link preparation alone, applied in place to fbuf (the reference
 * tests' helper kernel around :4798-4866). */
int icy2d_prepare_cut_links(const icy2d_grid* g, void* stream);
/* mode 1: streaming (:3699-3738; :3740-3785 when phase_only) in pull form;
 * mode 2: the macroscopic update (:3787-3813; :3815-3825 when phase_only);
 * mode 3: both in one pass (the step). */
int icy2d_stream(const icy2d_grid* g, int phase_only, int mode, void* stream);
/* The step's collision and streaming in one pass (:3241-3738): the same
 * post-collision populations as icy2d_collide(g, 1), pushed to where
 * icy2d_stream's pull would fetch them, in fbuf and hbuf (non-fluid cells
 * carry their populations over).  The caller then swaps f/fbuf and h/hbuf
 * and runs icy2d_stream(g, 0, 2), the macroscopic update; together they
 * give icy2d_collide(g, 1) then icy2d_stream(g, 0, 3).  fbuf and hbuf hold
 * no post-collision populations afterwards (icy2d_collide writes those). */
int icy2d_collide_stream(const icy2d_grid* g, void* stream);
/* :3860-3897; the population sum is the one recorded by the last mode-2/3 update. */
int icy2d_update_pressure(const icy2d_grid* g, void* stream);
int icy2d_refill(const icy2d_grid* g, void* stream);            /* :3163-3236 */
int icy2d_measure_outflow(const icy2d_grid* g, void* stream);   /* :2303-2338 */

/* Volume projection (:4150-4492) ------------------------------------------ */
int icy2d_clip_phase(const icy2d_grid* g, double max_bulk_l1, void* stream);
int icy2d_seed_projection(const icy2d_grid* g, void* stream);
int icy2d_dilate_projection(const icy2d_grid* g, int primary_to_next, void* stream);
/* All `radius` sweeps of icy2d_dilate_projection (alternating planes from
 * primary_to_next = 1) in one launch; radius even and <= 16; the band ends
 * in the primary plane, as after the sweeps. */
int icy2d_dilate_band(const icy2d_grid* g, int radius, void* stream);
int icy2d_evaluate_projection(const icy2d_grid* g, double lambda, void* stream);
int icy2d_apply_projection(const icy2d_grid* g, double lambda, void* stream);
int icy2d_projection_residual_weight(const icy2d_grid* g, double residual, void* stream);
int icy2d_apply_projection_residual(const icy2d_grid* g, double residual, double weight, void* stream);

/* Melt-momentum closure (:2735-2986) -------------------------------------- */
int icy2d_snapshot_melt_momentum(const icy2d_grid* g, void* stream);
int icy2d_reduce_provisional_momentum(const icy2d_grid* g, void* stream);
int icy2d_melt_weight_geometry(const icy2d_grid* g, void* stream); /* status -> control->melt_status */
int icy2d_apply_melt_correction(const icy2d_grid* g, void* stream);
int icy2d_reduce_final_momentum(const icy2d_grid* g, void* stream);
int icy2d_local_melt_correction(const icy2d_grid* g, void* stream);
int icy2d_finish_melt_momentum(const icy2d_grid* g, void* stream);

/* Thermal (MovingBodyThermal2D) ------------------------------------------- */
/* Also checks the volume against the capacity (:522-540) into error_flags. */
int icy2d_measure_aperture(const icy2d_grid* g, void* stream);             /* :633-714, :1792-1822 */
/* The targets (:716-827) and, once they are folded, the transfer's
 * |energy correction| of :829-859 into correction_abs; then the transfer
 * itself (the rest of :829-859).  Call them in this order. */
int icy2d_build_aperture_targets(const icy2d_grid* g, void* stream);       /* :716-827 */
int icy2d_apply_aperture_transfer(const icy2d_grid* g, void* stream);      /* :829-859 */
int icy2d_finish_aperture_transfer(const icy2d_grid* g, void* stream);     /* :861-877 */
int icy2d_transfer_aperture(const icy2d_grid* g, void* stream);            /* apply, then finish, in one pass */
/* The three passes of one synchronisation (measure, build, transfer). */
int icy2d_synchronize_aperture(const icy2d_grid* g, void* stream);         /* :511-548 */
/* A step's fixed launches between its fused collide-stream (and the swap of
 * the buffers) and the advection: macroscopic update, pressure, rigid body,
 * contact and raster, labels, refill, outflow. */
int icy2d_after_stream(const icy2d_grid* g, void* stream);                 /* :2203-2210, :2233-2247 */
/* The control block into host memory (pinned, or the copy blocks), complete
 * on return. */
int icy2d_read_control(const icy2d_grid* g, icy2d_control* host, void* stream);
int icy2d_body_conduction(const icy2d_grid* g, double dt, void* stream);   /* :879-907 */
/* axis 0 resets the boundary power (:630-631) before adding its faces; axis 1 adds. */
int icy2d_conduction_flux(const icy2d_grid* g, int axis, void* stream);    /* :909-1010, :1063-1164 */
int icy2d_advection_flux(const icy2d_grid* g, int axis, void* stream);     /* :1012-1061, :1166-1215 */
int icy2d_update_water(const icy2d_grid* g, double dt, int volume, void* stream); /* :1217-1246 */
int icy2d_reset_interval_sources(const icy2d_grid* g, void* stream);         /* :624-627 */
int icy2d_accumulate_boundary_heat(const icy2d_grid* g, double dt, void* stream); /* :1248-1250 */
int icy2d_exchange_heat(const icy2d_grid* g, double dt, void* stream);     /* :1252-1372 */
int icy2d_phase_change(const icy2d_grid* g, void* stream);                 /* :1374-1406 */
int icy2d_freeze_eligibility(const icy2d_grid* g, void* stream);           /* :1408-1422 */
int icy2d_inject_melt(const icy2d_grid* g, void* stream);                  /* :1424-1475 */
int icy2d_measure_fallback(const icy2d_grid* g, void* stream);             /* :1477-1502 */
int icy2d_apply_fallback(const icy2d_grid* g, int use_free, void* stream); /* :1504-1540 */
int icy2d_reduce_totals(const icy2d_grid* g, void* stream);                /* :1565-1583 */

/* Binding check: sizeof(icy2d_grid), sizeof(icy2d_control). */
void icy2d_abi_sizes(int32_t* grid, int32_t* control);
/* The stochastic FP16 rounding of the population stores on its own: each of
 * `count` values is stored as FP16 (values[i] * scale), then `steps` times
 * read back, raised by `lift` and stored again with rounding step
 * first_step + s; out[i] receives the final stored value / scale.  No
 * reference counterpart: it checks that repeated sub-ulp updates survive in
 * expectation. */
int icy2d_probe_rounding(const float* values, int count, float lift, int steps, uint32_t first_step, float scale,
                         float* out, void* stream);

/* Ensembles ---------------------------------------------------------------
 * No counterpart in the reference, which runs one case per process.  An
 * icy2d_batch covers many independent cases of any sizes (each with its
 * own icy2d_grid, buffers and control block); every icy2d_batch_* entry
 * point does what the single-case entry point of the same name does, for
 * every case, in one launch per kernel: block b of a launch belongs to the
 * case c with first_block[shape][c] <= b < first_block[shape][c + 1].
 * A ``const double*`` argument is a device array with one value per case.
 * Blocks of cases with active[c] == 0 return at once (active may be NULL).
 * The per-case results equal the single-case entry points' bit for bit
 * when collide_threads and stream_threads are 256. */
#define ICY2D_SHAPES 13 /* cells, body, x faces, y faces, one, totals, cells/128, cells/512, band tiles,
                           collision tiles of 128, 256 and 512 threads, cells/1024 */
typedef struct icy2d_batch {
  int32_t ncases;
  int32_t collide_threads;      /* 128, 256 or 512 (chosen by the autotuner) */
  int32_t stream_threads;       /* 128, 256 or 512 */
  int32_t storage;              /* 1 + the half_populations that all cases share, 0: not stated (any mix); a case
                                 * with another storage is left alone by the kernels that move populations,
                                 * and the next reduction sets bit 3 of its error_flags */
  const icy2d_grid* grids;      /* device array of ncases grids */
  const int32_t* active;        /* device, ncases flags, or NULL for all */
  const int32_t* first_block;   /* device, ICY2D_SHAPES * (ncases + 1) prefix sums */
  int32_t total_blocks[ICY2D_SHAPES];
} icy2d_batch;

/* Host: fills first_block (ICY2D_SHAPES * (ncases + 1)) and total_blocks
 * (ICY2D_SHAPES) from host copies of the grids, and checks that every
 * case's partials hold its largest reduction. */
int icy2d_batch_plan(const icy2d_grid* grids, int32_t ncases, int32_t* first_block, int32_t* total_blocks);

int icy2d_batch_body_fraction(const icy2d_batch* b, int only_if_projected, void* stream);
int icy2d_batch_commit_raster(const icy2d_batch* b, void* stream);
int icy2d_batch_contact_support(const icy2d_batch* b, int reduce, int only_if_projected, void* stream);
int icy2d_batch_integrate_rigid(const icy2d_batch* b, void* stream);
int icy2d_batch_project_inside(const icy2d_batch* b, void* stream);
int icy2d_batch_update_solid_mask(const icy2d_batch* b, int init, void* stream);
int icy2d_batch_reduce_mass_properties(const icy2d_batch* b, void* stream);
int icy2d_batch_apply_mass_properties(const icy2d_batch* b, int initialize, void* stream);
int icy2d_batch_collide(const icy2d_batch* b, int with_momentum, void* stream);
int icy2d_batch_stream(const icy2d_batch* b, int phase_only, int mode, void* stream);
int icy2d_batch_collide_stream(const icy2d_batch* b, void* stream);
/* Swaps f/fbuf and h/hbuf in every case's device grid (after
 * icy2d_batch_collide_stream; the host swaps its own copies). */
int icy2d_batch_swap_flow_planes(const icy2d_batch* b, void* stream);
int icy2d_batch_update_pressure(const icy2d_batch* b, void* stream);
int icy2d_batch_refill(const icy2d_batch* b, void* stream);
int icy2d_batch_measure_outflow(const icy2d_batch* b, void* stream);
int icy2d_batch_clip_phase(const icy2d_batch* b, double max_bulk_l1, void* stream);
int icy2d_batch_seed_projection(const icy2d_batch* b, void* stream);
int icy2d_batch_dilate_projection(const icy2d_batch* b, int primary_to_next, void* stream);
int icy2d_batch_dilate_band(const icy2d_batch* b, int radius, void* stream);
int icy2d_batch_evaluate_projection(const icy2d_batch* b, const double* lambda, void* stream);
int icy2d_batch_apply_projection(const icy2d_batch* b, const double* lambda, void* stream);
int icy2d_batch_projection_residual_weight(const icy2d_batch* b, const double* residual, void* stream);
int icy2d_batch_apply_projection_residual(const icy2d_batch* b, const double* residual, const double* weight,
                                          void* stream);
int icy2d_batch_snapshot_melt_momentum(const icy2d_batch* b, void* stream);
int icy2d_batch_reduce_provisional_momentum(const icy2d_batch* b, void* stream);
int icy2d_batch_melt_weight_geometry(const icy2d_batch* b, void* stream);
int icy2d_batch_apply_melt_correction(const icy2d_batch* b, void* stream);
int icy2d_batch_reduce_final_momentum(const icy2d_batch* b, void* stream);
int icy2d_batch_local_melt_correction(const icy2d_batch* b, void* stream);
int icy2d_batch_finish_melt_momentum(const icy2d_batch* b, void* stream);
int icy2d_batch_measure_aperture(const icy2d_batch* b, void* stream);
int icy2d_batch_build_aperture_targets(const icy2d_batch* b, void* stream);
int icy2d_batch_apply_aperture_transfer(const icy2d_batch* b, void* stream);
int icy2d_batch_finish_aperture_transfer(const icy2d_batch* b, void* stream);
int icy2d_batch_transfer_aperture(const icy2d_batch* b, void* stream);
int icy2d_batch_body_conduction(const icy2d_batch* b, const double* dt, void* stream);
int icy2d_batch_conduction_flux(const icy2d_batch* b, int axis, void* stream);
int icy2d_batch_advection_flux(const icy2d_batch* b, int axis, void* stream);
int icy2d_batch_update_water(const icy2d_batch* b, const double* dt, int volume, void* stream);
int icy2d_batch_reset_interval_sources(const icy2d_batch* b, void* stream);
int icy2d_batch_accumulate_boundary_heat(const icy2d_batch* b, const double* dt, void* stream);
int icy2d_batch_exchange_heat(const icy2d_batch* b, const double* dt, void* stream);
int icy2d_batch_phase_change(const icy2d_batch* b, void* stream);
int icy2d_batch_freeze_eligibility(const icy2d_batch* b, void* stream);
int icy2d_batch_inject_melt(const icy2d_batch* b, void* stream);
int icy2d_batch_measure_fallback(const icy2d_batch* b, void* stream);
int icy2d_batch_apply_fallback(const icy2d_batch* b, int use_free, void* stream);
int icy2d_batch_reduce_totals(const icy2d_batch* b, void* stream);
void icy2d_batch_abi_size(int32_t* batch);

/* HIP graphs: capture the launches enqueued on ``stream`` between begin and
 * end into an executable graph (returned as an opaque handle), replay it, and
 * free it.  No counterpart in the reference (Taichi launches every kernel). */
int icy2d_graph_begin(void* stream);
int icy2d_graph_end(void* stream, void** graph);
int icy2d_graph_launch(void* graph, void* stream);
int icy2d_graph_destroy(void* graph);
/* Stream-ordered copy of ``bytes`` between host (pinned) and device memory in
 * either direction: the ensemble's per-case value uploads and control-block
 * readbacks, one call each instead of a framework copy.  No counterpart in
 * the reference. */
int icy2d_copy_async(void* dst, const void* src, size_t bytes, void* stream);

/* The hash of the sources, headers and compiler flags the library was built
 * from (no reference counterpart): the Python loaders refuse a library whose
 * hash is not the current sources'. */
const char* icy2d_source_hash(void);

#ifdef __cplusplus
}
#endif
#endif
