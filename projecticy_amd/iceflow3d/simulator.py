"""``IceFlow3D``: the reference's 3D coupled solver API on MI355X.

Drop-in for ``iceflow3d.simulator.IceFlow3D`` (iceflow3d/simulator.py:40-947):
same constructor, ``step(n)``, ``flush_thermal()``, ``snapshot()``,
``diagnostics()``, ``check_stability()``, public field names and exception
behaviour.  State lives in PyTorch-ROCm tensors on ``cuda:0`` in GPU-friendly
layouts; every kernel is a hand-written gfx950 HIP kernel reached through the
C ABI of include/icy3d.h.  Rigid bodies integrate on the host in FP64 native
code.  There is no CPU path: without a HIP device the constructor raises.
"""

import ctypes
import math

import numpy as np
import torch

from .. import _native
from .._native import Control, Grid, check, int3, lib
from .config import IceFlowConfig, LatticeScales, integer
from .fields import ControlScalar, DerivedField, DeviceField, HostScalar
from .rigid import _RIGID_FIELDS, RigidBodies, _contact_error, _RigidArrays
from .viscosity import air_dynamic_viscosity_pa_s


def _require_device():
    if not torch.cuda.is_available():
        raise RuntimeError("IceFlow3D requires a HIP (ROCm) GPU; none is available")
    return torch.device("cuda", torch.cuda.current_device())


class IceFlow3D:
    """HOME D3Q27 momentum, D3Q7 AA phase, moving and melting ice (3D)."""

    def __init__(self, config: IceFlowConfig, *, rigid_on_device=False):
        """``rigid_on_device`` (no reference counterpart): integrate the
        bodies and resolve their contacts on the GPU in FP64
        (``icy3d_rigid_step_device``) instead of on the host, so the loads
        and the body state stay in device memory."""
        if not isinstance(config, IceFlowConfig):
            raise TypeError("config must be IceFlowConfig")
        if config.conserve_phase_volume:
            raise ValueError(
                "global phase-volume correction is commented out; set conserve_phase_volume=False"
            )
        if config.gas_state_repair:
            raise ValueError("HOME does not use gas-state repair")
        if len(config.bodies) > _native.MAX_BODIES:
            raise ValueError(f"at most {_native.MAX_BODIES} ice bodies are supported")
        self.device = _require_device()
        self._lib = lib()
        self._functions = {}
        self._step_stream = None
        self.config, self.scales = config, LatticeScales.from_iceflow_config(config)
        self.shape = (config.nx, config.ny, config.nz)
        self.nx, self.ny, self.nz = self.shape
        self.steps = 0
        self.body_count = len(config.bodies)
        self.rho_air = config.rho_air / config.rho_water
        self.gravity = tuple(np.array(config.gravity) * self.scales.dt_s**2 / self.scales.dx_m)
        dx = self.scales.dx_m
        self.sigma = config.surface_tension_n_m * self.scales.dt_s**2 / (config.rho_water * dx**3)
        self.mu_air = air_dynamic_viscosity_pa_s(config.thermal.initial_air_temperature_c)
        self.nu_air = self.mu_air / config.rho_air * self.scales.dt_s / dx**2
        props = config.thermal.properties
        self.dx = dx
        self.cell_volume = dx**3
        self.initial_cell_mass = config.rho_ice * self.cell_volume
        self.rho_cp = config.rho_water * props.specific_heat_water_j_kg_k
        self.tm = props.melting_temperature_c
        self.cp_ice = props.specific_heat_ice_j_kg_k
        self.k_water, self.k_ice = props.conductivity_water_w_m_k, props.conductivity_ice_w_m_k
        self.latent = props.latent_heat_j_kg
        self.pending_cells = 0
        self._parity = 0
        self._allocate()
        self.rigid = RigidBodies(self)
        self._call("initialize_material")
        self.rigid.update_mass()
        self._rasterize()
        # The first rasterisation recorded labels of a zeroed grid as the
        # previous labels; the first refresh must therefore cover the grid.
        self._raster_full = True
        self._call("initialize_phase")
        if config.phase_warmup_steps:
            parity = ctypes.c_int32(self._parity)
            check(self._lib.icy3d_phase_warmup(self._gp, config.phase_warmup_steps, ctypes.byref(parity),
                                               self._stream()), "phase warm-up")
            self._parity = parity.value
        self._call("initialize_water_heat")
        self._build_reference()
        self._gradients()
        self._forces(False)
        self._seed_populations()
        self.initial_ice_mass_kg = self.rigid.mass.copy() * self.scales.mass_kg
        self.initial_water_volume_m3 = float(self.water_volume.to_numpy().sum(dtype=float))
        self.initial_phase_volume_m3 = float(self.water_phase.to_numpy().sum(dtype=np.float64) * self.cell_volume)
        self._thermal_pending = 0
        self._gradient_cache_valid = True
        self._rigid_dev = None
        if rigid_on_device:
            self._enable_device_rigid()

    # ------------------------------------------------------------------ setup
    def _allocate(self):
        cfg, th, props = self.config, self.config.thermal, self.config.thermal.properties
        dev, f32, i8 = self.device, torch.float32, torch.int8
        N = self.shape
        B = self.body_count
        sizes = np.array([b.size_cells for b in cfg.bodies], dtype=np.int32)
        mshape = (B, *map(int, sizes.max(axis=0)))
        zeros = lambda *s, dtype=f32: torch.zeros(s, dtype=dtype, device=dev)  # noqa: E731
        self._t = t = {
            "home": zeros(10, *N), "home_post": zeros(10, *N), "h": zeros(7, *N),
            "phi": zeros(*N), "pressure": zeros(*N), "old_pressure": zeros(*N), "coverage": zeros(*N),
            "u": zeros(3, *N), "old_u": zeros(3, *N), "force": zeros(3, *N), "accel": zeros(3, *N),
            "grad": zeros(3, *N), "flux": zeros(3, *N),
            "id": zeros(*N, dtype=i8), "prev_id": zeros(*N, dtype=i8), "cov_id": zeros(*N, dtype=i8),
            "flag": zeros(*N, dtype=i8),
            "refill_state": zeros(5, *N), "refill_next": zeros(5, *N),
            "refill_valid": zeros(*N, dtype=i8), "refill_next_valid": zeros(*N, dtype=i8),
            "ref_density": zeros(self.ny), "ref_pressure": zeros(self.ny),
            "body": zeros(B, _native.STATE_STRIDE),
            "material_size": torch.from_numpy(sizes).to(dev),
            "body_t0": torch.tensor(
                [th.initial_ice_temperature_c if b.temperature_c is None else b.temperature_c for b in cfg.bodies],
                dtype=f32, device=dev),
            "material_mass": zeros(*mshape), "material_energy": zeros(*mshape), "material_heat": zeros(*mshape),
            "water_volume": zeros(*N), "water_energy": zeros(*N), "target_energy": zeros(*N),
            "water_volume_next": zeros(*N), "water_energy_next": zeros(*N),
            "sampled_ice_t": zeros(*N), "energy_flux": zeros(3, *N), "volume_flux": zeros(3, *N),
            "tank_cells": zeros(math.prod(N), dtype=torch.int32),
            "ice_cells": zeros(math.prod(N), dtype=torch.int32),
            "partials": zeros(self._partials_capacity(mshape)), "heat_acc": zeros(*mshape, dtype=torch.int64),
            "control": torch.zeros(ctypes.sizeof(Control), dtype=torch.uint8, device=dev),
        }
        self._control_host = torch.zeros(ctypes.sizeof(Control), dtype=torch.uint8).pin_memory()
        self._loads_host = torch.zeros(ctypes.sizeof(Control), dtype=torch.uint8).pin_memory()
        self._control_alias = Control.from_buffer(self._control_host.numpy())
        self._loads_ready = torch.cuda.Event()
        self._loads_control = Control.from_buffer(self._loads_host.numpy())
        self._upload_staging = torch.zeros((B, _native.STATE_STRIDE), dtype=torch.float32).pin_memory()
        self._upload_staging_view = self._upload_staging.numpy()
        self._upload_done = torch.cuda.Event()
        # The per-body loads inside the pinned copy of the control block.
        loads0 = Control.loads.offset
        self._loads_view = self._loads_host.numpy()[loads0 : loads0 + 24 * _native.MAX_BODIES].view(
            np.float32).reshape(_native.MAX_BODIES, 6)[:B]
        g = Grid()
        g.nx, g.ny, g.nz = self.shape
        g.boundary, g.bodies = cfg.boundary_cells, B
        g.mx, g.my, g.mz = mshape[1:]
        g.water_width, g.water_height = cfg.water_width, cfg.water_height
        g.floor_depth, g.check_stability = cfg.floor_water_depth_cells, int(cfg.check_stability)
        g.rho_air, g.gravity_y, g.sigma = self.rho_air, self.gravity[1], self.sigma
        g.width, g.mobility = cfg.interface_width, cfg.mobility
        g.normal_eps, g.bulk_rate = cfg.phase_normal_epsilon, cfg.cm_acoustic_relaxation_rate
        g.threshold, g.max_velocity = th.solid_liquid_threshold, cfg.maximum_velocity_lattice
        g.expansion, g.water_t0 = th.thermal_expansion_water_1_k, th.initial_water_temperature_c
        g.air_t, g.flux_limit = th.initial_air_temperature_c, cfg.phase_flux_acceleration_limit
        g.rho_water_si, g.rho_air_si, g.mu_air = cfg.rho_water, cfg.rho_air, self.mu_air
        g.nu_scale = self.scales.dt_s / self.dx**2
        g.tm, g.rho_cp, g.cp_ice = self.tm, self.rho_cp, self.cp_ice
        g.k_water, g.k_ice, g.latent = self.k_water, self.k_ice, self.latent
        g.cell_volume, g.dx = self.cell_volume, self.dx
        g.velocity_m_s, g.initial_cell_mass, g.mass_kg = self.scales.velocity_m_s, self.initial_cell_mass, self.scales.mass_kg
        for name in _native.GRID_POINTERS:
            setattr(g, name, t[name].data_ptr())
        g.partials_capacity = t["partials"].numel()
        g.control = t["control"].data_ptr()
        # Labels, link classes and boundary lists are rebuilt over the whole
        # grid until the first geometry refresh establishes the ice region.
        self._flags_valid = False
        self._raster_full = True
        self._box_history = None
        self._full_boxes = (np.zeros((1, 3), np.int32), np.array([self.shape], np.int32))
        self._merged = (np.zeros((_native.MAX_BODIES + 1, 3), np.int32), np.zeros((_native.MAX_BODIES + 1, 3), np.int32))
        cavity0 = Control.cavity_lower.offset
        self._cavity_view = self._loads_host.numpy()[cavity0 : cavity0 + 24].view(np.int32)
        self._grid = g
        self._gp = ctypes.pointer(g)
        self._body_state = np.zeros((B, _native.STATE_STRIDE), np.float32)
        self._control_offsets()
        self._make_fields()
        # Stability limits start at "nothing invalid".
        control = self._read_control()
        control.invalid_index = math.prod(self.shape)
        self._write_control(control)

    def _partials_capacity(self, mshape):
        """Block partial sums: three words per 256-cell block (the recovery's
        clip sum, maximum speed and first invalid cell; the list compaction
        needs two per 4096 cells), one float per material block, and the
        boundary-stream load slots."""
        blocks = lambda count: (count + 255) // 256  # noqa: E731
        return max(3 * blocks(math.prod(self.shape)), blocks(math.prod(mshape)),
                   _native.LIST_BLOCKS * _native.MAX_BODIES * 6)

    def _geometry_edited(self):
        """External edits of labels, coverage, material or body state: the
        next rasterisation covers the grid and link classes are rebuilt."""
        self._raster_full = True
        self._flags_valid = False

    # gradients.py:15-20: every phase and coverage dependency of a gradient
    # lies within this many cells.
    GRADIENT_DEPENDENCY_RADIUS = 6

    def _coverage_boxes(self, state=None):
        """Per body, the cells whose coverage can be nonzero for FP32 rows
        ``state`` (the uploaded rows by default): int32 (lo, hi), [B, 3]."""
        state = np.ascontiguousarray(self._body_state if state is None else state, dtype=np.float32)
        B = self.body_count
        lo, hi = np.zeros((B, 3), np.int32), np.zeros((B, 3), np.int32)
        sizes = self.rigid._step_arguments()["sizes"]
        check(self._lib.icy3d_rigid_coverage_boxes(state.ctypes.data, B, sizes.ctypes.data, int3(self.shape),
                                                   lo.ctypes.data, hi.ctypes.data), "coverage boxes")
        return lo, hi

    @staticmethod
    def _cavity_box(lower, upper):
        """(lo, hi) of the cells the last refill commit left unresolved or
        resolved (inclusive bounds from the device), or None."""
        lo, hi = np.array(lower, np.int32).reshape(1, 3), np.array(upper, np.int32).reshape(1, 3) + 1
        return None if np.any(hi <= lo) else (lo, hi)

    def _raster_boxes(self, current=None, cavity=()):
        """Disjoint boxes (int32 lo, hi: [count, 3]) holding every cell whose
        label, coverage or previous label can change in this refresh: each
        body's box for the uploaded rows and for the rows of the two
        refreshes before (the last refresh relabelled cells only inside its
        own boxes), plus ``cavity`` (the last commit's unresolved cells;
        read from the device when not given).  The reference refreshes the
        whole grid; every other cell keeps its label, coverage and previous
        label there.  The whole grid on the first refresh and after edits."""
        if current is None:
            current = self._coverage_boxes()
        history = self._box_history
        self._box_history = (current, None if history is None else history[0])
        if self._raster_full or history is None:
            self._raster_full = False
            return self._full_boxes
        if cavity == ():
            control = self._read_control()
            cavity = self._cavity_box(control.cavity_lower, control.cavity_upper)
        parts = [current, history[0]] + [part for part in (history[1], cavity) if part is not None]
        lo = np.ascontiguousarray(np.concatenate([part[0] for part in parts]), dtype=np.int32)
        hi = np.ascontiguousarray(np.concatenate([part[1] for part in parts]), dtype=np.int32)
        out_lo, out_hi = self._merged
        count = ctypes.c_int(0)
        code = self._lib.icy3d_merge_boxes(len(lo), lo.ctypes.data, hi.ctypes.data, len(out_lo), out_lo.ctypes.data,
                                           out_hi.ctypes.data, ctypes.byref(count))
        if code == 0:
            return out_lo[: count.value].copy(), out_hi[: count.value].copy()
        # More disjoint regions than one launch takes: their bounding box.
        keep = np.all(hi > lo, axis=1)
        return lo[keep].min(axis=0, keepdims=True), hi[keep].max(axis=0, keepdims=True)

    def _control_offsets(self):
        floats = self._t["control"].view(torch.float32)
        loads0 = Control.loads.offset // 4
        reduced0 = Control.reduced.offset // 4
        B = self.body_count
        self._loads = floats[loads0 : loads0 + 6 * _native.MAX_BODIES].view(_native.MAX_BODIES, 6)[:B]
        self._reduced = floats[reduced0 : reduced0 + _native.REDUCED_STRIDE * _native.MAX_BODIES].view(
            _native.MAX_BODIES, _native.REDUCED_STRIDE)[:B]

    def _make_fields(self):
        t = self._t
        vec = lambda name: DeviceField(t[name], components=3)  # noqa: E731
        self.home = DeviceField(t["home"], components=10)
        self.home_post = DeviceField(t["home_post"], components=10)
        self.h = DeviceField(t["h"], components=7)
        self.water_phase = DeviceField(t["phi"])
        self.pressure_lattice = DeviceField(t["pressure"])
        self.old_pressure = DeviceField(t["old_pressure"])
        self.velocity_lattice = vec("u")
        self.old_velocity = vec("old_u")
        self.force_density = vec("force")
        self.home_acceleration = vec("accel")
        self.phase_gradient_lattice = vec("grad")
        self.phase_mass_flux = vec("flux")
        self.capillary_stress = DerivedField(self._capillary_stress, (*self.shape, 3, 3))
        edited = self._geometry_edited
        self.coverage = DeviceField(t["coverage"], on_write=edited)
        self.solid_body_id = DeviceField(t["id"], logical_dtype=np.int32, on_write=edited)
        self.previous_body_id = DeviceField(t["prev_id"], logical_dtype=np.int32, on_write=edited)
        self.coverage_body_id = DeviceField(t["cov_id"], logical_dtype=np.int32, on_write=edited)
        self.refill_state = DeviceField(t["refill_state"], components=5)
        self.refill_next = DeviceField(t["refill_next"], components=5)
        self.refill_valid = DeviceField(t["refill_valid"])
        self.refill_next_valid = DeviceField(t["refill_next_valid"])
        self.reference_density = DeviceField(t["ref_density"])
        self.reference_pressure = DeviceField(t["ref_pressure"])
        body = t["body"]
        self.body_origin = DeviceField(body[:, 0:3], on_write=edited)
        self.body_rotation = _MatrixRows(body[:, 3:12], on_write=edited)
        self.body_center = DeviceField(body[:, 12:15])
        self.body_velocity = DeviceField(body[:, 15:18])
        self.body_angular_velocity = DeviceField(body[:, 18:21])
        self.hydrodynamic_force = DeviceField(self._loads[:, 0:3])
        self.hydrodynamic_torque = DeviceField(self._loads[:, 3:6])
        self.reduced_state = DeviceField(self._reduced)
        self.material_size = DeviceField(t["material_size"])
        self.initial_body_temperature = DeviceField(t["body_t0"])
        self.material_mass = DeviceField(t["material_mass"], on_write=edited)
        self.material_energy = DeviceField(t["material_energy"])
        self.material_heat = DeviceField(t["material_heat"])
        self.water_volume = DeviceField(t["water_volume"])
        self.water_energy = DeviceField(t["water_energy"])
        self.target_energy = DeviceField(t["target_energy"])
        self.sampled_ice_temperature = DeviceField(t["sampled_ice_t"])
        self.energy_flux = vec("energy_flux")
        self.volume_flux = vec("volume_flux")
        self.phase_parity = HostScalar(self, "_parity")
        scalars = {
            "invalid_index": np.int32, "maximum_speed": np.float32, "peak_speed": np.float32,
            "repair_count": np.int32, "phase_clip_volume": np.float32, "remap_energy": np.float32,
            "discarded_heat": np.float32, "max_outflow": np.float32, "thermal_invalid": np.int32,
            "openings": np.int32, "remaining": np.int32, "refill_lower": np.int32, "refill_upper": np.int32,
        }
        self._scalar_names = tuple(scalars)
        for name, dtype in scalars.items():
            setattr(self, name, ControlScalar(self, name, dtype))
        self._gradient_geometry_lower = ControlScalar(self, "geometry_lower", np.int32)
        self._gradient_geometry_upper = ControlScalar(self, "geometry_upper", np.int32)

    _GRID_FIELDS = (
        "home", "home_post", "h", "water_phase", "pressure_lattice", "old_pressure", "coverage",
        "velocity_lattice", "old_velocity", "force_density", "home_acceleration", "phase_gradient_lattice",
        "phase_mass_flux", "solid_body_id", "previous_body_id", "coverage_body_id", "refill_state",
        "refill_next", "refill_valid", "refill_next_valid", "reference_density", "reference_pressure",
        "body_origin", "body_rotation", "body_center", "body_velocity", "body_angular_velocity",
        "hydrodynamic_force", "hydrodynamic_torque", "material_size", "initial_body_temperature",
        "material_mass", "material_energy", "material_heat", "water_volume", "water_energy",
        "target_energy", "sampled_ice_temperature", "energy_flux", "volume_flux", "capillary_stress",
    )

    def fields(self):
        """Restart-state fields by reference name (checkpoint._fields)."""
        out = {name: getattr(self, name) for name in self._GRID_FIELDS}
        out["phase_parity"] = self.phase_parity
        for name in self._scalar_names:
            out[name] = getattr(self, name)
        return out

    # --------------------------------------------------------------- plumbing
    def _torch_stream(self):
        """The stream every launch goes to: torch's current stream, fixed for
        the length of one ``step`` call (so the loop asks torch once)."""
        held = self._step_stream
        return held[0] if held is not None else torch.cuda.current_stream(self.device)

    def _stream(self):
        held = self._step_stream
        return held[1] if held is not None else ctypes.c_void_p(torch.cuda.current_stream(self.device).cuda_stream)

    def _call(self, name, *args):
        fn = self._functions.get(name)
        if fn is None:
            fn = self._functions[name] = getattr(self._lib, "icy3d_" + name)
        check(fn(self._gp, *args, self._stream()), name)

    def _read_control(self):
        return Control.from_buffer_copy(self._sync_control())

    def _sync_control(self):
        """The control block copied into the pinned host buffer, returned as a
        struct that aliases that buffer (valid until the next copy)."""
        self._call("read_control", self._control_host.data_ptr())
        return self._control_alias

    def _write_control(self, control):
        raw = np.frombuffer(bytes(control), dtype=np.uint8)
        self._t["control"].copy_(torch.from_numpy(raw.copy()))

    def _rigid_step(self, loads):
        """rigid.py:178-347 and the upload of simulator.py:259-286 in one
        native call: the packed rows go straight into the pinned staging
        buffer and are queued for upload; returns their per-body coverage
        boxes."""
        self._upload_done.synchronize()  # the previous upload has left the staging buffer
        staging = self._upload_staging_view
        self.rigid.advance_packed(loads, staging)
        self._body_state[...] = staging
        check(self._lib.icy3d_copy_async(self._t["body"].data_ptr(), staging.ctypes.data, staging.nbytes,
                                         self._stream()), "body upload")
        self._upload_done.record(self._torch_stream())
        return self._coverage_boxes(staging)

    # Field widths of the FP64 rigid arrays, in _RIGID_FIELDS order.
    _RIGID_WIDTHS = (3, 4, 3, 3, 3, 1, 9, 3, 3)

    def _enable_device_rigid(self):
        """Keep the FP64 rigid state in device memory, field after field in
        one buffer, and step it with ``icy3d_rigid_step_device``.
        ``self.rigid`` then holds a copy that every ``step()`` call brings up
        to date when it returns; ``rigid.upload()`` sends host edits back."""
        B = self.body_count
        flat = torch.zeros(sum(self._RIGID_WIDTHS) * B, dtype=torch.float64, device=self.device)
        arrays, offset = _RigidArrays(B), 0
        for name, width in zip(_RIGID_FIELDS, self._RIGID_WIDTHS):
            setattr(arrays, name, ctypes.cast(flat.data_ptr() + 8 * offset * B, ctypes.POINTER(ctypes.c_double)))
            offset += width
        self._rigid_dev = {
            "flat": flat, "arrays": arrays,
            "host": torch.zeros(flat.numel(), dtype=torch.float64).pin_memory(),
            "rows": torch.zeros((B, _native.STATE_STRIDE), dtype=torch.float32).pin_memory(),
        }
        self._push_rigid()

    def _push_rigid(self):
        """Host FP64 rigid arrays -> the device copy (stream-ordered)."""
        d = self._rigid_dev
        self.rigid._arrays()
        d["host"].numpy()[...] = np.concatenate([getattr(self.rigid, name).ravel() for name in _RIGID_FIELDS])
        with torch.cuda.stream(self._torch_stream()):
            d["flat"].copy_(d["host"], non_blocking=True)
        self._torch_stream().synchronize()

    def _pull_rigid(self):
        """The device FP64 rigid state -> ``self.rigid`` (in place)."""
        d = self._rigid_dev
        with torch.cuda.stream(self._torch_stream()):
            d["host"].copy_(d["flat"], non_blocking=True)
        self._torch_stream().synchronize()
        self.rigid._arrays()
        flat, offset, B = d["host"].numpy(), 0, self.body_count
        for name, width in zip(_RIGID_FIELDS, self._RIGID_WIDTHS):
            target = getattr(self.rigid, name)
            target[...] = flat[offset * B : (offset + width) * B].reshape(target.shape)
            offset += width

    def _rigid_step_device(self, stream=None):
        """Queue the FP64 rigid update on the device (on ``stream``, else the
        step's stream): loads from the control block, rows into the grid's
        body buffer and into pinned memory, the status and coverage boxes
        into ``control.rigid``."""
        d = self._rigid_dev
        stream = stream if stream is not None else self._torch_stream()
        args = self.rigid._step_arguments()
        control = self._t["control"].data_ptr()
        check(self._lib.icy3d_rigid_step_device(
            ctypes.byref(d["arrays"]), ctypes.c_void_p(control + Control.loads.offset), args["pointers"][0],
            args["linear"], args["angular"], args["shape"], args["boundary"], args["iterations"],
            ctypes.c_void_p(self._t["material_size"].data_ptr()), ctypes.c_void_p(self._t["body"].data_ptr()),
            ctypes.c_void_p(control + Control.rigid.offset), ctypes.c_void_p(stream.cuda_stream)), "device rigid step")
        with torch.cuda.stream(stream):
            d["rows"].copy_(self._t["body"], non_blocking=True)

    def _device_rigid_outcome(self, result):
        """After the device rigid step's results reached the host: raise its
        error as the host solver would, else take the rows and return the
        per-body coverage boxes."""
        status = int(result.status)
        if status == -4:
            raise RuntimeError(
                f"rigid displacement exceeds half a cell at step {self.steps + 1}, body {int(result.failed_body)}")
        if status in (-5, -6):
            _contact_error(status, self.steps, list(result.residual))
        check(status, "device rigid step")
        B = self.body_count
        self._body_state[...] = self._rigid_dev["rows"].numpy()
        lo = np.array(result.box_lo, dtype=np.int32)[:B]
        hi = np.array(result.box_hi, dtype=np.int32)[:B]
        return lo, hi

    def _upload_rigid_state(self, state):
        """rigid.py:136-151 device side: one small host-to-device copy,
        queued from pinned memory so that the host does not wait for the
        kernels still ahead of it on the stream."""
        state = np.ascontiguousarray(state, dtype=np.float32)
        self._body_state[...] = state
        self._upload_done.synchronize()  # the previous upload has left the staging buffer
        self._upload_staging.numpy()[...] = state
        self._t["body"].copy_(self._upload_staging, non_blocking=True)
        self._upload_done.record(self._torch_stream())

    def _reduce_mass_state(self):
        self._call("reduce_mass")
        control = self._read_control()
        return np.array(control.reduced, dtype=np.float32)[: self.body_count]

    def _download_loads(self):
        return np.array(self._read_control().loads, dtype=np.float32)[: self.body_count]

    def _capillary_stress(self):
        out = torch.empty((9, *self.shape), dtype=torch.float32, device=self.device)
        self._call("capillary_stress", ctypes.c_void_p(out.data_ptr()))
        return np.moveaxis(out.cpu().numpy(), 0, -1).reshape(*self.shape, 3, 3)

    def invalidate_gradient_cache(self):
        """Call after externally editing phase, coverage, or fluid/solid masks."""
        self._gradient_cache_valid = False

    def _restored(self, keep_gradients):
        """After every field was written from a restart file: the host copy of
        the uploaded body rows follows the device; labels, coverage and
        previous labels were saved together with those rows, so the next
        refresh covers the bodies' boxes for those rows (as the saved run's
        did) and the box of every cell whose label differs from its previous
        label or is unresolved (which the saved run's box history covered),
        and the link classes are rebuilt from the labels.  The saved phase
        gradient is the cache the saved run would have used next (it may
        precede the last geometry update outside the refreshed boxes), so it
        is kept when the file comes from these sources and rebuilt
        otherwise."""
        self._body_state[...] = self._t["body"].cpu().numpy()
        self._flags_valid = False
        self._raster_full = False
        ids, previous = self._t["id"], self._t["prev_id"]
        unsettled = ((ids != previous) | (ids == -3) | (previous == -3)).nonzero()
        stale = None
        if len(unsettled):
            stale = (unsettled.min(dim=0).values.cpu().numpy().astype(np.int32).reshape(1, 3),
                     unsettled.max(dim=0).values.cpu().numpy().astype(np.int32).reshape(1, 3) + 1)
        self._box_history = (self._coverage_boxes(), stale)
        control = self._read_control()
        control.cavity_lower[:] = self.shape
        control.cavity_upper[:] = (-1, -1, -1)
        self._write_control(control)
        self._gradient_cache_valid = bool(keep_gradients)

    @property
    def physical_time_s(self):
        return self.steps * self.scales.dt_s

    # ------------------------------------------------- reference kernel methods
    def _classify_home(self):
        self._call("classify", None, None)
        self._flags_valid = True

    def _gradients(self, classified=False):
        if not classified:
            self._classify_home()
        self._call("gradients", None, None)

    def _collide_phase(self, moving_walls=True):
        self._call("collide_phase", self._parity, int(moving_walls))
        self._parity = 1 - self._parity

    def _recover_phase(self, recover_flow=False):
        self._call("recover_phase", self._parity, int(recover_flow))

    def _recover_pressure(self):
        self._call("recover_pressure")

    def _scan_stability(self):
        self._call("scan_stability")

    def _forces(self, with_flux, moment_pressure=False):
        self._call("forces", int(with_flux), int(moment_pressure))
        self._flags_valid = True

    def _collide_momentum(self):
        self._call("collide_momentum")

    def _stream_home(self, classified=False):
        if not classified:
            self._classify_home()
        self._call("stream_home")

    def _collide_stream_home(self, classified=False):
        """``_collide_momentum`` then ``_stream_home`` in one fused pass (the
        loads are cleared and accumulated as by the step)."""
        if not classified:
            self._classify_home()
        self._call("collide_stream_home")
        self._swap_home()

    def _swap_home(self):
        """After a fused collide-stream the streamed moments are in the
        home_post buffer: the two buffers trade places (grid pointers,
        tensors and field views)."""
        t, g = self._t, self._grid
        t["home"], t["home_post"] = t["home_post"], t["home"]
        g.home, g.home_post = g.home_post, g.home
        self.home.t, self.home_post.t = t["home"], t["home_post"]

    def _seed_populations(self):
        self._call("seed_populations")

    def _set_equilibrium_all(self, velocity=None, pressure=None, with_phase=True):
        if velocity is not None:
            self.velocity_lattice.from_numpy(
                np.where((self.solid_body_id.to_numpy() == -1)[..., None], np.asarray(velocity, np.float32),
                         self.velocity_lattice.to_numpy()))
        use = pressure is not None
        self._call("set_equilibrium_all", self._parity, int(with_phase), int(use), float(pressure or 0.0))

    def _rasterize(self, boxes=None):
        """simulator.py:288-323 over ``boxes`` (int32 lo, hi: [count, 3];
        by default those of the next refresh)."""
        lo, hi = self._raster_boxes() if boxes is None else boxes
        self._call("rasterize_boxes", len(lo), lo.ctypes.data, hi.ctypes.data)
        self._flags_valid = False

    def _repair_phase_layout(self, boxes=None):
        """phase.py:163-184 over ``boxes`` (int32 lo, hi: [count, 3], whose
        copies extended one cell down are disjoint; the whole grid by
        default).  A link (I, I+e) is swapped by the thread of I, so each box
        is extended one cell down."""
        lo, hi = self._full_boxes if boxes is None else boxes
        lo = np.ascontiguousarray(np.maximum(lo - 1, 0), dtype=np.int32)
        self._call("repair_phase_layout_boxes", self._parity, len(lo), lo.ctypes.data, hi.ctypes.data)

    def _synchronize_water(self):
        self._call("synchronize_water")

    def _thermal_fluxes(self, advect):
        self._call("thermal_fluxes", int(advect))

    def _apply_thermal_fluxes(self, dt, advect):
        self._call("apply_thermal_fluxes", float(dt), int(advect))

    def _advect_water(self, dt):
        """``_thermal_fluxes(True)`` then ``_apply_thermal_fluxes(dt, True)``
        in one pass into the spare water planes, which then trade places
        with the water planes (the flux fields are not written)."""
        self._into_spare_water("advect_water", float(dt))

    def _conduct_water(self, dt):
        """``_thermal_fluxes(False)`` then ``_apply_thermal_fluxes(dt, False)``
        in one pass into the spare energy plane, which then trades places
        with the water energy plane (the flux fields are not written)."""
        t, g = self._t, self._grid
        self._call("conduct_water", float(dt), ctypes.c_void_p(t["water_energy_next"].data_ptr()))
        t["water_energy"], t["water_energy_next"] = t["water_energy_next"], t["water_energy"]
        g.water_energy = t["water_energy"].data_ptr()
        self.water_energy.t = t["water_energy"]

    def _synchronize_water_fused(self):
        """``_synchronize_water`` in one pass into the spare water planes
        (target_energy is not written)."""
        self._into_spare_water("synchronize_water_into")

    def _remap_advect_remap(self, dt):
        """``_synchronize_water_fused``, ``_advect_water(dt)`` and
        ``_synchronize_water_fused`` in one pass into the spare water planes."""
        self._into_spare_water("remap_advect_remap", float(dt))

    def _into_spare_water(self, name, *args):
        t, g = self._t, self._grid
        self._call(name, *args, ctypes.c_void_p(t["water_volume_next"].data_ptr()),
                   ctypes.c_void_p(t["water_energy_next"].data_ptr()))
        t["water_volume"], t["water_volume_next"] = t["water_volume_next"], t["water_volume"]
        t["water_energy"], t["water_energy_next"] = t["water_energy_next"], t["water_energy"]
        g.water_volume, g.water_energy = t["water_volume"].data_ptr(), t["water_energy"].data_ptr()
        self.water_volume.t, self.water_energy.t = t["water_volume"], t["water_energy"]

    def _measure_outflow(self):
        self._call("measure_outflow")

    def _body_conduction(self, dt):
        self._call("body_conduction", float(dt))

    def _thermal_ice_bounds(self):
        """thermal.py:295-306 from the uploaded FP32 body state."""
        state = self._body_state
        shape = np.array(self.shape)
        lo, hi = shape.copy(), np.zeros(3, dtype=int)
        sizes = np.array([b.size_cells for b in self.config.bodies], dtype=np.float32)
        for b in range(self.body_count):
            half = np.float32(0.5) * sizes[b] + np.float32(1.0)
            rot = np.abs(state[b, 3:12].reshape(3, 3))
            extent = (rot @ half).astype(np.float32)
            origin = state[b, 0:3]
            lower = np.floor(origin - extent).astype(int) - 3
            upper = np.ceil(origin + extent).astype(int) + 3
            lo, hi = np.minimum(lo, lower), np.maximum(hi, upper)
        return np.maximum(lo, 0), np.minimum(hi, shape)

    def _exchange_heat(self, dt):
        lo, hi = self._thermal_ice_bounds()
        self._call("exchange_heat", float(dt), int3(lo), int3(hi))

    def _exchange_heat_full(self, dt):
        self._call("exchange_heat", float(dt), int3((0, 0, 0)), int3(self.shape))

    def _apply_melting(self):
        self._call("apply_melting")

    def _reduce_mass(self):
        self._call("reduce_mass")

    def _sample_ice_temperature(self):
        self._call("sample_ice_temperature")

    def _check_heat(self):
        self._call("check_heat")

    def _project_refill(self):
        control = self._read_control()
        lo = np.array(control.refill_lower)
        hi = np.array(control.refill_upper) + 1
        self._call("project_refill", self._parity, int3(lo), int3(hi))

    def _write_gradient_all(self):
        self._call("write_gradient_all")

    def boundary_flags(self):
        self._classify_home()
        return DeviceField(self._t["flag"]).to_numpy().astype(np.int32)

    def generic_forces(self):
        out = torch.empty((6, *self.shape), dtype=torch.float32, device=self.device)
        self._call("generic_forces", ctypes.c_void_p(out.data_ptr()))
        return np.moveaxis(out.cpu().numpy(), 0, -1)

    def _stress_neighbor_velocity(self, cell, c):
        out = torch.zeros(4, dtype=torch.float32, device=self.device)
        self._call("probe_stress_velocity", int3(cell), int3(c), ctypes.c_void_p(out.data_ptr()))
        return out[:3].cpu().numpy().astype(float)

    def mirror_probe(self, cell, c):
        out = torch.zeros(4, dtype=torch.float32, device=self.device)
        self._call("probe_mirror", int3(cell), int3(c), ctypes.c_void_p(out.data_ptr()))
        return out.cpu().numpy().astype(float)

    def export_phase_populations(self, out=None):
        """phase.py:186-191: logical D3Q7 populations [nx, ny, nz, 7]."""
        buf = torch.empty((7, *self.shape), dtype=torch.float32, device=self.device)
        self._call("export_phase", self._parity, ctypes.c_void_p(buf.data_ptr()))
        result = np.moveaxis(buf.cpu().numpy(), 0, -1)
        if out is not None:
            out[...] = result
        return result

    # ------------------------------------------------------------ host logic
    def _build_reference(self):
        """simulator.py:349-383: frozen hydrostatic reference (host NumPy)."""
        cfg = self.config
        phase = self.water_phase.to_numpy()
        ids = self.solid_body_id.to_numpy()
        ref = (np.arange(self.ny) < cfg.boundary_cells + cfg.floor_water_depth_cells).astype(float)
        full_width = cfg.water_width == self.nx - cfg.boundary_cells
        mask = ids == -1
        if full_width:
            ref = (np.arange(self.ny) < cfg.water_height).astype(float)
        else:
            mask[: cfg.water_width] = False
        if cfg.floor_water_depth_cells or full_width:
            counts = mask.sum(axis=(0, 2))
            sums = np.where(mask, phase, 0).sum(axis=(0, 2), dtype=float)
            np.divide(sums, counts, out=ref, where=counts > 0)
        rho = self.rho_air + (1 - self.rho_air) * ref
        p = -self.gravity[1] * (np.cumsum(rho[::-1])[::-1] - 0.5 * rho)
        excess = np.where(ids == -1, (phase - ref[None, :, None]) * (1 - self.rho_air), 0.0)
        dynamic = -self.gravity[1] * (np.cumsum(excess[:, ::-1, :], axis=1)[:, ::-1, :] - 0.5 * excess)
        self.reference_density.from_numpy(rho.astype(np.float32))
        self.reference_pressure.from_numpy(p.astype(np.float32))
        self.pressure_lattice.from_numpy(dynamic.astype(np.float32))

    def _raise_unstable(self, index):
        cell = (index // (self.ny * self.nz), index // self.nz % self.ny, index % self.nz)
        phi = self.water_phase.to_numpy()[cell]
        velocity = self.velocity_lattice.to_numpy()[cell]
        raise RuntimeError(f"unstable fluid at step {self.steps + 1}, cell {cell}: phi={phi}, velocity={velocity}")

    def _raise_if_unstable(self, saved_rigid, saved_rows, gradients_pending):
        """After the flow step: if its stability scan found an invalid cell,
        restore the body state from before this step's rigid update, run the
        gradient pass the step deferred to after the refresh (the reference
        has it before its check), and raise the reference's error."""
        if not self.config.check_stability:
            return
        control = self._read_control()
        if control.invalid_index >= math.prod(self.shape):
            return
        if self._rigid_dev is not None:
            if saved_rigid is not None:
                with torch.cuda.stream(self._torch_stream()):
                    self._rigid_dev["flat"].copy_(saved_rigid)
        else:
            self.rigid.restore(saved_rigid)
        self._upload_rigid_state(saved_rows)
        if gradients_pending:
            self._gradients(classified=True)
        self._raise_unstable(control.invalid_index)

    def check_stability(self, scanned=False):
        """simulator.py:807-821."""
        if not scanned:
            self._scan_stability()
        control = self._read_control()
        if control.invalid_index < math.prod(self.shape):
            self._raise_unstable(control.invalid_index)
        return float(control.maximum_speed)

    def _refresh_geometry(self, phase_changed=True, current=None, cavity=(), full_gradients=False, guarded=False,
                          remap=True):
        """simulator.py:708-736 over the boxes of ``_raster_boxes`` (outside
        them the reference's passes change nothing); the refill loop reads
        one counter per sweep.  ``current``: the bodies' coverage boxes and
        ``cavity``: the last commit's unresolved cells, when the caller has
        them.  ``full_gradients``: the flow step left out its gradient pass,
        which runs over the whole grid here after the class refresh.
        ``guarded``: the refresh was queued before the host read the flow
        step's stability scan; if that scan found an invalid cell, the
        refresh kernels changed nothing, and None is returned with the box
        history as it was.  ``remap`` False: the caller remaps the water to
        the refreshed phase itself, before anything reads it."""
        history, raster_full = self._box_history, self._raster_full
        boxes = self._raster_boxes(current, cavity)
        count, lo_p, hi_p = len(boxes[0]), boxes[0].ctypes.data, boxes[1].ctypes.data
        self._grid.refresh_guard = 1 if guarded else 0
        try:
            self._call("refresh_begin_boxes", self._parity, count, lo_p, hi_p)
        finally:
            self._grid.refresh_guard = 0
        self._flags_valid = False
        # After this read the GPU waits for the host until the next launch:
        # the struct aliases the pinned copy and the box arithmetic is on
        # plain ints (three components).
        control = self._sync_control()
        if guarded and self.config.check_stability and control.invalid_index < math.prod(self.shape):
            self._box_history, self._raster_full = history, raster_full
            self._flags_valid = True
            return None
        remaining, covered = int(control.openings), int(control.covered)
        shape = self.shape
        lower, upper = tuple(control.refill_lower), tuple(control.refill_upper)
        # gradients.py:198-209: changed box plus the dependency radius.  Every
        # change lies in a raster box, so the library refreshes only the parts
        # of that box near the raster boxes; elsewhere the reference's pass
        # rewrites the same values.
        lo = tuple(map(min, lower, control.geometry_lower))
        hi = tuple(map(max, upper, control.geometry_upper))
        reference_box = (None, None)
        if all(h >= l for l, h in zip(lo, hi)):
            radius = self.GRADIENT_DEPENDENCY_RADIUS
            reference_box = (int3(max(v - radius, 0) for v in lo),
                             int3(min(v + radius + 1, n) for v, n in zip(hi, shape)))
        if remaining > 0:
            box_lo = int3(max(v - 1, 0) for v in lower)
            box_hi = int3(min(v + 2, n) for v, n in zip(upper, shape))
            self._call("seed_refill_region", box_lo, box_hi)
        has_openings = remaining > 0
        self.pending_cells = 0
        while remaining:
            self._call("propagate_refill", box_lo, box_hi)
            new = int(self._sync_control().remaining)
            self._call("accept_refill", box_lo, box_hi)
            if new == remaining:
                self.pending_cells = new
                break
            remaining = new
        self._call("refresh_end_boxes", count, lo_p, hi_p, *reference_box, int(full_gradients))
        # Labels changed only inside the refreshed boxes, which were reclassified.
        self._flags_valid = True
        if has_openings or covered:
            self._call("project_refill", self._parity, int3(lower), int3(v + 1 for v in upper))
        if remap and (phase_changed or has_openings or covered):
            self._synchronize_water_fused()
        return Control.from_buffer_copy(control)

    def _advance_water(self, speed_bound=None):
        """The remap to the refreshed phase and thermal.py:208-226.  One
        substep whose count needs no measurement is fused with the remaps
        around it."""
        th = self.config.thermal
        if th.advection_enabled and speed_bound is not None and 3 * speed_bound <= th.max_courant_number:
            self._remap_advect_remap(self.scales.dt_s)
            return
        self._synchronize_water_fused()
        self._advance_advection(speed_bound)

    def _advance_advection(self, speed_bound=None):
        """thermal.py:208-226."""
        th = self.config.thermal
        if not th.advection_enabled:
            return
        rate = 3 * speed_bound if speed_bound is not None else math.inf
        if rate > th.max_courant_number:
            self._measure_outflow()
            rate = float(self._sync_control().max_outflow)
        if not math.isfinite(rate):
            raise RuntimeError(f"nonfinite thermal velocity at step {self.steps + 1}")
        substeps = max(1, math.ceil(rate / th.max_courant_number))
        self._check_substeps(substeps)
        for _ in range(substeps):
            self._advect_water(self.scales.dt_s / substeps)
            self._synchronize_water_fused()

    def _check_substeps(self, count):
        if count > self.config.thermal.max_substeps_per_update:
            raise RuntimeError(f"thermal update needs {count} substeps at step {self.steps + 1}")

    def _advance_conduction(self, dt):
        """thermal.py:234-258."""
        alpha = max(self.k_water / self.rho_cp, self.k_ice / (self.config.rho_ice * self.cp_ice))
        substeps = max(1, math.ceil(alpha * dt / (self.dx**2 * self.config.thermal.max_fourier_number)))
        self._check_substeps(substeps)
        for _ in range(substeps):
            self._body_conduction(dt / substeps)
            self._conduct_water(dt / substeps)
            self._exchange_heat(dt / substeps)
            self._apply_melting()
            if self._rigid_dev is not None:
                self._pull_rigid()
            self.rigid.update_mass(upload=False)
            self.rigid.resolve_contacts()
            self.rigid.upload()
            self._refresh_geometry(phase_changed=False)
        if self.config.check_stability:
            self._check_heat()
            if int(self._read_control().thermal_invalid):
                raise RuntimeError(f"invalid thermal state at step {self.steps + 1}")

    # Kernel-group names of the fused flow step (include/icy3d.h).
    PROFILE_GROUPS = ("phase_collide", "forces", "home_collide_stream", "phase_recover", "gradients")

    def attach_profiler(self):
        """Time each kernel group of the flow step with HIP events on the
        solver's stream until ``detach_profiler()``; returns the running
        totals through ``profile_totals()``."""
        if getattr(self, "_profile", None) is None:
            handle = ctypes.c_void_p()
            check(self._lib.icy3d_profile_create(ctypes.byref(handle)), "profile_create")
            self._profile = handle

    def profile_totals(self):
        """{group: (total milliseconds, steps)} accumulated so far."""
        totals = (ctypes.c_double * len(self.PROFILE_GROUPS))()
        count = ctypes.c_int64()
        check(self._lib.icy3d_profile_read(self._profile, totals, ctypes.byref(count)), "profile_read")
        return {name: (totals[i], count.value) for i, name in enumerate(self.PROFILE_GROUPS)}

    def detach_profiler(self):
        if getattr(self, "_profile", None) is not None:
            self._lib.icy3d_profile_destroy(self._profile)
            self._profile = None

    def step(self, num_steps=1):
        """simulator.py:823-850: one fused device launch sequence for the
        flow part, then host rigid bodies, geometry refresh and heat."""
        num_steps = integer("num_steps", num_steps, 0)
        stream = torch.cuda.current_stream(self.device)
        self._step_stream = (stream, ctypes.c_void_p(stream.cuda_stream))
        try:
            self._run_steps(num_steps)
            if self._rigid_dev is not None:
                self._pull_rigid()
        finally:
            self._step_stream = None

    def _run_steps(self, num_steps):
        profile = getattr(self, "_profile", None)
        device_rigid = self._rigid_dev is not None
        for _ in range(num_steps):
            refresh = not self._gradient_cache_valid
            classify = int(not self._flags_valid)
            saved_flat = None
            if profile is None:
                # The loads are final after the stream: copy them out, queue the
                # recovery, and integrate the bodies on the host while the GPU
                # runs it.  The step's gradient pass runs once, after the
                # geometry refresh (the field the reference has after its
                # refresh: outside its refresh box nothing the gradients
                # depend on changes in between).
                self._call("flow_step_begin", self._parity, int(refresh), classify)
                self._swap_home()
                if device_rigid:
                    # The recovery reads neither the body rows nor the rigid
                    # state, so the solver goes first and the host waits for
                    # its results while the recovery runs.
                    if self.config.check_stability:
                        saved_flat = self._rigid_dev["flat"].clone()
                    self._rigid_step_device()
                self._loads_host.copy_(self._t["control"], non_blocking=True)
                self._loads_ready.record(self._torch_stream())
                self._call("flow_step_recover", self._parity)
                self._loads_ready.synchronize()
                loads = self._loads_view
                cavity = self._cavity_box(self._cavity_view[:3], self._cavity_view[3:])
                rigid_result = self._loads_control.rigid if device_rigid else None
            else:
                check(self._lib.icy3d_flow_step_profiled(self._gp, self._parity, int(refresh), classify, profile,
                                                         self._stream()), "flow_step")
                self._swap_home()
                if device_rigid:
                    if self.config.check_stability:
                        saved_flat = self._rigid_dev["flat"].clone()
                    self._rigid_step_device()
                control = self._read_control()
                rigid_result = control.rigid
                loads = np.array(control.loads, dtype=np.float32)[: self.body_count]
                cavity = self._cavity_box(control.cavity_lower, control.cavity_upper)
                check(self._lib.icy3d_profile_collect(profile), "profile_collect")
            self._gradient_cache_valid = True
            self._flags_valid = True
            self._parity = 1 - self._parity
            # simulator.py:835-839 checks stability before the bodies move.
            # Here the host integrates them while the recovery and its scan
            # run, and queues the refresh before it reads the scan; the
            # refresh kernels do nothing after an unstable scan, and the
            # body state is put back before the error is raised.
            saved_rows = self._body_state.copy()
            saved_rigid = saved_flat if device_rigid else self.rigid.save()
            try:
                current = self._device_rigid_outcome(rigid_result) if device_rigid else self._rigid_step(loads)
            except RuntimeError:
                self._raise_if_unstable(saved_rigid, saved_rows, profile is None)
                raise
            # The geometry refresh's first control read follows the recovery's
            # stability scan in stream order.
            control = self._refresh_geometry(current=current, cavity=cavity, full_gradients=profile is None,
                                             guarded=True, remap=False)
            if control is None:
                self._raise_if_unstable(saved_rigid, saved_rows, profile is None)
            speed_bound = None
            if self.config.check_stability:
                speed_bound = float(control.maximum_speed)
            self._advance_water(speed_bound)
            self._thermal_pending += 1
            if self._thermal_pending >= self.config.thermal.update_interval_lbm_steps:
                self._advance_conduction(self._thermal_pending * self.scales.dt_s)
                self._thermal_pending = 0
            self.steps += 1

    def flush_thermal(self):
        """Resolve the final partial thermal interval at the end of a run."""
        if self._thermal_pending:
            self._advance_conduction(self._thermal_pending * self.scales.dt_s)
            self._thermal_pending = 0

    def snapshot(self):
        """simulator.py:858-889."""
        th = self.config.thermal
        ids = self.solid_body_id.to_numpy()
        phi = self.water_phase.to_numpy()
        volume, energy = self.water_volume.to_numpy(), self.water_energy.to_numpy()
        cp = self.config.rho_water * th.properties.specific_heat_water_j_kg_k
        temp = np.full(self.shape, th.initial_air_temperature_c, np.float32)
        wet = volume > 1e-30
        temp[wet] = (energy[wet] / (cp * volume[wet]) + th.properties.melting_temperature_c).astype(np.float32)
        self._sample_ice_temperature()
        ice = self.sampled_ice_temperature.to_numpy()
        temp[ids >= 0] = ice[ids >= 0]
        return {
            "water_phase": phi,
            "solid_body_id": ids,
            "ice_fraction": self.coverage.to_numpy(),
            "velocity_m_s": self.velocity_lattice.to_numpy() * self.scales.velocity_m_s,
            "pressure_pa": (self.pressure_lattice.to_numpy() + self.reference_pressure.to_numpy()[None, :, None])
            * self.scales.pressure_pa,
            "temperature_c": temp,
        }

    def diagnostics(self):
        """simulator.py:891-947."""
        self._scan_stability()
        control = self._read_control()
        volume = self.water_volume.to_numpy()
        rigid = self.rigid
        centers = self.body_center.to_numpy() * self.scales.dx_m
        result = {
            "step": self.steps,
            "time_s": self.physical_time_s,
            "water_volume_m3": float(volume.sum(dtype=float)),
            "water_volume_change_ratio": (
                float(volume.sum(dtype=float) / self.initial_water_volume_m3 - 1)
                if self.initial_water_volume_m3 > 0 else None
            ),
            "water_energy_j": float(self.water_energy.to_numpy().sum(dtype=float)),
            "ice_sensible_energy_j": float(self.material_energy.to_numpy().sum(dtype=float)),
            "maximum_fluid_speed_lattice": float(control.maximum_speed),
            "peak_fluid_speed_lattice": float(control.peak_speed),
            "phase_volume_change_ratio": float(
                self.water_phase.to_numpy().sum(dtype=np.float64) * self.cell_volume / self.initial_phase_volume_m3 - 1
            ),
            "phase_volume_projection_m3": 0.0,
            "phase_projection_momentum_x_n_s": 0.0,
            "phase_projection_momentum_y_n_s": 0.0,
            "phase_projection_momentum_z_n_s": 0.0,
            "ice_mass_kg": float(rigid.mass.sum() * self.scales.mass_kg),
            "melted_mass_kg": float(self.initial_ice_mass_kg.sum() - rigid.mass.sum() * self.scales.mass_kg),
            "gas_repair_count": int(control.repair_count),
            "phase_clip_volume_m3": float(control.phase_clip_volume) * self.scales.dx_m**3,
            "thermal_remap_energy_j": float(control.remap_energy),
            "discarded_melt_heat_j": float(control.discarded_heat),
            "pending_refill_cells": self.pending_cells,
        }
        for b in range(self.body_count):
            result[f"ice_{b}_mass_kg"] = float(rigid.mass[b] * self.scales.mass_kg)
            for a, label in enumerate("xyz"):
                result[f"ice_{b}_{label}_m"] = float(centers[b, a])
                result[f"ice_{b}_v{label}_m_s"] = float(rigid.velocity[b, a] * self.scales.velocity_m_s)
                result[f"ice_{b}_omega_{label}_s_1"] = float(rigid.omega[b, a] / self.scales.dt_s)
            for a, label in enumerate("wxyz"):
                result[f"ice_{b}_q{label}"] = float(rigid.q[b, a])
        return result


class _MatrixRows(DeviceField):
    """[B, 9] device rows exposed as [B, 3, 3] matrices."""

    @property
    def shape(self):
        return (self.t.shape[0], 3, 3)

    def to_numpy(self):
        return self.t.detach().cpu().numpy().reshape(-1, 3, 3).copy()

    def from_numpy(self, value):
        value = np.array(np.broadcast_to(np.asarray(value, dtype=np.float32), self.shape))
        self.t.copy_(torch.from_numpy(value.reshape(-1, 9)))
        if self.on_write is not None:
            self.on_write()
