"""Tile edges of the 3D flow kernels against the FP64 oracle: grids whose y
and z extents leave partial tiles, need several tiles, or fit into one, and
x extents of one and of several slab chunks.  Tolerance: the single-kernel
bar of the parity tests (2e-5 of the field scale in FP32)."""

import numpy as np
import pytest

from test_parity3d import KERNELS, assert_close, prepared

pytestmark = pytest.mark.gpu

SHAPES = [(14, 13, 100), (16, 37, 66), (14, 70, 14), (300, 13, 12)]


def tank(nx, ny, nz):
    from projecticy_amd.iceflow3d import IceBodyConfig, IceFlowConfig

    def factory(**kwargs):
        angle = 0.15
        return IceFlowConfig(
            nx=nx, ny=ny, nz=nz, domain_size_m=(nx * 1e-3, ny * 1e-3, nz * 1e-3), boundary_cells=1,
            water_width=5, water_height=8, floor_water_depth_cells=4, phase_warmup_steps=0,
            ice_bodies=(IceBodyConfig((9.0, 5.5, 0.5 * nz), (4, 4, 4), (np.cos(angle), 0.0, np.sin(angle), 0.0)),),
            **kwargs)

    return factory


@pytest.mark.parametrize("kernel", ["forces", "stream", "collide_stream"])
@pytest.mark.parametrize("shape", SHAPES)
def test_tiled_kernel_matches_oracle(kernel, shape):
    run, outputs = KERNELS[kernel]
    sim, ref = prepared(tank(*shape), seed=sum(shape))
    run(ref)
    run(sim)
    for name in outputs:
        assert_close(getattr(sim, name).to_numpy(), getattr(ref, name).to_numpy(), 2e-5, f"{kernel}:{name}")


@pytest.mark.parametrize("shape", SHAPES)
def test_fused_water_update_equals_its_three_passes(shape):
    """The step's remap, advection and remap in one pass give the water planes
    and the remap energy of the three passes: the same expressions, with FMA
    contraction chosen per kernel (2 FP32 ulps of scale; the remap energy's
    sum over N cells in another order: sqrt(N) ulps of the largest energy for
    the terms and 4 ulps of the sum for its two partial and two final adds).
    The phase moves by a cell so that cells dry out and newly wet, and the
    velocity is strong enough that the advection empties some."""
    from tests.cases3d import restore_fields, snapshot_fields

    sim, _ = prepared(tank(*shape), seed=7 + sum(shape))
    rng = np.random.default_rng(3)
    phi = np.roll(sim.water_phase.to_numpy(), 1, axis=1)
    phi[rng.random(phi.shape) < 0.02] = 1.1e-3
    sim.water_phase.from_numpy(phi * (sim.solid_body_id.to_numpy() == -1))
    u = sim.velocity_lattice.to_numpy()
    sim.velocity_lattice.from_numpy(150.0 * u)
    saved = snapshot_fields(sim)
    dt = sim.scales.dt_s
    sim.remap_energy[None] = 0.0
    sim._synchronize_water_fused()
    sim._advect_water(dt)
    emptied = (sim.water_volume.to_numpy() <= 1e-30) & (phi > 1e-3) & (sim.solid_body_id.to_numpy() == -1)
    sim._synchronize_water_fused()
    expected = {name: getattr(sim, name).to_numpy() for name in ("water_volume", "water_energy")}
    remap = float(sim.remap_energy[None])
    restore_fields(sim, saved)
    sim.remap_energy[None] = 0.0
    sim._remap_advect_remap(dt)
    assert emptied.any()
    np.testing.assert_array_equal(sim.water_volume.to_numpy(), expected["water_volume"])
    got, value = sim.water_energy.to_numpy(), expected["water_energy"]
    assert np.abs(got - value).max() <= 2.0 ** -22 * np.abs(value).max()
    assert abs(float(sim.remap_energy[None]) - remap) <= 2.0 ** -23 * (np.sqrt(value.size) * np.abs(value).max()
                                                                      + 4.0 * abs(remap))


@pytest.mark.parametrize("shape,box", [((18, 516, 520), ((0, 5, 400), (18, 40, 520))),
                                       ((24, 516, 330), ((3, 480, 0), (21, 516, 70))),
                                       ((24, 13, 20), ((5, 0, 3), (12, 13, 20)))])
def test_gradient_sweep_lengths(shape, box):
    """A full pass sweeps 16, 8 and 4 slabs a block on these grids, the pass
    over the box 4: the same stencil at the same cells, so the same bits."""
    import torch

    from projecticy_amd._native import int3
    from projecticy_amd.iceflow3d import IceFlow3D

    sim = IceFlow3D(tank(*shape)())
    torch.manual_seed(5)
    phi = sim._t["phi"]
    phi.copy_(torch.rand(phi.shape, device=phi.device) * (sim._t["id"] == -1))
    sim._call("gradients", None, None)
    grad = sim._t["grad"]
    full = grad.clone()
    inside = tuple(slice(a, b) for a, b in zip(*box))
    grad[(slice(None), *inside)] = 7.0
    sim._call("gradients", int3(box[0]), int3(box[1]))
    assert full.abs().max() > 0.1
    assert torch.equal(grad, full)
