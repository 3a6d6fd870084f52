"""2D kernels that leave out what cannot matter: cells beyond the body's
reach take no pose, and the aperture transfer forms its totals from what it
writes.  Against the FP64 oracle's coverage and masks at angles where the
corners reach furthest, and against the two separate entry points.  Kernels
compiled for one population storage against the general ones."""

import math

import numpy as np
import pytest

from cases2d import submerged_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degrees", [0.0, 3.0, 44.0, 45.0])
def test_coverage_and_mask_at_any_angle(degrees):
    from oracle.iceflow2d_oracle import Oracle2D
    from projecticy_amd.iceflow2d import IceFlow2D

    config = submerged_config(ice_initial_angle=math.radians(degrees), phase_warmup_steps=0)
    sim, ref = IceFlow2D(config), Oracle2D(config)
    got, expected = sim._moving_body_fraction.to_numpy(), np.asarray(ref.state()["coverage"])
    # the coverage is formed in FP64 and stored once in FP32
    np.testing.assert_allclose(got, expected, rtol=2.0 ** -22, atol=2.0 ** -24)
    np.testing.assert_array_equal(sim.solid_mask.to_numpy(), np.asarray(ref.state()["solid_mask"]))


def test_transfer_equals_apply_then_finish():
    from projecticy_amd.iceflow2d import IceFlow2D

    results = []
    for calls in (("apply_aperture_transfer", "finish_aperture_transfer"), ("transfer_aperture",)):
        sim = IceFlow2D(submerged_config())
        sim.step(3)
        sim._call("measure_aperture")
        sim._call("build_aperture_targets")
        for name in calls:
            sim._call(name)
        control = sim._read_control()
        results.append((sim.thermal.water_volume_m2.to_numpy(), sim.thermal.water_sensible_energy.to_numpy(),
                        np.array(control.transfer[:])))
    for a, b in zip(*results):  # the same cells' values, summed in the same blocks
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("storage,step", [("fp32", 2.0 ** -24), ("fp16-momentum-sr", 2.0 ** -24),
                                          ("fp16-rel-sr", 2.0 ** -11)])
def test_kernels_compiled_for_a_storage(storage, step):
    """A batch that states its cases' common storage runs kernels compiled
    for it, one that does not the general ones; the two may contract
    differently.  The bound: in each of three steps a phase is the sum of nine
    populations below 1, each off by some roundings (32 allowed) of its
    storage's step."""
    from projecticy_amd.iceflow2d.ensemble import IceFlowEnsemble2D

    phases = []
    for stated in (True, False):
        batch = IceFlowEnsemble2D([submerged_config(), submerged_config()], population_storage=storage,
                                  use_graph=False)
        assert batch._batch.storage == 1 + batch.cases[0]._g.half_populations
        if not stated:
            batch._batch.storage = 0
        batch.step(3)
        phases.append([case.water_phase.to_numpy() for case in batch.cases])
    for a, b in zip(*phases):
        np.testing.assert_allclose(a, b, rtol=0.0, atol=3 * 9 * 32 * step)
