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
