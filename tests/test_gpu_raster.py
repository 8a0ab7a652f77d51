"""The raster form of the 3D march (k_fused): in FP64 on request, and on every plane of 4 GiB or more,
which the role form's 32-bit offsets do not reach; the kernel a sim names is the one it runs."""
import numpy as np
import pytest

from shaderous_amd.sim import Sim, SimConfig, config_for
from test_gpu_shapes import random_flow, runs_alike

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("limiter", ["mc", "koren"])
@pytest.mark.parametrize("n,bc", [((17, 16, 5), (0, 0, 0)), ((16, 33, 40), (2, 1, 1))])
def test_fp64_raster_tile_gives_the_plain_bits(n, bc, limiter):
    pb = random_flow(n, bc, limiter)
    with Sim(config_for(pb, precision=64, tile=(28, 12, 0))) as sim:
        assert sim.kernel_name() == "k_fused"
        assert sim.autotune()[2] == min(32, n[2])
    with Sim(config_for(pb, precision=64)) as sim:
        assert sim.kernel_name() == "k_fused_r"
    assert runs_alike(pb, 64, tile=(28, 12, 0))


@pytest.mark.parametrize("ny,asked,kernel", [(16384, (0, 0, 0), "k_fused"), (16384, (32, 16, 0), "k_fused"),
                                             (16383, (0, 0, 0), "k_fused_r")])
def test_wide_planes_take_the_raster_tile(ny, asked, kernel):
    """16384^2 cells of 16 bytes are 4 GiB (34 GB of state on the device; nothing is stepped)."""
    with Sim(SimConfig(n=(16384, ny, 2), ndim=3, dx=1.0 / 16384, limiter="mc", isentropic=False, tile=asked)) as sim:
        assert sim.kernel_name() == kernel
