"""Faces whose star densities are not positive, on an MI355X against the FP64 oracle: gas so cold and
dense that a side's sound speed is below the rounding of its velocity, moving apart through the
cells' faces (riemann falls back to the HLL state there). One step along x, y (the flat kernels) and z
(the 3D march); the tolerance is that of test_gpu_riemann.py."""
import numpy as np
import pytest

from shaderous_amd import problems
from shaderous_amd.sim import Sim, config_for

oracle = pytest.importorskip("oracle")
from oracle import params, wgsl64  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_cold_faces_match_the_oracle(axis):
    # sound speed sqrt(1.4e-14 / 1e20) = 1.2e-17, half an ulp of 1 is 5.6e-17
    rho = np.repeat([1e20, 2e20, 1e20, 4e20, 3e20, 1e20], 3)
    vn = np.repeat([-1.0, 1.0, -1.0, 1.0, 0.75, 1.25], 3)
    assert (vn - np.sqrt(1.4e-14 / rho) == vn).all()
    n = [20, 20, 20] if axis == 2 else [20, 20, 1]
    n[axis] = len(rho)
    shape = [1, 1, 1]
    shape[2 - axis] = len(rho)
    full = tuple(n[::-1])
    at = [np.broadcast_to(v.reshape(shape), full).copy() for v in (rho, vn)]
    pr = {"rho": at[0], "p": np.full(full, 1e-14), "s": np.ones(full)}
    for a, k in enumerate(("vx", "vy", "vz")):
        pr[k] = at[1] if a == axis else np.zeros(full)
    bc = [0, 0, 0]
    bc[axis] = 1
    pb = problems.Problem(id="cold", n=tuple(n), box=n[0] / 64.0, gamma=1.4, bc_lo=tuple(bc), bc_hi=tuple(bc),
                          limiter="mc", isentropic=False, cfl=0.3, prims=pr)
    cfg = config_for(pb, precision=64)
    prm = params(pb.n, ndim=cfg.ndim, dx=cfg.dx, gamma=cfg.gamma, cfl=cfg.cfl, limiter="mc", isentropic=False,
                 bc_lo=cfg.bc_lo, bc_hi=cfg.bc_hi)
    u1, u2 = pb.state(np.float64)
    o1, o2, clk = u1.copy(), u2.copy(), np.zeros(4)
    wgsl64.step(prm, o1, o2, clk)
    assert np.isfinite(o1).all() and not np.array_equal(o1, u1)
    for path in ("fused", "plain"):
        with Sim(config_for(pb, precision=64, path=path)) as sim:
            sim.set_state(u1, u2)
            sim.step(1)
            g1, g2 = sim.read_state()
        assert np.abs(g1 - o1).max() <= 1e-11 * np.abs(o1).max()
        assert np.abs(g2 - o2).max() <= 1e-11 * np.abs(o2).max()
