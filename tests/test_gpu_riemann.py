"""Every state the face solver tells apart, on an MI355X against the FP64 oracle: supersonic to
either side, the star state left and right of the contact, faces whose star densities are not
positive or whose cells are flagged as shocks (the HLL state), a contact at rest. One step of a
line of cells with those pairs of states side by side, along x and y (the flat kernels) and z (the
3D march); FP64, so that what differs is the order of operations alone: a step's fluxes go through
some tens of roundings of values up to the Mach number squared times the state, here 1e3, and
2.2e-16 * 1e3 * 50 is 1e-11 of the largest value."""
import numpy as np
import pytest

from shaderous_amd import problems
from shaderous_amd.sim import Sim, config_for

oracle = pytest.importorskip("oracle")
from oracle import params, wgsl64  # noqa: E402

pytestmark = pytest.mark.gpu

# (rho, normal velocity, p) of neighbouring cells, in runs of three so that some faces lie between
# equal cells
PAIRS = [(1.0, 0.0, 1.0), (0.125, 0.0, 0.1), (1.0, 8.0, 1.0), (2.0, 30.0, 0.5), (1.0, -12.0, 1.0), (0.5, -0.4, 0.8),
         (1.0, 0.6, 1.1), (0.1, 3.0, 0.02), (1.0, -3.0, 1.0), (4.0, 0.0, 1.0), (1.0, 0.0, 1.0), (1e-3, 2.0, 1e-3),
         (1.0, 1.5, 20.0), (1.0, -1.5, 20.0), (0.3, 0.3, 0.3)]


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("limiter,isen,riemann", [("mc", False, "hllc"), ("koren", True, "hllc")])
def test_every_face_state_matches_the_oracle(axis, limiter, isen, riemann):
    rho, vn, p = (np.repeat([s[k] for s in PAIRS], 3) for k in range(3))
    n = [20, 20, 20] if axis == 2 else [20, 20, 1]
    n[axis] = len(rho)
    shape = [1, 1, 1]
    shape[2 - axis] = len(rho)
    full = tuple(n[::-1])
    pr = {k: np.broadcast_to(v.reshape(shape), full).copy() for k, v in (("rho", rho), ("p", p))}
    for a, k in enumerate(("vx", "vy", "vz")):
        v = vn if a == axis else 0.2 * np.cos(np.arange(len(vn)) + a) * (n[2] > 1 or a < 2)
        pr[k] = np.broadcast_to(np.asarray(v).reshape(shape), full).copy()
    pr["s"] = pr["rho"] ** 0.5
    bc = [0, 0, 0]
    bc[axis] = 1
    pb = problems.Problem(id="faces", n=tuple(n), box=n[0] / 64.0, gamma=1.4, bc_lo=tuple(bc), bc_hi=tuple(bc),
                          limiter=limiter, isentropic=isen, riemann=riemann, cfl=0.3, prims=pr)
    cfg = config_for(pb, precision=64)
    prm = params(pb.n, ndim=cfg.ndim, dx=cfg.dx, gamma=cfg.gamma, cfl=cfg.cfl, limiter=limiter, isentropic=isen,
                 riemann=riemann, bc_lo=cfg.bc_lo, bc_hi=cfg.bc_hi)
    u1, u2 = pb.state(np.float64)
    o1, o2, clk = u1.copy(), u2.copy(), np.zeros(4)
    wgsl64.step(prm, o1, o2, clk)
    for path in ("fused", "plain"):
        with Sim(config_for(pb, precision=64, path=path)) as sim:
            sim.set_state(u1, u2)
            sim.step(1)
            g1, g2 = sim.read_state()
        assert np.abs(g1 - o1).max() <= 1e-11 * np.abs(o1).max()
        assert np.abs(g2 - o2).max() <= 1e-11 * np.abs(o2).max()
