"""Cycles of per-block timesteps keep their values to the bit: eight cycles of eight substeps of a
blast in gas at rest, refined twice, against recorded checksums (golden/bins_cycles.json: per leaf
the CRC-32 of its cells, and the clock). The scheme's shock flag takes the sign of velocity
differences at the rounding level there (beside coarser blocks, where a neighbour is an empty edge
texel), so arithmetic that is equal up to rounding gives states up to 1e-5 apart and cells up to
3e-3: there is no tolerance between the bits and that. The inputs are multiples of 1/1024 from
integer draws, the same on every host.

``python tests/test_gpu_bins_pinned.py FILE`` records what the library gives."""
import json
import os
import sys
import zlib

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

from shaderous_amd import amr_tree  # noqa: E402
from shaderous_amd.amr import AmrSim  # noqa: E402
from shaderous_amd.sim import SimConfig  # noqa: E402

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "bins_cycles.json")
# (dimensions, precision, limiter, Riemann solver, compensated means)
CASES = [(3, 32, "mc", "hllc", True), (3, 32, "koren", "hllc", False), (3, 32, "minmod", "hll", True),
         (3, 64, "mc", "hllc", True), (2, 32, "koren", "hllc", True), (2, 32, "vanleer", "hllc", False),
         (2, 64, "koren", "hllc", True)]


def cycles(ndim, precision, limiter, riemann, compensated):
    root = (2, 2, 2) if ndim == 3 else (3, 3, 1)
    n = 16 * root[0]

    def refine(level, c):
        # the blocks that meet a ball of radius 0.2 about a point off the box's centre
        h = 1.0 / (root[0] << level)
        gap = [max(c[a] * h - 0.45, 0.45 - (c[a] + 1) * h, 0.0) for a in range(ndim)]
        return sum(g * g for g in gap) < 0.04 / (1 << level)

    blocks = amr_tree.build_tree(root, 2, refine, ndim=ndim)
    rng = np.random.default_rng(5)

    def blast(x, y, z):
        hot = (x + 0.05) ** 2 + (y + 0.05) ** 2 + (z + 0.05) ** 2 * (ndim == 3) < 0.02
        return {"rho": 1.0 + rng.integers(0, 8, x.shape) / 1024, "p": np.where(hot, 16.0, 0.125),
                "s": rng.integers(0, 1024, x.shape) / 1024}

    dtype = np.float64 if precision == 64 else np.float32
    u1, u2 = amr_tree.blocks_state(blocks, 1.0 / n, blast, 1.5, dtype, ndim=ndim)
    cfg = SimConfig(n=(n, n, n if ndim == 3 else 1), ndim=ndim, dx=1.0 / n, gamma=1.5, cfl=0.4, limiter=limiter,
                    riemann=riemann, isentropic=limiter == "koren", precision=precision)
    sim = AmrSim(cfg, blocks, root, path="passes", compensated=compensated, time_bins=3)
    try:
        sim.set_state(u1, u2)
        sim.step(64)
        g1, g2 = sim.read_state()
        work = sim.bins()[1]
        clock = [float(v).hex() for v in sim.clock()[:4]]
    finally:
        sim.destroy()
    assert work["cycles"] == 8 and work["updates"] < work["single"]
    leaf = np.flatnonzero(amr_tree.leaf_mask(blocks))
    g1, g2 = g1.reshape(len(blocks), -1), g2.reshape(len(blocks), -1)
    return {"clock": clock, "leaves": [zlib.crc32(g2[b].tobytes(), zlib.crc32(g1[b].tobytes())) for b in leaf]}


def key(case):
    return "-".join(str(v) for v in case)


@pytest.mark.parametrize("case", CASES, ids=key)
def test_cycles_keep_their_bits(case):
    with open(GOLDEN) as f:
        want = json.load(f)[key(case)]
    got = cycles(*case)
    assert got["clock"] == want["clock"]
    bad = [i for i, (a, b) in enumerate(zip(got["leaves"], want["leaves"])) if a != b]
    assert len(got["leaves"]) == len(want["leaves"]) and not bad, f"leaves {bad} of {len(want['leaves'])} differ"


if __name__ == "__main__":
    with open(sys.argv[1], "w") as f:
        json.dump({key(c): cycles(*c) for c in CASES}, f, separators=(",", ":"))
