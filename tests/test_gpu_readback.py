"""Reading a state back gives the bytes that were set, on an MI355X: states smaller than one pinned
slot, of exactly one, a little past it and of many, in both precisions; into pinned memory, from
several threads at once, and after a re-mesh to a larger state."""
import ctypes as C
import threading

import numpy as np
import pytest
import torch

from shaderous_amd import _lib, amr_tree, problems
from shaderous_amd.amr import AmrSim
from shaderous_amd.ensemble import Ensemble
from shaderous_amd.sim import Sim, SimConfig

pytestmark = pytest.mark.gpu


def states(ncell, dtype, seed=1):
    rng = np.random.default_rng(seed)
    return [rng.uniform(0.5, 1.5, (ncell, 4)).astype(dtype) for _ in range(2)]


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("n", [(2, 2, 1), (128, 128, 1), (129, 128, 1), (181, 183, 1), (64, 64, 64), (129, 127, 65),
                               (160, 161, 83)])
def test_uniform_state_round_trip(n, precision):
    dtype = np.float64 if precision == 64 else np.float32
    u1, u2 = states(n[0] * n[1] * n[2], dtype)
    with Sim(SimConfig(n=n, ndim=2 if n[2] == 1 else 3, dx=1 / n[0], limiter="mc", isentropic=False,
                       precision=precision)) as sim:
        sim.set_state(u1, u2)
        for _ in range(2):
            got = sim.read_state()
            assert np.array_equal(got[0], u1) and np.array_equal(got[1], u2)
        # several readers at once
        out = [None] * 4

        def read(i):
            out[i] = sim.read_state()
        threads = [threading.Thread(target=read, args=(i,)) for i in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert all(np.array_equal(o[0], u1) and np.array_equal(o[1], u2) for o in out)
        # pinned destinations
        p1, p2 = (torch.empty(u1.shape, dtype=torch.from_numpy(u1).dtype, pin_memory=True) for _ in range(2))
        f = C.POINTER(C.c_double if precision == 64 else C.c_float)
        read_into = _lib.load().shx_read_state_f64 if precision == 64 else _lib.load().shx_read_state
        assert read_into(sim._h, C.cast(p1.data_ptr(), f), C.cast(p2.data_ptr(), f)) == 0
        assert np.array_equal(p1.numpy(), u1) and np.array_equal(p2.numpy(), u2)


def test_ensemble_states_round_trip():
    sizes = [(8, 8), (700, 650), (40, 33), (128, 128)]
    ens = Ensemble(SimConfig(n=(8, 8, 1), ndim=2, limiter="mc", isentropic=False), sizes)
    want = [states(a * b, np.float32, i) for i, (a, b) in enumerate(sizes)]
    for i, w in enumerate(want):
        ens.set_state(i, *w)
    for i, w in enumerate(want):
        got = ens.read_state(i)
        assert np.array_equal(got[0], w[0]) and np.array_equal(got[1], w[1])
    ens.destroy()


def test_blocks_read_after_growing():
    small, dx0, prim = problems.amr_blast(seed=7, root=4, max_level=0)[:3]
    large = problems.amr_blast(seed=7, root=4, max_level=1)[0]
    u1, u2 = amr_tree.blocks_state(small, dx0, prim, 1.4, ndim=3)
    cfg = SimConfig(n=(64, 64, 64), dx=dx0, limiter="mc", isentropic=False)
    sim = AmrSim(cfg, small, (4, 4, 4), path="passes")
    sim.set_state(u1, u2)
    got = sim.read_state()
    assert np.array_equal(got[0].ravel(), u1.ravel()) and np.array_equal(got[1].ravel(), u2.ravel())
    sim.regrid(large)
    assert len(sim.blocks) == len(large) > len(small)
    got = sim.read_state()
    # level-0 leaves keep their cells
    at = {tuple(b): i for i, b in enumerate(np.asarray(large).tolist())}
    keep = amr_tree.leaf_mask(large)
    for i, b in enumerate(np.asarray(small).tolist()):
        j = at[tuple(b)]
        if keep[j]:
            assert np.array_equal(got[0][4096 * j:4096 * (j + 1)], u1.reshape(-1, 4)[4096 * i:4096 * (i + 1)])
    sim.destroy()
