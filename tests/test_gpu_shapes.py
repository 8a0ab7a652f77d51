"""The launch shapes an untuned sim takes (by the grid's size, scheme and precision) and every
strip height of the row march give the plain path's bits, on an MI355X: grids from two cells an
axis to past a tile's edge, one and several chunks of planes, periodic and walled. Bit for bit, so
there is no tolerance."""
import numpy as np
import pytest

from shaderous_amd import amr_tree, problems
from shaderous_amd.amr import AmrSim
from shaderous_amd.ensemble import Ensemble
from shaderous_amd.sim import Sim, SimConfig, config_for

pytestmark = pytest.mark.gpu


def random_flow(n, bc, limiter, seed=1):
    rng = np.random.default_rng(seed)
    shape = n[::-1]
    return problems.Problem(id="random", n=n, box=1.0, gamma=1.4, bc_lo=bc, bc_hi=bc, cfl=0.3, limiter=limiter,
                            isentropic=limiter == "koren",
                            prims={"rho": 1 + 0.3 * rng.random(shape), "vx": 0.5 * rng.normal(size=shape),
                                   "vy": 0.5 * rng.normal(size=shape), "p": 1 + 0.5 * rng.random(shape),
                                   "vz": 0.5 * rng.normal(size=shape) if n[2] > 1 else np.zeros(shape),
                                   "s": rng.random(shape)})


def runs_alike(pb, precision, steps=3, **fused):
    out = []
    for path, over in (("plain", {}), ("fused", fused)):
        with Sim(config_for(pb, path=path, precision=precision, **over)) as sim:
            sim.set_state(*pb.state(np.float64 if precision == 64 else np.float32))
            sim.step(steps)
            out.append((*sim.read_state(), sim.clock()))
    return all(np.array_equal(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("limiter", ["mc", "koren"])
@pytest.mark.parametrize("n,bc", [((2, 2, 2), (0, 0, 0)), ((3, 17, 2), (0, 0, 0)), ((33, 16, 5), (0, 0, 0)),
                                  ((16, 33, 67), (2, 1, 1)), ((70, 15, 9), (1, 2, 0)), ((5, 4, 40), (2, 2, 2)),
                                  ((64, 48, 30), (0, 0, 1)), ((2, 5, 1), (0, 0, 0)), ((17, 61, 1), (1, 2, 0)),
                                  ((260, 130, 1), (2, 1, 0))])
def test_untuned_shapes_give_the_plain_bits(n, bc, limiter, precision):
    assert runs_alike(random_flow(n, bc, limiter), precision)


@pytest.mark.parametrize("rows", [1, 5, 13, 64])
@pytest.mark.parametrize("bc", [(0, 0, 0), (2, 1, 0)])
def test_strips_of_any_height_give_the_plain_bits(rows, bc):
    assert runs_alike(random_flow((130, 61, 1), bc, "koren"), 32, tile=(60, rows, 1))


def test_runs_of_steps_of_an_ensemble_equal_single_steps():
    """A run of steps in one call goes out eight, two and one to a graph: the single steps' bits."""
    cfg = SimConfig(n=(64, 64, 1), ndim=2, dx=1.0 / 64, gamma=1.4, bc_lo=(1, 1, 0), bc_hi=(1, 1, 0), limiter="mc",
                    isentropic=False, cfl=0.4)
    out = []
    for counts in ((19, 3), (1,) * 22):
        ens = Ensemble(cfg, [(64, 64), (100, 37)])
        for i, n in enumerate((64, 100)):
            pb = problems.riemann_quadrants(n, 7 + i)
            u1, u2 = pb.state()
            cells = (64 * 64, 100 * 37)[i]
            ens.set_state(i, u1[:cells], u2[:cells])
        for c in counts:
            ens.step(c)
        out.append([ens.read_state(i) for i in range(2)])
        ens.destroy()
    for a, b in zip(*out):
        assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("cells,levels,walls", [((3, 3, 3), 0, False), ((8, 8, 7), 0, False), ((8, 8, 8), 0, True),
                                                ((4, 4, 4), 2, True), ((8, 8, 8), 2, False)])
def test_march_queue_equals_passes_bitwise(cells, levels, walls, precision):
    """The fused march's queue on meshes of one round and several, whose last round holds single
    blocks or pairs, with leaves that wait for finer ones at two levels: the passes' bits."""
    if levels:
        blocks, dx0, prim = problems.amr_blast(seed=3, root=cells[0], max_level=levels)[:3]
    else:
        blocks = np.array([(0, x, y, z) for z in range(cells[2]) for y in range(cells[1]) for x in range(cells[0])],
                          dtype=np.int32)
        prim = problems.amr_blast(seed=3, root=4, max_level=0)[2]
        dx0 = 1 / (16 * cells[0])
    u1, u2 = amr_tree.blocks_state(blocks, dx0, prim, 1.4, ndim=3)
    bc = (2, 1, 0) if walls else (0, 0, 0)
    cfg = SimConfig(n=tuple(16 * c for c in cells), dx=dx0, gamma=1.4, cfl=0.4, bc_lo=bc, bc_hi=bc, limiter="mc",
                    isentropic=False, precision=precision)
    t = np.float64 if precision == 64 else np.float32
    out = []
    for path in ("passes", "fused"):
        sim = AmrSim(cfg, blocks, cells, path=path)
        sim.set_state(u1.astype(t), u2.astype(t))
        sim.step(3)
        out.append((*sim.read_state(), sim.clock()))
        sim.destroy()
    leaves = np.repeat(amr_tree.leaf_mask(blocks), 4096)
    assert np.all(np.isfinite(out[0][0]))
    for a, b in zip(out[0][:2], out[1][:2]):
        assert np.array_equal(a.reshape(-1, 4)[leaves], b.reshape(-1, 4)[leaves])
    assert np.array_equal(out[0][2], out[1][2])


@pytest.mark.parametrize("scheme", [("mc", False, "hllc"), ("koren", True, "hllc"), ("vanleer", False, "hll"),
                                    ("koren", False, "hll")])
@pytest.mark.parametrize("root,levels,bc,compensated", [((4, 4, 1), 2, (0, 0, 0), True), ((4, 4, 1), 2, (2, 2, 0), False),
                                                        ((8, 8, 1), 3, (0, 1, 0), True), ((8, 8, 1), 1, (1, 2, 0), True),
                                                        ((1, 1, 1), 0, (0, 0, 0), True), ((3, 2, 1), 0, (1, 3, 0), True),
                                                        ((5, 5, 1), 2, (0, 0, 0), True)])
def test_flat_blocks_step_equals_the_passes_bitwise(root, levels, bc, compensated, scheme):
    """The batched step of 2D blocks (ghosts, then the rest in one kernel) against the passes run
    level by level: periodic, walled and outflow, faces on coarser and refined leaves."""
    if levels:
        blocks, dx0 = problems.kh_adaptive(root=root[0], max_level=levels)[:2]
    else:
        blocks = np.array([(0, x, y, 0) for y in range(root[1]) for x in range(root[0])], dtype=np.int32)
        dx0 = 1 / (16 * root[0])
    blocks = np.asarray(blocks, np.int32)
    rng = np.random.default_rng(5)

    def prims(x, y, z):
        return {"rho": 1 + 0.4 * np.sin(7 * x + 3 * y) + 0.1 * rng.random(x.shape), "vx": 0.5 * np.cos(5 * y) + 0 * x,
                "vy": 0.4 * np.sin(6 * x) + 0.05 * rng.random(x.shape), "vz": 0.1 * np.sin(4 * x) + 0 * y,
                "p": 1 + 0.5 * rng.random(x.shape), "s": rng.random(x.shape)}
    u1, u2 = amr_tree.blocks_state(blocks, dx0, prims, 1.4, ndim=2)
    limiter, isen, riemann = scheme
    cfg = SimConfig(n=(16 * root[0], 16 * root[1], 1), ndim=2, dx=dx0, gamma=1.4, cfl=0.4, bc_lo=bc, bc_hi=bc,
                    limiter=limiter, isentropic=isen, riemann=riemann)
    out = []
    for path in ("levels", "passes"):
        sim = AmrSim(cfg, blocks, root, path=path, compensated=compensated)
        sim.set_state(u1, u2)
        sim.step(4)
        out.append((*sim.read_state(), sim.clock()))
        sim.destroy()
    leaves = np.repeat(amr_tree.leaf_mask(blocks), 256)
    assert np.all(np.isfinite(out[0][0].reshape(-1, 4)[leaves]))
    for a, b in zip(out[0][:2], out[1][:2]):
        assert np.array_equal(a.reshape(-1, 4)[leaves], b.reshape(-1, 4)[leaves])
    assert np.array_equal(out[0][2], out[1][2])
