"""GPU parity of a rebuild inside the step loop (ghosts, cells, lists made
from the cell-ordered mirrors in one pass without a host round trip) against
the CPU oracle, at the sizes where its launches change shape: a single block
of locals, whole and ragged blocks, class counts scanned by the emitting
blocks or by launches of their own, grids whose tiles are counted by the sort
or by a launch of their own, and more ghosts than there was room for."""
import numpy as np
import pytest

import pyoracle as po
from common import RC, SKIN, announce, make_pair, perturbed_fcc

pytestmark = pytest.mark.gpu

DT = 0.005


@pytest.fixture(scope="module")
def tm():
    import tinymd_amd
    _, cus = tinymd_amd.device_info()
    if cus == 0:
        pytest.fail("no HIP device visible to libtinymd_amd")
    return tinymd_amd


def same_structure(sim, orc):
    """Ghost table, cells and lists entry for entry."""
    assert sim.nghost == orc.ng
    gt, go = sim.ghost_table(), orc.ghosts()
    for key in ("owner", "img", "src", "flag"):
        assert np.array_equal(gt[key], go[key]), key
    st, parts, pcell = sim.cells()
    so, po_, pco = orc.cells()
    assert np.array_equal(st, so) and np.array_equal(parts, po_) and np.array_equal(pcell, pco)
    cg, lg = sim.neighbor_lists()
    co, lo = orc.neighbor_lists()
    assert np.array_equal(cg, co)
    m = min(lg.shape[1], lo.shape[1])
    cols = np.arange(m)[None, :] < cg[:, None]
    assert np.array_equal(np.where(cols, lg[:, :m], -1), np.where(cols, lo[:, :m], -1))


# (4, 4, 4): 256 atoms, one block; (5, 4, 7): ragged; (20, 20, 25):
# 157 blocks, the most whose counts the blocks scan themselves; 22^3: 167
@pytest.mark.parametrize("shape", [(4, 4, 4), (5, 4, 7), (8, 8, 4), (20, 20, 25), (22, 22, 22)])
def test_rebuild_in_loop_exact(tm, shape):
    announce(f"rebuild in the loop {shape}")
    aabb, m, x, v = perturbed_fcc(*shape, amp=0.05, seed=11)
    sim, orc = make_pair(aabb, m, x, v)
    sim.setup(False, RC, SKIN)
    orc.setup(False, po.HALF_GHOST_FULL, RC + SKIN)
    same_structure(sim, orc)
    sim.lennard_jones(False, RC)
    orc.lj(False, RC)
    # the second rebuild starts from the first one's mirrors
    sim.run_lj(45, 20, DT)
    orc.run_lj(45, 20, DT)
    same_structure(sim, orc)
    _, xg, vg, fg = sim.state()
    xo, vo, fo = orc.state()
    assert np.array_equal(xg, xo) and np.array_equal(vg, vo) and np.array_equal(fg, fo)


def test_rebuild_sparse_grid_dem(tm):
    """A grid of 35,937 cells for 28,000 spheres: a thread per cell sorts,
    tiles are counted by their own launch; ghost velocities and the ghost
    index follow the rebuilds.  Contact forces differ from the oracle's by
    summation rounding only."""
    announce("rebuild, sparse DEM grid")
    nc = 24
    m, x, v = tm.generate_granular_gas(nc, vmax=3.0)
    L = nc * 1.6796
    aabb = np.array([0.0, L] * 3)
    sim = tm.Simulation(m, x, v, aabb, 1.3, dem_radius=0.5)
    sim.copy_to_accelerator()
    orc = po.OracleSim(m, x, v, aabb, 1.3, threads=4)
    sim.setup(True, 1.0, 0.3)
    orc.setup(True, po.HALF_GHOST_FULL, 1.3)
    assert sim.grid_info()["ncells"] > 16384
    sim.dem(True, 1.0)
    orc.dem(True, 1.0)
    sim.run_dem(45, 20, 0.001)
    orc.run_dem(45, 20, 0.001)
    gt, go = sim.ghost_table(), orc.ghosts()
    assert sim.nghost == orc.ng
    for key in ("owner", "img", "src", "flag"):
        assert np.array_equal(gt[key], go[key]), key
    _, xg, vg, _ = sim.state()
    xo, vo, _ = orc.state()
    assert np.allclose(xg, xo, rtol=1e-12, atol=1e-12) and np.allclose(vg, vo, rtol=1e-12, atol=1e-12)


def test_ghosts_outgrow_their_room(tm):
    """A sheet of three layers that drifts from 4 to 0.5 cells' lengths of the
    lower x face between two rebuilds: 1.5 ghosts an atom where the volume of
    the shell made room for 0.5 (and 4,096), so the rebuild in the loop has to
    grow its arrays and repeat.  Bit for bit the oracle's."""
    announce("ghosts outgrow their room")
    L, ny = 48.0, 43
    a = L / ny
    g = np.arange(ny) * a
    z, y, k = np.meshgrid(g, g, np.arange(3), indexing="ij")
    x = np.stack([4.0 + 1.1 * k.ravel(), y.ravel(), z.ravel()], axis=1)
    rng = np.random.default_rng(3)
    v = rng.normal(0.0, 0.3, x.shape)
    v[:, 0] -= 35.0
    aabb = np.array([0.0, L] * 3)
    m = np.ones(len(x))
    room = 1.25 * len(x) * ((1 + 5.6 / L) ** 3 - 1) + 4096
    sim, orc = make_pair(aabb, m, x, v)
    sim.setup(False, RC, SKIN)
    orc.setup(False, po.HALF_GHOST_FULL, RC + SKIN)
    assert sim.nghost == orc.ng < room
    sim.lennard_jones(False, RC)
    orc.lj(False, RC)
    sim.run_lj(22, 20, DT)
    orc.run_lj(22, 20, DT)
    assert orc.ng > room
    same_structure(sim, orc)
    _, xg, vg, fg = sim.state()
    xo, vo, fo = orc.state()
    assert np.array_equal(xg, xo) and np.array_equal(vg, vo) and np.array_equal(fg, fo)


# threads 64: lanes that own several atoms; (4, 4, 4): the smallest box, up to seven
# images of an atom; 45 steps: two rebuilds, whose ghost index the
# steps after them use
@pytest.mark.parametrize("precision", ["fp64", "fp32mixed"])
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("shape,threads", [((4, 4, 4), 0), ((9, 4, 5), 64), ((13, 11, 12), 0)])
def test_step_pass_writes_ghosts(tm, shape, threads, half, precision):
    """A step whose force pass also drifts the atoms and their ghosts against
    the separate calls: the same operations, so bit for bit."""
    announce(f"step pass with ghosts {shape} {threads} {half} {precision}")
    aabb, m, x, v = perturbed_fcc(*shape, amp=0.05, seed=5)
    out = []
    for run in ("run_lj", "run_abi_lj"):
        sim = tm.Simulation(m, x, v, aabb, RC + SKIN, precision=precision)
        if threads:
            sim.set_tile(3, 2, 2, threads)
        sim.copy_to_accelerator()
        sim.setup(half, RC, SKIN)
        sim.lennard_jones(half, RC)
        getattr(sim, run)(45, 20, DT, half)
        out.append(sim.state()[1:] + tuple(sim.ghost_state()[:2]))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


# lattice 0.7: a quarter of the list cutoff, so whole shells of pairs lie at
# the cutoff to the last bit and FP32 decides none of them; gas of 40 atoms a
# cell: most of a chunk's candidates accepted at once; thin gas: empty chunks;
# window of 6 x 6 x 6 cells of 40: larger than the LDS
@pytest.mark.parametrize("half,literal", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("atoms,tile", [("lattice", (2, 1, 1)), ("gas", (1, 2, 1)), ("gas", (4, 4, 4)), ("thin", (3, 3, 3))])
def test_lists_exact_at_the_cutoff(tm, atoms, tile, half, literal):
    announce(f"lists at the cutoff, {atoms} {tile} {half} {literal}")
    rng = np.random.default_rng(7)
    if atoms == "lattice":
        L = 0.7 * 18
        g = (np.arange(18) + 0.5) * 0.7
        x = np.stack(np.meshgrid(g, g, g, indexing="ij"), axis=-1).reshape(-1, 3)
    else:
        L = 2.8 * 4.4
        x = rng.random((3400 if atoms == "gas" else 60, 3)) * L
    aabb = np.array([0.0, L] * 3)
    mode = "ref_literal" if literal else "ghost_full"
    sim = tm.Simulation(np.ones(len(x)), x, np.zeros_like(x), aabb, RC + SKIN, nb_cap=400, half_mode=mode)
    sim.set_tile(*tile)
    sim.copy_to_accelerator()
    sim.setup(half, RC, SKIN)
    orc = po.OracleSim(np.ones(len(x)), x, np.zeros_like(x), aabb, RC + SKIN, nb_cap=400, threads=4)
    orc.setup(half, po.HALF_REF_LITERAL if literal else po.HALF_GHOST_FULL, RC + SKIN)
    same_structure(sim, orc)


# 6,912 and 7,200 atoms: either side of FP32-mixed's line for four lanes an
# atom, 10,976 and 11,760 of the others'; (4, 4, 5): fewer atoms a tile than
# one wavefront's 16; cutoffs 1.2 and 3: lists within one round of 16 entries and
# over several fetches of 32
@pytest.mark.parametrize("shape,rc,half,precision,par", [
    ((4, 4, 5), 2.5, False, "fp64", (1.0, 1.0, True)),
    ((4, 4, 5), 1.2, True, "fp32mixed", (1.0, 1.0, False)),
    ((7, 6, 8), 3.0, True, "fp64", (1.3, 0.9, False)),
    ((7, 6, 8), 3.0, False, "fp32mixed", (1.3, 0.9, True)),
    ((7, 6, 8), 3.0, True, "fp32kahan", (0.8, 1.1, True)),
    ((7, 6, 8), 2.5, False, "fp32kahan", (1.0, 1.0, False)),
    ((12, 12, 12), 2.5, False, "fp32mixed", (1.0, 1.0, False)),
    ((12, 15, 10), 2.5, False, "fp32mixed", (1.0, 1.0, False)),
    ((14, 14, 14), 2.5, True, "fp64", (1.0, 1.0, False)),
    ((14, 15, 14), 2.5, True, "fp64", (1.0, 1.0, False)),
])
def test_lanes_of_an_atom(tm, shape, rc, half, precision, par):
    """The step pass of small boxes against the separate calls: bit for bit."""
    announce(f"lanes of an atom {shape} {rc} {half} {precision} {par}")
    eps, sigma, shift = par
    aabb, m, x, v = perturbed_fcc(*shape, amp=0.03, seed=5)
    out = []
    for run in ("run_lj", "run_abi_lj"):
        sim = tm.Simulation(m, x, v, aabb, rc + SKIN, precision=precision, lj_shift=shift)
        sim.copy_to_accelerator()
        sim.setup(half, rc, SKIN)
        sim.lennard_jones(half, rc, eps, sigma)
        getattr(sim, run)(25, 10, 0.002, half, rc, SKIN, eps, sigma)
        out.append(sim.state()[1:] + tuple(sim.ghost_state()[:2]))
    for a, b in zip(*out):
        assert np.array_equal(a, b)


# one-cell tiles, ordered over the reached part of the grid (layers beyond it
# on all sides, on x and y, on z) or dealt in runs (with such layers on x and
# y, with none), against few tiles in their plain order
@pytest.mark.parametrize("shape", [(15, 10, 20), (16, 15, 14), (14, 14, 20), (15, 15, 22), (14, 12, 22)])
@pytest.mark.parametrize("half", [False, True])
def test_order_of_the_tiles(tm, shape, half):
    """The order of the blocks changes no bit."""
    announce(f"order of the tiles {shape} {half}")
    aabb, m, x, v = perturbed_fcc(*shape, amp=0.05, seed=7)
    out = []
    for tile in (1, 5):
        sim = tm.Simulation(m, x, v, aabb, RC + SKIN)
        sim.set_tile(tile)
        sim.copy_to_accelerator()
        sim.setup(half, RC, SKIN)
        sim.lennard_jones(half, RC, 1.0, 1.0)
        sim.run_lj(25, 10, 0.005, half, RC, SKIN, 1.0, 1.0)
        out.append(sim.state()[1:])
    for a, b in zip(*out):
        assert np.array_equal(a, b)


# spheres a cell of 1.3: lists of about 2 (one group or none), 8 (either side
# of a group), 20 and 45 entries (several rounds of two groups, most of them in
# contact); one tile shape whose blocks hold more locals than threads
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("n,tile", [(700, None), (2600, None), (6500, (2, 2, 2)), (14500, (3, 2, 2))])
def test_dem_step_pass_dense_lists(tm, n, tile, half):
    """Overlapping spheres at random against the oracle, which sums in another
    order: rounding of up to 50 terms below 100 a force, 2e-12, times a time
    step of 1e-4."""
    announce(f"DEM step pass {n} {tile} {half}")
    rng = np.random.default_rng(n)
    L = 1.3 * 11.3
    x, v = rng.random((n, 3)) * L, rng.normal(0.0, 0.3, (n, 3))
    m, aabb = np.ones(n), np.array([0.0, L] * 3)
    sim = tm.Simulation(m, x, v, aabb, 1.3, dem_radius=0.5, nb_cap=160)
    if tile:
        sim.set_tile(*tile, 64)
    sim.copy_to_accelerator()
    orc = po.OracleSim(m, x, v, aabb, 1.3, nb_cap=160, threads=4)
    sim.setup(half, 1.0, 0.3)
    orc.setup(half, po.HALF_GHOST_FULL, 1.3)
    sim.dem(half, 1.0)
    orc.dem(half, 1.0)
    sim.run_dem(7, 3, 1e-4, half)
    orc.run_dem(7, 3, 1e-4, half)
    _, xg, vg, fg = sim.state()
    xo, vo, fo = orc.state()
    assert np.allclose(xg, xo, rtol=1e-13, atol=1e-13) and np.allclose(vg, vo, rtol=1e-13, atol=1e-13)
    assert np.allclose(fg, fo, rtol=1e-12, atol=2e-12 * max(1.0, np.abs(fo).max() / 100.0))


# a rebuild inside the loop, from the mirrors and, at the first step, from atom
# order
@pytest.mark.parametrize("dem", [False, True])
@pytest.mark.parametrize("reneigh", [5, 1])
def test_atom_lost_in_the_loop(tm, dem, reneigh):
    """An atom that leaves the box by many lengths before a rebuild: an error,
    after which the locals, the lost one too, are as they were at that rebuild,
    wrapped, bit for bit as the separate calls leave them."""
    announce(f"atom lost in the loop dem={dem} {reneigh}")
    if dem:
        m, x, v = tm.generate_granular_gas(9, vmax=2.0)
        aabb, rc, dt = np.array([0.0, 9 * 1.6796] * 3), 1.0, 0.001
    else:
        aabb, m, x, v = perturbed_fcc(6, amp=0.05, seed=5)
        rc, dt = RC, DT
    v = v.copy()
    v[len(x) // 2] = 1e6

    def force(sim):
        sim.dem(True, rc) if dem else sim.lennard_jones(False, rc)

    def make():
        sim = tm.Simulation(m, x, v, aabb, rc + SKIN, dem_radius=0.5 if dem else None)
        sim.copy_to_accelerator()
        sim.setup(dem, rc, SKIN)
        force(sim)
        return sim

    ref = make()
    for j in range(reneigh):
        ref.initial_integration(dt)
        if j + 1 < reneigh:
            ref.synchronize_ghost_layer()
            force(ref)
            ref.final_integration(dt)
    ref.enforce_pbc()
    _, xr, vr, _ = ref.state()
    sim = make()
    with pytest.raises(tm.TinyMDError, match="outside the periodic box"):
        sim.run_dem(9, reneigh, dt) if dem else sim.run_lj(9, reneigh, dt)
    tm.load().tmd_clear_error()
    _, xs, vs, _ = sim.state()
    assert np.array_equal(xs, xr) and np.array_equal(vs, vr)
    sim.close()


@pytest.mark.parametrize("shape", [(4, 4, 5), (11, 9, 10), (17, 16, 18)])
def test_without_a_ghost_index(tm, shape):
    """With room for more ghosts than the index numbers (2^26; here for any),
    each step's ghosts follow in a pass of their own: bit for bit the same step
    loops and gradients."""
    announce(f"without a ghost index {shape}")
    out = []
    for limit in (0, 1):
        aabb, m, x, v = perturbed_fcc(*shape, amp=0.05, seed=5)
        res = []
        for half, precision in ((False, "fp32mixed"), (True, "fp64")):
            sim = tm.Simulation(m, x, v, aabb, RC + SKIN, precision=precision)
            tm.load().tmd_set_ghost_index_limit(limit)
            sim.copy_to_accelerator()
            sim.setup(half, RC, SKIN)
            sim.lennard_jones(half, RC)
            sim.run_lj(25, 10, DT, half)
            res += list(sim.state()[1:]) + list(sim.ghost_state()[:2])
        sim = tm.Simulation(m, x, v, aabb, RC + SKIN, lj_shift=True)
        tm.load().tmd_set_ghost_index_limit(limit)
        sim.copy_to_accelerator()
        r = sim.traj_adjoint(13, 5, DT, RC, SKIN, 1.0, 1.0, -4.0, 1.0)
        res += [r[key] for key in ("ubar", "pbar", "grad_eps", "grad_sigma", "grad_x0", "grad_v0")]
        m, x, v = tm.generate_granular_gas(shape[0], vmax=2.0)
        sim = tm.Simulation(m, x, v, np.array([0.0, shape[0] * 1.6796] * 3), 1.3, dem_radius=0.5)
        tm.load().tmd_set_ghost_index_limit(limit)
        sim.copy_to_accelerator()
        sim.setup(True, 1.0, 0.3)
        sim.dem(True, 1.0)
        sim.run_dem(25, 10, 0.001, True)
        res += list(sim.state()[1:]) + list(sim.ghost_state()[:3])
        out.append(res)
        sim.close()
    tm.load().tmd_set_ghost_index_limit(0)
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_larger_tiles_after_smaller_ones(tm):
    """The first list build with larger tiles does not run with the window sizes
    of the smaller ones before: it takes less than twice the next one's time
    (its windows were read from global memory, several times as long)."""
    announce("larger tiles after smaller ones")
    aabb, m, x, v = perturbed_fcc(16, amp=0.05, seed=5)
    sim = tm.Simulation(m, x, v, aabb, RC + SKIN)
    sim.copy_to_accelerator()

    def build(tile):  # ms of the list build that a run begins with
        sim.set_tile(tile)
        sim.profile(True)
        sim.profile_reset()
        sim.run_lj(1, 20, 0.0)
        ms, count = sim.profile_get("neighbor")
        sim.profile(False)
        assert count == 1
        return ms

    first, again = [], []
    for _ in range(5):
        build(1)
        first.append(build(4))
        again.append(build(4))
    print(first, again)
    assert min(first) < 2.0 * min(again), (first, again)
    sim.close()


def test_ghosts_outgrow_their_room_dem(tm):
    """The drifting sheet of spheres: the rebuild inside the DEM loop has to grow
    its arrays and repeat from mirrors that hold the ghosts' velocities too.
    Contact forces differ from the oracle's by summation rounding only."""
    announce("ghosts outgrow their room, DEM")
    L = 76.0
    g = np.arange(76) + 0.5
    z, y, k = np.meshgrid(g, g, np.arange(2), indexing="ij")
    x = np.stack([3.0 + 0.95 * k.ravel(), y.ravel(), z.ravel()], axis=1)
    v = np.random.default_rng(3).normal(0.0, 0.3, x.shape)
    v[:, 0] -= 28.0
    aabb, m = np.array([0.0, L] * 3), np.ones(len(x))
    room = 1.25 * len(x) * ((1 + 2.6 / L) ** 3 - 1) + 4096
    tm.load().md_deallocate_grid()
    sim = tm.Simulation(m, x, v, aabb, 1.3, dem_radius=0.5)
    sim.copy_to_accelerator()
    orc = po.OracleSim(m, x, v, aabb, 1.3, threads=4)
    sim.setup(True, 1.0, 0.3)
    orc.setup(True, po.HALF_GHOST_FULL, 1.3)
    assert sim.nghost == orc.ng < room
    sim.dem(True, 1.0)
    orc.dem(True, 1.0)
    sim.run_dem(110, 100, 0.001)
    orc.run_dem(110, 100, 0.001)
    assert orc.ng > room
    gt, go = sim.ghost_table(), orc.ghosts()
    assert sim.nghost == orc.ng
    for key in ("owner", "img", "src", "flag"):
        assert np.array_equal(gt[key], go[key]), key
    _, xg, vg, _ = sim.state()
    xo, vo, _ = orc.state()
    assert np.allclose(xg, xo, rtol=1e-11, atol=1e-11) and np.allclose(vg, vo, rtol=1e-11, atol=1e-11)
    _, xh, vh, _ = sim.ghost_state()
    assert np.array_equal(vh, vg[gt["owner"]]) and np.array_equal(xh, xg[gt["owner"]] + gt["img"] * L)
    sim.close()


@pytest.mark.parametrize("shape,seed", [((6, 5, 7), 10), ((8, 7, 6), 44), ((8, 7, 6), 53)])
def test_lanes_of_an_atom_compensated_half_lists(tm, shape, seed):
    """Compensated sums over both columns of a half list by four lanes an atom:
    bit for bit the separate calls' (a zero for each absent entry between the
    columns moved these boxes' sums by a rounding now and then)."""
    announce(f"lanes of an atom, compensated {shape} {seed}")
    rng = np.random.default_rng(seed)
    m, x, _ = tm.generate_fcc(*shape)
    L = np.array(shape) * 1.6796
    aabb = np.stack([0.0 * L, L], axis=1).ravel()
    x = np.mod(x + rng.uniform(-0.05, 0.05, x.shape), L)
    v = rng.normal(0.0, 1.2, x.shape)
    out = []
    for run in ("run_lj", "run_abi_lj"):
        sim = tm.Simulation(m, x, v, aabb, RC + SKIN, precision="fp32kahan")
        sim.copy_to_accelerator()
        sim.setup(True, RC, SKIN)
        sim.lennard_jones(True, RC)
        getattr(sim, run)(60, 20, DT, True)
        out.append(sim.state()[1:])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
