"""Batched replicas on the GPU against the same boxes run one at a time
through the md_* path: each replica's positions, velocities and forces are
bit-identical (FP64 and FP32-mixed), for any tile and block size, across
capacity retries, and with a non-default cell spacing when the single run
uses the same spacing."""
import threading
import time

import numpy as np
import pytest

from common import RC, SKIN, announce

pytestmark = pytest.mark.gpu
DT, REN = 0.005, 20


@pytest.fixture(scope="module")
def tm():
    import tinymd_amd
    name, cus = tinymd_amd.device_info()
    if cus == 0:
        pytest.fail("no HIP device visible to libtinymd_amd")
    return tinymd_amd


@pytest.fixture(scope="module")
def boxes(tm):
    return tm.replica_boxes(seed=7, nrep=5, cells=(6, 9))


def single(tm, box, steps, precision, spacing=1.0, runs=None, ren=REN):
    aabb, x, v = box
    sim = tm.Simulation(np.ones(len(x)), x, v, aabb, (RC + SKIN) * spacing, precision=precision)
    sim.copy_to_accelerator()
    sim.setup(False, RC, SKIN)
    sim.lennard_jones(False, RC)
    for s in (runs or [steps]):
        sim.run_lj(s, ren, DT, False, RC, SKIN)
    _, xs, vs, fs = sim.state()
    th = sim.thermo(RC)
    ng = sim.nghost
    sim.close()
    return xs, vs, fs, th, ng


def assert_bitwise(tm, b, boxes, steps, precision, spacing=1.0, runs=None, ren=REN):
    for r, box in enumerate(boxes):
        xs, vs, fs, _, _ = single(tm, box, steps, precision, spacing, runs, ren)
        xb, vb, fb = b.state(r)
        assert np.array_equal(xb, xs), f"replica {r} positions"
        assert np.array_equal(vb, vs), f"replica {r} velocities"
        assert np.array_equal(fb, fs), f"replica {r} forces"


@pytest.mark.parametrize("precision", ["fp64", "fp32mixed"])
def test_batch_bitwise_vs_single(tm, boxes, precision):
    announce(f"batch 5 replicas {precision} 45 steps vs single runs")
    b = tm.Batch(boxes, precision=precision)
    assert b.run(45) == 45
    assert_bitwise(tm, b, boxes, 45, precision)
    info = b.info()
    for r, box in enumerate(boxes):
        assert info[r]["ghosts"] == single(tm, box, 45, precision)[4]
    b.close()


def test_batch_short_reneighbour(tm, boxes):
    """Rebuilds every third step: each rebuild copies the replicas' state
    back from the step loop's mirrors and rebuilds their ghosts; the
    replicas stay bit-identical to single runs with the same interval."""
    announce("batch 5 replicas fp64, rebuild every 3 steps, 14 steps")
    b = tm.Batch(boxes, precision="fp64", reneigh=3)
    assert b.run(14) == 14
    assert_bitwise(tm, b, boxes, 14, "fp64", ren=3)
    b.close()


def test_batch_thermo_vs_single(tm, boxes):
    announce("batch thermo vs single thermo")
    b = tm.Batch(boxes, precision="fp64")
    b.run(30)
    th = b.thermo()
    for r, box in enumerate(boxes):
        ts = single(tm, box, 30, "fp64")[3]
        for k in ("T", "KE", "PE", "virial", "P"):
            assert th[r][k] == pytest.approx(ts[k], rel=1e-12, abs=1e-12), (r, k)
        assert th[r]["pairs"] == ts["pairs"]
    b.close()


@pytest.mark.parametrize("tile,threads", [(2, 256), (4, 512), (1, 64), (3, 0), (3, 768)])
def test_batch_launch_config_invariance(tm, boxes, tile, threads):
    announce(f"batch config tile={tile} threads={threads}")
    b = tm.Batch(boxes, precision="fp64")
    b.configure(tile=tile, threads=threads)
    b.run(45)
    assert_bitwise(tm, b, boxes, 45, "fp64")
    b.close()


def test_batch_cell_spacing_matches_single_with_same_spacing(tm, boxes):
    announce("batch spacing factor 1.1")
    b = tm.Batch(boxes, precision="fp64")
    b.configure(spacing=1.1)
    b.run(45)
    assert_bitwise(tm, b, boxes, 45, "fp64", spacing=1.1)
    b.close()


def test_batch_ghost_and_list_overflow_retry(tm, boxes):
    """Deliberately small ghost room and list headroom: the set-up grows the
    ghost room and the list capacity; results stay bit-identical."""
    announce("batch capacity retry")
    b = tm.Batch(boxes, precision="fp64")
    b.configure(ghost_headroom=0.25, list_headroom=1.0)
    b.run(45)
    assert_bitwise(tm, b, boxes, 45, "fp64")
    info = b.info()
    assert all(i["ghost_room"] >= i["ghosts"] for i in info)
    b.close()


def test_batch_consecutive_runs(tm, boxes):
    announce("batch run(25) + run(20) vs single run_lj(25) + run_lj(20)")
    b = tm.Batch(boxes, precision="fp64")
    b.run(25)
    b.run(20)
    assert_bitwise(tm, b, boxes, 45, "fp64", runs=[25, 20])
    b.close()


def test_batch_autotune_keeps_results(tm, boxes):
    announce("batch autotune")
    b = tm.Batch(boxes, precision="fp32mixed")
    cfg = b.autotune(trial_steps=20)
    assert cfg["threads"] % 64 == 0 and 64 <= cfg["threads"] <= 1024
    assert cfg["spacing"] in (1.0, 1.1) and cfg["ms_per_step"] > 0
    b.run(45)
    assert_bitwise(tm, b, boxes, 45, "fp32mixed", spacing=cfg["spacing"])
    b.close()


def test_batch_graph_reuse_across_tile_edges(tm, boxes):
    """A run captured under one tile edge is not reused under another: the
    launch shapes and LDS sizes a graph bakes in follow the configuration.
    configure(tile 3) run, configure(tile 4) run: bit-identical to a fresh
    batch configured with tile 4."""
    announce("batch graph reuse: tile 3 run, tile 4 run vs fresh tile 4")
    b = tm.Batch(boxes, precision="fp64")
    b.configure(tile=3)
    b.run(25)
    b.configure(tile=4)
    b.run(25)
    f = tm.Batch(boxes, precision="fp64")
    f.configure(tile=4)
    f.run(25)
    for r in range(len(boxes)):
        for a, c in zip(b.state(r), f.state(r)):
            assert np.array_equal(a, c), r
    b.close()
    f.close()


def expanding_box(n_side=9, spacing=1.25, L=22.4, rate=9.0):
    """A simple-cubic block of atoms in the middle of a periodic box, with
    velocities pointing away from the centre (v = rate * (x - c)): no atom is
    within a cell spacing of a face at t = 0 (no ghosts), but after 20 steps
    the outer layers are, so the ghost room sized at set-up overflows at the
    first rebuild inside the run."""
    g = (np.arange(n_side) - (n_side - 1) / 2.0) * spacing
    X, Y, Z = np.meshgrid(g, g, g, indexing="ij")
    d = np.stack([X.ravel(), Y.ravel(), Z.ravel()], axis=1)
    c = L / 2.0
    return np.array([0.0, L, 0.0, L, 0.0, L]), c + d, rate * d


def test_batch_ghost_overflow_inside_run(tm):
    """Ghost room exhausted at the step-20 rebuild of a run: the run restores
    its starting state, grows the room, rebuilds and runs again.  The result
    is bit-identical to the single-box path, and the room grew."""
    announce("batch ghost overflow at a rebuild inside the run (expanding block)")
    box = expanding_box()
    box2 = expanding_box(n_side=8, spacing=1.3)
    b = tm.Batch([box, box2], precision="fp64")
    b.configure(ghost_headroom=0.25)
    room0 = [i["ghost_room"] for i in b.info()]
    assert all(i["ghosts"] == 0 for i in b.info())
    assert b.run(25) == 25
    info = b.info()
    assert any(i["ghost_room"] > r0 for i, r0 in zip(info, room0)), (room0, info)
    assert all(i["ghost_room"] >= i["ghosts"] for i in info)
    for r, bx in enumerate((box, box2)):
        xs, vs, fs, _, _ = single(tm, bx, 25, "fp64")
        xb, vb, fb = b.state(r)
        assert np.array_equal(xb, xs) and np.array_equal(vb, vs) and np.array_equal(fb, fs), r
    b.close()


@pytest.mark.parametrize("shapes", [
    [(4, 4, 4), (5, 7, 4), (9, 6, 8)],  # up to 7 images of an atom
    [(3, 3, 3), (4, 3, 5), (6, 6, 6)],  # boxes under two cells long: up to 26
])
@pytest.mark.parametrize("precision", ["fp64", "fp32mixed"])
def test_batch_force_pass_writes_ghosts(tm, shapes, precision):
    """One run of 15 steps, whose force passes write the ghosts, against 15
    runs of one step, which start with the ghost pass: bit for bit."""
    from common import perturbed_fcc
    announce(f"batch ghosts {shapes} {precision}")
    boxes = []
    for r, shape in enumerate(shapes):
        aabb, _, x, v = perturbed_fcc(*shape, amp=0.05, seed=r)
        boxes.append((aabb, x, v))
    out = []
    for runs in ([15], [1] * 15):
        b = tm.Batch(boxes, cutoff=RC, skin=SKIN, dt=0.005, precision=precision)
        for n in runs:
            b.run(n)
        out.append([a for r in range(len(boxes)) for a in b.state(r)])
        b.close()
    for a, c in zip(*out):
        assert np.array_equal(a, c)


# tiles of two cells, of about 100 atoms, of full size
@pytest.mark.parametrize("shapes", [
    [(4, 4, 4), (5, 6, 4)],
    [(4, 4, 4), (6, 6, 6), (9, 7, 12), (16, 5, 8), (11, 11, 11)],
    [(6, 6, 6), (34, 34, 34)],
])
def test_batch_tile_shapes(tm, shapes):
    """Automatic tiles, another shape for each box, against cubes of two
    cells: bit for bit."""
    from common import perturbed_fcc
    announce(f"batch tile shapes {shapes}")
    boxes = []
    for r, shape in enumerate(shapes):
        aabb, _, x, v = perturbed_fcc(*shape, amp=0.05, seed=r)
        boxes.append((aabb, x, v))
    out = []
    for tile in (0, 2):
        b = tm.Batch(boxes, cutoff=RC, skin=SKIN, dt=0.005)
        b.configure(tile=tile)
        b.run(25)
        out.append([a for r in range(len(boxes)) for a in b.state(r)])
        b.close()
    for a, c in zip(*out):
        assert np.array_equal(a, c)


def test_first_reads_by_ascending_size(tm):
    """A new handle's replicas read by ascending size take less than twice as
    long as by descending size: the buffer that they pass through is not made
    anew for every larger one (then about three times as long here)."""
    announce("first reads of a batch, ascending and descending")
    boxes = []
    for nc in range(8, 23):
        _, x, v = tm.generate_fcc(nc, nc, nc)
        boxes.append((np.array([0.0, nc * 1.6796] * 3), x, v))
    best = []
    for order in (range(15), range(14, -1, -1)):
        times = []
        for _ in range(3):
            b = tm.Batch(boxes)
            t = time.perf_counter()
            for r in order:
                x, v, _ = b.state(r)
                assert np.array_equal(x, boxes[r][1]) and np.array_equal(v, boxes[r][2])
            times.append(time.perf_counter() - t)
            b.close()
        best.append(min(times))
    assert best[0] < 2.0 * best[1], best


def test_replicas_read_by_several_threads(tm):
    """Host threads that read different replicas of one handle at a time."""
    announce("replicas read by several threads")
    boxes = []
    for nc in (5, 12, 6, 14, 7, 13):
        _, x, v = tm.generate_fcc(nc, nc, nc)
        boxes.append((np.array([0.0, nc * 1.6796] * 3), x, v))
    b = tm.Batch(boxes)
    wrong = []

    def read(r):
        for _ in range(100):
            x, v, _ = b.state(r)
            if not (np.array_equal(x, boxes[r][1]) and np.array_equal(v, boxes[r][2])):
                wrong.append(r)

    threads = [threading.Thread(target=read, args=(r,)) for r in range(len(boxes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    b.close()


def test_many_replicas_choose_tiles_quickly(tm):
    """A restart of 3,072 replicas of 108 and 256 atoms chooses each one's tile;
    it takes less than 1.2 times as long as with a given tile (35 ms of 127 went
    into it once, a third again)."""
    announce("tiles of many replicas")
    b = tm.Batch(tm.replica_boxes(seed=3, nrep=48, cells=(3, 4)) * 64)
    best = []
    for tile in (4, 0):
        b.configure(tile=tile)
        times = []
        for _ in range(5):
            t = time.perf_counter()
            b.reset()
            times.append(time.perf_counter() - t)
        best.append(min(times))
    print(best, [i["tile"] for i in b.info()[:8]])
    assert best[1] < 1.2 * best[0], best
    b.close()
