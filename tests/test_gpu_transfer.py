"""Host arrays to the device and back, and a simulation made over another
one: the values that went in come back bit for bit, and nothing of the
replaced simulation is left in the new one's results."""
import ctypes

import numpy as np
import pytest

from common import RC, SKIN, announce, perturbed_fcc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tm():
    import tinymd_amd
    _, cus = tinymd_amd.device_info()
    if cus == 0:
        pytest.fail("no HIP device visible to libtinymd_amd")
    return tinymd_amd


# 85, 86: either side of a block's 256 doubles; 90,000: more doubles than one
# sweep of the grid; 300,001: host copies by several threads
@pytest.mark.parametrize("n", [1, 85, 86, 90000, 300001])
def test_round_trip(tm, n):
    announce(f"host arrays out and back, {n} atoms")
    rng = np.random.default_rng(n)
    aabb = np.array([0.0, 80.0] * 3)
    m, x, v = rng.random(n), rng.random((n, 3)) * 80.0, rng.normal(size=(n, 3))
    sim = tm.Simulation(m, x, v, aabb, RC + SKIN)
    for upload in (False, True):  # the host's copy alone, then through the device
        if upload:
            sim.copy_to_accelerator()
        m1, x1, v1, f1 = sim.state()
        assert np.array_equal(m1, m) and np.array_equal(x1, x) and np.array_equal(v1, v)
        assert not f1.any()
    sim.borders()
    mg, xg, vg, fg = sim.ghost_state()
    own = sim.ghost_table()["owner"]
    assert len(mg) == len(own) and np.array_equal(mg, m[own]) and np.array_equal(vg, v[own])
    shift = (xg - x[own]) / 80.0
    assert np.allclose(shift, np.rint(shift), atol=1e-12) and not fg.any()
    _, x1, _, _ = sim.state()
    assert np.array_equal(x1, x)
    sim.close()


def _run(tm, shape, half, precision, dem):
    if dem:
        m, x, v = tm.generate_granular_gas(shape[0], vmax=2.0)
        sim = tm.Simulation(m, x, v, np.array([0.0, shape[0] * 1.6796] * 3), 1.3, precision=precision, dem_radius=0.5)
        sim.copy_to_accelerator()
        sim.setup(half, 1.0, 0.3)
        sim.dem(half, 1.0)
        sim.run_dem(45, 20, 0.001, half)
        return sim.state()
    aabb, m, x, v = perturbed_fcc(*shape, amp=0.05, seed=9)
    sim = tm.Simulation(m, x, v, aabb, RC + SKIN, precision=precision)
    sim.copy_to_accelerator()
    sim.setup(half, RC, SKIN)
    sim.lennard_jones(half, RC)
    sim.run_lj(45, 20, 0.005, half)
    out = sim.state()
    return out + (np.array(list(sim.thermo(RC).values())),)


# same size; smaller and larger within the memory at hand; less than half of
# it; larger than it; another kind of simulation
@pytest.mark.parametrize("first,second", [
    (((10, 10, 10), False, "fp64", False), ((10, 10, 10), True, "fp32mixed", False)),
    (((10, 9, 11), True, "fp64", False), ((9, 9, 9), False, "fp64", False)),
    (((16, 16, 16), False, "fp32mixed", False), ((5, 6, 7), True, "fp64", False)),
    (((6, 6, 6), False, "fp64", False), ((16, 15, 17), False, "fp32mixed", False)),
    (((14, 14, 14), False, "fp64", False), ((17, 0, 0), True, "fp64", True)),
])
def test_simulation_over_another(tm, first, second):
    announce(f"{second} over {first}")
    tm.load().md_deallocate_grid()
    alone = _run(tm, *second)
    tm.load().md_deallocate_grid()
    _run(tm, *first)
    over = _run(tm, *second)
    for a, b in zip(alone, over):
        assert np.array_equal(a, b)


def test_refused_simulation_leaves_none(tm):
    announce("refused simulation")
    aabb, m, x, v = perturbed_fcc(5, 5, 5, amp=0.05, seed=9)
    tm.Simulation(m, x, v, aabb, RC + SKIN)
    with pytest.raises(tm.TinyMDError, match="box length"):
        tm.Simulation(m, x, v, np.array([0.0, 5.0] * 3), RC + SKIN)
    assert tm.load().md_get_number_of_particles() == 0
    tm.load().tmd_clear_error()


def test_cells_of_the_last_binning(tm):
    """The cells stay those of the last binning when the ghosts go or become
    fewer, no entry is written behind the caller's arrays, and a simulation
    made over another one has none before its own."""
    announce("cells after the ghosts changed")
    L = tm.load()
    aabb, m, x, v = perturbed_fcc(7, amp=0.05, seed=9)
    x = 0.3 + x * ((7 * 1.6796 - 0.6) / (7 * 1.6796))  # no atom within 0.3 of a face
    v = np.where(x > 5.9, -1.0, 1.0)                   # all move inwards
    sim = tm.Simulation(m, x, v, aabb, RC + SKIN)
    sim.copy_to_accelerator()
    sim.setup(False, RC, SKIN)
    start, parts, cell = sim.cells()
    n, ng = sim.nlocal, sim.nghost

    def cells():
        nall = sim.nlocal + sim.nghost
        at = np.full(n + ng + 64, -7, dtype=np.int32)
        st, pa = np.zeros_like(start), np.zeros_like(parts)
        ptr = lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_int))
        assert L.tmd_get_cells(ptr(st), ptr(pa), ptr(at)) == len(parts)
        assert np.array_equal(st, start) and np.array_equal(pa, parts)
        assert np.array_equal(at[:nall], cell[:nall]) and np.all(at[nall:] == -7)

    cells()
    sim.exchange()
    assert sim.nghost == 0
    cells()
    sim.initial_integration(0.5)
    sim.borders()
    assert 0 < sim.nghost < ng
    cells()
    aabb2, m2, x2, v2 = perturbed_fcc(6, amp=0.05, seed=9)
    sim = tm.Simulation(m2, x2, v2, aabb2, RC + SKIN)
    sim.copy_to_accelerator()
    with pytest.raises(tm.TinyMDError, match="not binned"):
        sim.cells()
    L.tmd_clear_error()
    sim.setup(False, RC, SKIN)
    st, pa, at = sim.cells()
    for c in range(len(st) - 1):
        assert np.all(at[pa[st[c]:st[c + 1]]] == c)
    sim.close()


# a drop in the middle of its box has no ghosts; without a ghost index they
# follow in a pass of their own
@pytest.mark.parametrize("kind", ["full", "drop", "no_index", "dem"])
def test_state_put_back_between_runs(tm, kind):
    """Reading the state and uploading it again between two runs on the same
    lists changes nothing."""
    announce(f"state put back between runs, {kind}")
    out = []
    for put_back in (False, True):
        if kind == "dem":
            m, x, v = tm.generate_granular_gas(9, vmax=2.0)
            sim = tm.Simulation(m, x, v, np.array([0.0, 9 * 1.6796] * 3), 1.3, dem_radius=0.5)
        else:
            aabb, m, x, v = perturbed_fcc(6, 5, 7, amp=0.05, seed=9)
            if kind == "drop":
                x, aabb = x + 14.0, np.array([0.0, 40.0] * 3)
            sim = tm.Simulation(m, x, v, aabb, RC + SKIN)
            tm.load().tmd_set_ghost_index_limit(1 if kind == "no_index" else 0)
        sim.copy_to_accelerator()
        rc = 1.0 if kind == "dem" else RC
        sim.setup(kind == "dem", rc, SKIN)
        sim.dem(True, rc) if kind == "dem" else sim.lennard_jones(False, rc)
        assert (sim.nghost == 0) == (kind == "drop")
        res = []
        for steps in (7, 6, 25):
            sim.run_dem(steps, 20, 0.001) if kind == "dem" else sim.run_lj(steps, 20, 0.005)
            res += sim.state()[1:]
            if put_back:
                sim.copy_to_accelerator()
        out.append(res)
        tm.load().tmd_set_ghost_index_limit(0)
    sim.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
