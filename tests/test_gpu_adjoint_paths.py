"""GPU parity of the one-launch trajectory and reverse steps against the
oracle's scatter-form adjoint, on the branches that ordinary boxes do not
take: windows read from the mirrors because they outgrow LDS, the plain
cutoff, eps and sigma other than one, an interval of one state and a run
shorter than one interval."""
import numpy as np
import pytest

import pyoracle as po
from common import RC, SKIN, announce, perturbed_fcc

pytestmark = pytest.mark.gpu

DT = 0.005


@pytest.fixture(scope="module")
def tm():
    import tinymd_amd
    _, cus = tinymd_amd.device_info()
    if cus == 0:
        pytest.fail("no HIP device visible to libtinymd_amd")
    return tinymd_amd


@pytest.mark.parametrize("tile,shift,eps,sigma,steps,ck", [
    (0, True, 1.0, 1.0, 25, 20),     # staged, as ordinary runs
    (8, True, 1.0, 1.0, 25, 20),     # one tile, window beyond LDS
    (1, True, 1.05, 0.98, 23, 10),   # one-cell tiles, general eps and sigma
    (8, False, 1.05, 0.98, 21, 20),  # plain cutoff from the mirrors
    (0, False, 1.0, 1.0, 12, 5),     # plain cutoff, staged
    (2, True, 1.0, 1.0, 20, 20),     # the last interval is one state
    (0, True, 1.0, 1.0, 3, 20),      # shorter than an interval
    (0, True, 1.0, 1.0, 4, 1),       # a rebuild every step
])
def test_adjoint_branches_match_oracle(tm, tile, shift, eps, sigma, steps, ck):
    announce(f"adjoint tile={tile} shift={shift} eps={eps} sigma={sigma} steps={steps} ck={ck}")
    aabb, m, x, v = perturbed_fcc(7, 6, 8, amp=0.05, seed=9)
    sim = tm.Simulation(m, x, v, aabb, RC + SKIN, lj_shift=shift)
    if tile:
        sim.set_tile(tile)
    sim.copy_to_accelerator()
    r = sim.traj_adjoint(steps, ck, DT, RC, SKIN, eps, sigma, -4.0, 1.0)
    o = po.OracleSim(m, x, v, aabb, RC + SKIN, threads=4)
    o.setup(False, po.HALF_GHOST_FULL, RC + SKIN)
    o.lj(False, RC, eps, sigma, shift=int(shift))
    q = o.traj_adjoint(steps, ck, DT, RC, SKIN, eps, sigma, shift=int(shift), u_target=-4.0, p_target=1.0)
    assert r["ubar"] == pytest.approx(q["ubar"], rel=1e-12)
    assert r["pbar"] == pytest.approx(q["pbar"], rel=1e-10)
    assert r["grad_eps"] == pytest.approx(q["grad_eps"], rel=1e-9)
    assert r["grad_sigma"] == pytest.approx(q["grad_sigma"], rel=1e-9)
    for key in ("grad_x0", "grad_v0"):
        d = np.linalg.norm(r[key] - q[key]) / np.linalg.norm(q[key])
        assert d <= 1e-9, key
    # the call leaves the state at x0
    _, xa, va, _ = sim.state()
    assert np.array_equal(xa, x) and np.array_equal(va, v)


def test_states_no_longer_kept(tm):
    """A sheet that drifts to the face between two rebuilds, so the rebuild
    makes room for more ghosts and the rest of the forward pass is not kept:
    every interval is recomputed.  And the same run again, kept whole now
    that the room is there: bit for bit the same gradients."""
    announce("adjoint, ghosts outgrow their room")
    L, ny = 48.0, 43
    a = L / ny
    g = np.arange(ny) * a
    z, y, k = np.meshgrid(g, g, np.arange(3), indexing="ij")
    x = np.stack([4.0 + 1.1 * k.ravel(), y.ravel(), z.ravel()], axis=1)
    v = np.random.default_rng(3).normal(0.0, 0.3, x.shape)
    v[:, 0] -= 35.0
    aabb = np.array([0.0, L] * 3)
    m = np.ones(len(x))
    tm.load().md_deallocate_grid()
    sim = tm.Simulation(m, x, v, aabb, RC + SKIN, lj_shift=True)
    sim.copy_to_accelerator()
    r = sim.traj_adjoint(25, 20, DT, RC, SKIN, 1.0, 1.0, -4.0, 1.0)
    again = sim.traj_adjoint(25, 20, DT, RC, SKIN, 1.0, 1.0, -4.0, 1.0)
    o = po.OracleSim(m, x, v, aabb, RC + SKIN, threads=4)
    o.setup(False, po.HALF_GHOST_FULL, RC + SKIN)
    o.lj(False, RC, 1.0, 1.0, shift=1)
    q = o.traj_adjoint(25, 20, DT, RC, SKIN, 1.0, 1.0, shift=1, u_target=-4.0, p_target=1.0)
    assert r["grad_eps"] == pytest.approx(q["grad_eps"], rel=1e-9)
    for key in ("grad_x0", "grad_v0"):
        assert np.linalg.norm(r[key] - q[key]) / np.linalg.norm(q[key]) <= 1e-9, key
        assert np.array_equal(r[key], again[key]), key


@pytest.mark.parametrize("shape,shift", [
    ((16, 16, 16), True),   # 16,384 atoms: the last box with four lanes an atom
    ((16, 16, 17), True),   # the first with two
    ((16, 16, 32), False),  # 32,768 atoms: the last with two, plain cutoff
    ((16, 16, 33), True),   # one lane an atom
])
def test_lanes_of_an_atom(tm, shape, shift):
    announce(f"adjoint lanes {shape} shift={shift}")
    aabb, m, x, v = perturbed_fcc(*shape, amp=0.05, seed=5)
    sim = tm.Simulation(m, x, v, aabb, RC + SKIN, lj_shift=shift)
    sim.copy_to_accelerator()
    r = sim.traj_adjoint(5, 3, DT, RC, SKIN, 1.0, 1.0, -4.0, 1.0)
    o = po.OracleSim(m, x, v, aabb, RC + SKIN, threads=4)
    o.setup(False, po.HALF_GHOST_FULL, RC + SKIN)
    o.lj(False, RC, 1.0, 1.0, shift=int(shift))
    q = o.traj_adjoint(5, 3, DT, RC, SKIN, 1.0, 1.0, shift=int(shift), u_target=-4.0, p_target=1.0)
    assert r["ubar"] == pytest.approx(q["ubar"], rel=1e-12)
    assert r["grad_eps"] == pytest.approx(q["grad_eps"], rel=1e-9)
    assert r["grad_sigma"] == pytest.approx(q["grad_sigma"], rel=1e-9)
    for key in ("grad_x0", "grad_v0"):
        assert np.linalg.norm(r[key] - q[key]) / np.linalg.norm(q[key]) <= 1e-9, key


def test_sheet_leaves_its_room(tm):
    """The sheet of test_states_no_longer_kept has more ghosts after its rebuild
    than a simulation made anew has room for, so that test's first gradient
    recomputes its intervals."""
    announce("adjoint, room of the sheet")
    L, ny = 48.0, 43
    g = np.arange(ny) * (L / ny)
    z, y, k = np.meshgrid(g, g, np.arange(3), indexing="ij")
    x = np.stack([4.0 + 1.1 * k.ravel(), y.ravel(), z.ravel()], axis=1)
    v = np.random.default_rng(3).normal(0.0, 0.3, x.shape)
    v[:, 0] -= 35.0
    room = 1.25 * len(x) * ((1 + 2 * (RC + SKIN) / L) ** 3 - 1) + 4096
    tm.load().md_deallocate_grid()
    sim = tm.Simulation(np.ones(len(x)), x, v, np.array([0.0, L] * 3), RC + SKIN, lj_shift=True)
    sim.copy_to_accelerator()
    sim.setup(False, RC, SKIN)
    assert sim.nghost < room
    sim.lennard_jones(False, RC)
    sim.run_lj(20, 20, DT)
    assert sim.nghost > room
    sim.close()
