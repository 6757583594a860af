"""GPU: meshes of more than 1024 tiles, whose passes list their tiles, on what
the smaller meshes of the other files cover for the launch of a workgroup per
tile.  The meshes get their size from thin or mostly void members, so that the
oracle stays quick.  Bar: bit-identical to the oracle; the bed-friction gradient
at rtol 1e-12 (its partial sums are ordered by tile)."""
import sys

import numpy as np
import pytest

from discrete_adjoint_amd import _lib
from discrete_adjoint_amd.solver import Ensemble, Simulation
from helpers import small_flow_problem, with_materials

pytestmark = pytest.mark.gpu

MANY = (8, 4160)   # a member of 1040 tiles of 64 x 4


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _U(pb):
    return [pb.h.copy(), pb.hu.copy(), pb.hv.copy()]


def _box(pb):
    """A box that cuts through the pile (one that holds all of it has the total
    mass for its functional, whose gradient is rounding noise)."""
    L, W = pb.nx * pb.dx, pb.ny * pb.dy
    return pb.box_weights((0.4 * L, 0.8 * L, 0.0, 0.5 * W)).reshape(3, -1)


def _members(nsteps):
    return [small_flow_problem(130, 70, nsteps), small_flow_problem(*MANY, nsteps),
            small_flow_problem(40, 21, nsteps, slope=20.0, phi_bed=18.0)]


def _references(oracle_lib, mem, weights):
    return [oracle_lib.Oracle.from_problem(pb).forward_adjoint(_U(pb), pb.nsteps, w,
                                                               want_dphi=True)
            for pb, w in zip(mem, weights)]


def _sweep_equals(ens, mem, weights, refs, what):
    ens.set_state(*[np.concatenate([getattr(p, f) for p in mem]) for f in ("h", "hu", "hv")])
    ens.run(mem[0].nsteps)
    lam, dphi = ens.dual_solver(weights, want_dphi=True)
    for b, (UN, dts, lam_ref, dphi_ref) in enumerate(refs):
        assert np.array_equal(ens.member_dt_record(b), dts), (what, b)
        assert np.array_equal(ens.member_state(b), UN), (what, b)
        assert np.array_equal(lam[b], lam_ref), (what, b)
        assert dphi[b] == pytest.approx(dphi_ref, rel=1e-12, abs=1e-300), (what, b)


@pytest.mark.parametrize("graph", [0, 1])
def test_selections_and_autotune(oracle_lib, graph):
    """Every pass in its own variant, changed between sweeps on one context, and
    the autotuner's choice: the coefficient pass runs in the update's variant,
    which the selection says and the choice is made for."""
    mem = _members(24)
    _say(f"case list path selections graph={graph}")
    weights = [_box(p) for p in mem]
    refs = _references(oracle_lib, mem, weights)
    with Ensemble(mem, checkpoint_every=7, use_graph=graph) as ens:
        assert ens.tile_selection() == [3, 3, 0]
        _sweep_equals(ens, mem, weights, refs, "built-in")
        for sel in [(3, 3, 3), (0, 1, 2), None, (1, 0, 3), (3, 2, 0), (2, 2, 2)]:
            if sel is None:
                var, ms = ens.autotune(reps=3)
                assert var[0] == var[1] and ens.tile_selection() == var
                assert (ms > 0).all()
                assert ms[:2, var[0]].sum() == ms[:2].sum(axis=0).min()
                assert ms[2, var[2]] == ms[2].min()
            else:
                ens.select_tiles(sel)
                assert ens.tile_selection() == [sel[1], sel[1], sel[2]]
            _sweep_equals(ens, mem, weights, refs, sel)


def test_selection_of_a_small_mesh_is_per_pass():
    pb = small_flow_problem(64, 64, 4)
    _say("case selection of a small mesh")
    with Simulation(pb) as sim:
        assert sim.tile_selection() == [0, 0, 0]
        sim.select_tiles((1, 2, 3))
        assert sim.tile_selection() == [1, 2, 3]
    with Simulation(pb, precision=_lib.TG_MIXED) as sim:
        sim.select_tiles((1, 2, 3))
        assert sim.tile_selection() == [1, 2, 3]


@pytest.mark.parametrize("precision", [_lib.TG_FP64, _lib.TG_FWD64_ADJ32])
def test_run_replay_and_stored_states(oracle_lib, precision):
    """A run, its recomputed and its stored states, and its replay (the FP32
    adjoint's forward passes are the FP64 ones)."""
    mem = _members(20)
    _say(f"case list path run and replay precision {precision}")
    weights = [_box(p) for p in mem]
    refs = _references(oracle_lib, mem, weights)
    for k, stored in ((6, 0), (6, 8), (1, 0)):
        store = 24 * sum(p.n for p in mem) * stored
        with Ensemble(mem, precision=precision, checkpoint_every=k, store_bytes=store) as ens:
            for rep in range(2):
                ens.set_state(*[np.concatenate([getattr(p, f) for p in mem])
                                for f in ("h", "hu", "hv")])
                ens.run(20)
                for b, (UN, dts, _, _) in enumerate(refs):
                    assert np.array_equal(ens.member_state(b), UN), (k, stored, rep, b)
                    assert np.array_equal(ens.member_dt_record(b), dts), (k, stored, rep, b)
                lam, dphi = ens.dual_solver(weights, want_dphi=True)
                for b, (_, _, lam_ref, dphi_ref) in enumerate(refs):
                    if precision == _lib.TG_FP64:
                        assert np.array_equal(lam[b], lam_ref), (k, stored, rep, b)
                        assert dphi[b] == pytest.approx(dphi_ref, rel=1e-12), (k, stored, rep, b)
                    else:  # the bar of this mode's sweeps
                        err = np.linalg.norm(lam[b] - lam_ref)
                        assert err <= 1e-4 * np.linalg.norm(lam_ref), (k, stored, rep, b)
    one = small_flow_problem(192, 1500, 6)
    orc = oracle_lib.Oracle.from_problem(one)
    U = _U(one)
    dts = orc.run(U, 6)
    with Simulation(one, precision=precision, max_steps=8) as sim:
        sim.replay(dts)
        assert np.array_equal(sim.get_state(), U)
        assert np.array_equal(sim.trajectory_state(6), U)


@pytest.mark.parametrize("time0,maxtime", [(0.25, 0.0), (0.5, 0.5)])
def test_steps_with_dt_not_positive(oracle_lib, time0, maxtime):
    """A negative dt and one of 0 on -0.0 in dry cells: the dry list's formula,
    bit for bit with its signs, also where a block is dry, listed and void."""
    pb = small_flow_problem(140, 1400, 4)
    dry = (pb.h == 0) & (np.arange(pb.n) // 140 > 500)
    for f in (pb.h, pb.hu, pb.hv):
        f[dry] = -0.0
    pb.h[dry.nonzero()[0][::97]] = -1e-3     # clamped
    pb.h[dry.nonzero()[0][::89]] = 5e-5      # below tiny, moving
    pb.hu[dry.nonzero()[0][::89]] = -1e-6
    _say(f"case list path clock {time0} maxtime {maxtime}")
    orc = oracle_lib.Oracle.from_problem(pb)
    orc.params.maxtime = maxtime
    orc.time = time0
    U = _U(pb)
    with Simulation(pb, max_steps=4, use_graph=0) as sim:
        sim.params.maxtime = maxtime
        sim.set_clock(0, time0)
        for s in range(3):
            dt_ref, _ = orc.step(U, s)
            st = sim.step()
            assert dt_ref <= 0 and st.dt == dt_ref, s
            got = sim.get_state()
            assert np.array_equal(got, U) and np.array_equal(np.signbit(got), np.signbit(U)), s
    orc = oracle_lib.Oracle.from_problem(pb)
    U, dts = _U(pb), [0.03, -0.02, 0.0, 0.04]
    for s, dt in enumerate(dts):
        orc.step(U, s, dt)
    with Simulation(pb, max_steps=4) as sim:
        sim.replay(np.array(dts))
        got = sim.get_state()
        assert np.array_equal(got, U) and np.array_equal(np.signbit(got), np.signbit(U))


@pytest.mark.parametrize("variants", [None, (1, 1, 2), (2, 2, 3)])
def test_materials(oracle_lib, variants):
    mem = [with_materials(p, phis, split=s)
           for p, phis, s in zip(_members(20)[:2], ((15.0, 24.0), (12.0, 30.0)), (0.42, 0.5))]
    mem.append(_members(20)[2])               # one material beside them
    _say(f"case list path materials {variants}")
    weights = [_box(p) for p in mem]
    refs = _references(oracle_lib, mem, weights)
    with Ensemble(mem, checkpoint_every=6) as ens:
        if variants:
            ens.select_tiles(variants)
        for rep in range(2):
            _sweep_equals(ens, mem, weights, refs, (variants, rep))
    plain = _references(oracle_lib, _members(20)[:1], weights)
    assert not np.array_equal(plain[0][0][1], refs[0][0][1])   # (the materials matter)


@pytest.mark.parametrize("graph,stored", [(0, 0), (1, 0), (1, 12)])
def test_maxh_record_and_functional_at_its_step(oracle_lib, graph, stored):
    """The box record of every step, and the reverse sweep from the step of its
    maximum, of a mesh with more than 1024 tiles."""
    pb = small_flow_problem(140, 1400, 40)
    mask = np.zeros(pb.n, bool)
    i, j = np.arange(pb.n) % 140, np.arange(pb.n) // 140
    front = np.flatnonzero(pb.h > 0) % 140
    # a strip inside the pile's lower edge: it fills, then drains
    mask[(abs(i - front.max() + 1) < 2) & (i < front.max()) & (abs(j - 700) < 8)] = True
    _say(f"case list path maxh graph={graph} stored={stored}")
    orc, U, rec = oracle_lib.Oracle.from_problem(pb), _U(pb), []
    for s in range(pb.nsteps):
        orc.step(U, s)
        rec.append(U[0][mask].max(initial=0.0))
    at = int(np.argmax(rec)) + 1
    assert 1 < at < pb.nsteps
    w = np.zeros((3, pb.n))
    w[0, mask] = 1.0
    orc = oracle_lib.Oracle.from_problem(pb)
    _, _, lam_ref, dphi_ref = orc.forward_adjoint(_U(pb), at, w, want_dphi=True)
    with Simulation(pb, checkpoint_every=7, use_graph=graph,
                    store_bytes=24 * pb.n * stored) as sim:
        sim.set_maxh_region(mask)
        for rep in range(2):
            sim.set_state(*_U(pb))
            sim.run()
            assert np.array_equal(sim.box_record(), rec), rep
            hm, st = sim.maxh()
            assert hm[0] == max(rec) and st[0] == at, rep
            lam, dphi = sim.dual_solver(w, want_dphi=True, step=at)
            assert np.array_equal(lam, lam_ref), rep
            assert dphi == pytest.approx(dphi_ref, rel=1e-12), rep


@pytest.mark.parametrize("tile", [(0, 0), (64, 4), (32, 8), (16, 16)])
def test_reverse_steps_by_the_list(oracle_lib, tile):
    """Single reverse steps with the gradient over wet, thin, void and boundary
    cells, those of lambda^{s+1} != 0 on void tiles among them."""
    nx, ny = 140, 1400
    _say(f"case list path reverse step tile {tile}")
    rng = np.random.default_rng(5)
    pb = small_flow_problem(nx, ny, 4)
    rows = np.arange(pb.n) // nx
    flow = (rows < 41) | (abs(rows - 700) < 30) | (rows > ny - 9)
    pb.h = np.where(flow, rng.uniform(0.0, 5.0, pb.n), 0.0)
    pb.h[rng.uniform(size=pb.n) < 0.2] = 0.0
    thin = flow & (rng.uniform(size=pb.n) < 0.1)
    pb.h[thin] = 1e-4 * rng.choice([0.5, 1.0, 1.5], thin.sum())
    pb.hu, pb.hv = (pb.h * rng.normal(scale=6.0, size=pb.n) for _ in range(2))
    lam = rng.normal(size=(3, pb.n)) * (flow | (abs(rows - 300) < 20))
    orc = oracle_lib.Oracle.from_problem(pb)
    with Simulation(pb, max_steps=64, tile_x=tile[0], tile_y=tile[1]) as sim:
        for s, dt in ((3, 0.03), (60, 0.05)):
            ref, dphi = orc.adjoint_step(_U(pb), s, dt, lam, want_dphi=True)
            got, g = sim.adjoint_step_grad(s, dt, lam)
            assert np.array_equal(got, np.asarray(ref).reshape(3, -1)), s
            assert np.array_equal(sim.adjoint_step(s, dt, lam), got), s
            # each cell's term lambda . dU/dphi is rounded some 30 times, and the
            # terms are added one by one: 1e-12 of their absolute sum
            terms = np.abs(lam * orc.dstep_dphi(_U(pb), s, dt).reshape(3, -1)).sum()
            assert abs(g - dphi) <= 1e-12 * terms, s
            assert abs(dphi) > 1e-6 * terms


@pytest.mark.parametrize("rows", [300, 3000])   # 2400 and 24,000 thin cells
def test_fp32_thin_cells_of_a_very_large_mesh(oracle_lib, rows):
    """Past 32,768 tiles the cells next to a thin layer go to one of two kernels,
    by their number (16,384).  Bar: that of the FP32 reverse step elsewhere, 1e-4
    in norm; a second step repeats the first bit for bit."""
    nx, ny = 8, 131200
    _say(f"case list path fp32 thin cells {nx}x{ny} rows {rows}")
    pb = small_flow_problem(nx, ny, 4)
    rng = np.random.default_rng(rows)
    at = np.arange(pb.n) // nx
    thin = (at >= 700) & (at < 700 + rows)
    pb.h[thin], pb.hu[thin], pb.hv[thin] = 5e-4, 3e-3, -2e-3
    lam = rng.normal(size=(3, pb.n)) * (pb.h > 0)
    orc = oracle_lib.Oracle.from_problem(pb)
    ref, dphi = orc.adjoint_step(_U(pb), 60, 0.05, lam, want_dphi=True)
    terms = np.abs(lam * orc.dstep_dphi(_U(pb), 60, 0.05)).sum()
    ref = np.asarray(ref).reshape(3, -1)
    with Simulation(pb, max_steps=64, precision=_lib.TG_FWD64_ADJ32) as sim:
        got, g = sim.adjoint_step_grad(60, 0.05, lam)
        assert np.linalg.norm(got - ref) <= 1e-4 * np.linalg.norm(ref)
        assert np.linalg.norm((got - ref)[:, thin]) <= 1e-4 * np.linalg.norm(ref[:, thin])
        assert abs(g - dphi) <= 1e-4 * terms
        again, _ = sim.adjoint_step_grad(60, 0.05, lam)
        assert np.array_equal(again, got)
        lam[:, thin] = 0.0                            # and after one without them
        sim.adjoint_step(60, 0.05, lam)
        assert np.array_equal(sim.adjoint_step(60, 0.05, lam),
                              sim.adjoint_step_grad(60, 0.05, lam)[0])
