"""GPU: forward steps whose dt is not a positive finite number, against the
oracle bit for bit.  The update's short path writes a dry tile as
update_states' zero-flux formula U - dt/dx (0 - 0) - dt/dy (0 - 0) with h
clamped at 0, and skips tiles whose input and output hold +0.0 only while dt
is finite; these cases check that the formula, not a copy, is what lands:
the clock past maxtime (negative dt) and at maxtime (dt = 0), on states with
-0.0 in dry cells (a negative dt turns them into +0.0); an all-dry domain
(dt = inf: non-finite, reported); steps replayed with a negative dt."""
import sys

import numpy as np
import pytest

from discrete_adjoint_amd import _lib
from discrete_adjoint_amd.solver import Ensemble, Simulation, TgError
from helpers import small_flow_problem

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _negative_zeros(pb):
    """The problem with -0.0 in h, hu, hv of its dry cells."""
    dry = pb.h == 0
    for f in (pb.h, pb.hu, pb.hv):
        f[dry] = -0.0
    assert dry.sum() > pb.n // 2
    return pb


def _same(a, b):
    return all(np.array_equal(x, y) and np.array_equal(np.signbit(x), np.signbit(y))
               for x, y in zip(a, b))


@pytest.mark.parametrize("time0,maxtime", [(0.25, 0.0), (0.5, 0.5)])
def test_steps_with_dt_not_positive(oracle_lib, time0, maxtime):
    pb = _negative_zeros(small_flow_problem(70, 45, 10))
    _say(f"case dt edge: clock {time0}, maxtime {maxtime}")
    orc = oracle_lib.Oracle.from_problem(pb)
    orc.params.maxtime = maxtime
    orc.time = time0
    U = [pb.h.copy(), pb.hu.copy(), pb.hv.copy()]
    with Simulation(pb, max_steps=4, use_graph=0) as sim:
        sim.params.maxtime = maxtime
        sim.set_clock(0, time0)
        for s in range(3):
            dt_ref, _ = orc.step(U, s)
            st = sim.step()
            assert dt_ref <= 0 and st.dt == dt_ref, s
            assert _same(sim.get_state(), U), s
    if time0 > maxtime:  # the formula turned -0.0 of dry cells into +0.0
        assert (~np.signbit(U[1][pb.h == 0])).any()


def test_all_dry_domain_is_reported(oracle_lib):
    pb = small_flow_problem(40, 30, 4)
    for f in (pb.h, pb.hu, pb.hv):
        f[:] = 0.0
    _say("case dt edge: all dry")
    orc = oracle_lib.Oracle.from_problem(pb)
    with pytest.raises(FloatingPointError):
        orc.step([pb.h.copy(), pb.hu.copy(), pb.hv.copy()], 0)
    with Simulation(pb, max_steps=4, use_graph=0) as sim:
        with pytest.raises(TgError) as e:
            sim.step()
        assert e.value.code == _lib.TG_ERR_NONFINITE


def test_replayed_negative_dt(oracle_lib):
    pb = _negative_zeros(small_flow_problem(70, 45, 10))
    _say("case dt edge: replay with a negative dt")
    dts = [0.05, -0.03, 0.04, 0.0]
    orc = oracle_lib.Oracle.from_problem(pb)
    U = [pb.h.copy(), pb.hu.copy(), pb.hv.copy()]
    for s, dt in enumerate(dts):
        orc.step(U, s, dt)
    with Simulation(pb, max_steps=8, use_graph=0) as sim:
        sim.replay(np.array(dts))
        assert _same(sim.get_state(), U)


@pytest.mark.parametrize("ny", [300, 1500])   # 225 tiles, 1125 tiles
@pytest.mark.parametrize("precision", [_lib.TG_FP64, _lib.TG_FWD64_ADJ32, _lib.TG_MIXED,
                                       _lib.TG_FP32])
def test_dt_not_finite_leaves_no_finite_cell(precision, ny):
    """A step whose dt is not finite makes every cell so, those of blocks that
    the marks let the steps before leave alone too, on meshes of either launch:
    replayed, and as a single step."""
    nx = 192
    _say(f"case dt edge: dt not finite {nx}x{ny} precision {precision}")
    pb = small_flow_problem(nx, ny, 10)
    with Simulation(pb, precision=precision, max_steps=8, use_graph=0) as sim:
        for bad in (np.inf, np.nan):
            sim.set_state(pb.h, pb.hu, pb.hv)
            sim.replay(np.array([0.02, 0.03]))
            assert np.isfinite(sim.get_state()).all()
            sim.set_state(pb.h, pb.hu, pb.hv)
            with pytest.raises(TgError) as e:
                sim.replay(np.array([0.02, 0.03, bad]))
            assert e.value.code == _lib.TG_ERR_NONFINITE
            assert not np.isfinite(sim.get_state()).all(axis=0).any(), bad
        sim.set_state(pb.h, pb.hu, pb.hv)
        sim.run(2)
        sim.params.maxtime = -np.inf      # the next dt: maxtime - time
        with pytest.raises(TgError) as e:
            sim.step()
        assert e.value.code == _lib.TG_ERR_NONFINITE
        assert not np.isfinite(sim.get_state()).all(axis=0).any()


def test_members_beside_one_whose_dt_is_not_finite(oracle_lib):
    """An ensemble of more than 1024 tiles with an all-dry member: its dt is
    infinite and its cells become NaN; the others' states are their own."""
    mem = [small_flow_problem(70, 45, 3), small_flow_problem(40, 30, 3),
           small_flow_problem(192, 1500, 3)]
    for f in (mem[1].h, mem[1].hu, mem[1].hv):
        f[:] = 0.0
    _say("case dt edge: all-dry member of an ensemble")
    with Ensemble(mem, precision=_lib.TG_FP64, max_steps=4) as ens:
        with pytest.raises(TgError) as e:
            ens.run(3)
        assert e.value.code == _lib.TG_ERR_NONFINITE
        assert np.isnan(ens.member_state(1)).all()
        for b in (0, 2):
            orc = oracle_lib.Oracle.from_problem(mem[b])
            U = [mem[b].h.copy(), mem[b].hu.copy(), mem[b].hv.copy()]
            orc.run(U, 3)
            assert _same(ens.member_state(b), U), b
