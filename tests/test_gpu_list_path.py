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
from helpers import small_flow_problem

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
