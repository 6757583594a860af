"""GPU: a front that runs into new mark blocks (64 x 16 cells) over many steps.
Whether a workgroup leaves its tile alone hangs on marks that the workgroups of
the neighbouring tiles write in the same launch; the sweeps below meet every
state of them: blocks that the forward front enters, blocks that the reverse
sweep leaves, segments recomputed and whole runs repeated into buffers that hold
an earlier one, with a workgroup per tile (up to 1024 tiles) and with the tile
list.  Bar: bit-identical to the oracle, which has no marks, at every repeat."""
import sys

import numpy as np
import pytest

from discrete_adjoint_amd import _lib
from discrete_adjoint_amd.solver import Simulation
from helpers import analytic_problem, paraboloid

pytestmark = pytest.mark.gpu

NX, NY, STEPS = 128, 160, 140
# the block alone (80 tiles of 64 x 4 cells) and inside a mesh of 1125, where its
# surroundings stay void
MESHES = [(NX, NY, 0, 0), (192, 1500, 37, 1001)]


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _problem():
    """A pile thrown across the block, mostly up, where blocks are 16 cells
    high: its front enters several tiles and a new block every few steps."""
    L, W = NX * 5.0, NY * 5.0
    pb = analytic_problem(NX, NY, 5.0, slope_x_deg=6.0, slope_y_deg=26.0,
                          h=paraboloid(0.4 * L, 0.2 * W, 120.0, 50.0, 6.0), phi_int=33.0,
                          phi_bed=12.0, nsteps=STEPS, curv=(5e-4, -2e-4))
    pb.hu, pb.hv = 5.0 * pb.h, 25.0 * pb.h
    return pb


def _weights(pb):
    """Depth in a box that the front enters in the second half."""
    L, W = NX * pb.dx, NY * pb.dy
    return pb.box_weights((0.3 * L, 0.7 * L, 0.29 * W, 0.9 * W)).reshape(3, -1)


def _grow(f, nx, ny, i0, j0):
    """[k, NY * NX] fields of the block as those of a mesh that holds it at (i0,
    j0), zero elsewhere."""
    f = np.atleast_2d(f)
    out = np.zeros((len(f), ny, nx))
    out[:, j0:j0 + NY, i0:i0 + NX] = f.reshape(len(f), NY, NX)
    return out.reshape(len(f), -1)


def _embedded(pb, nx, ny, i0, j0):
    big = analytic_problem(nx, ny, pb.dx, slope_x_deg=6.0, slope_y_deg=26.0, phi_int=33.0,
                           phi_bed=12.0, nsteps=STEPS, curv=(5e-4, -2e-4))
    big.h, big.hu, big.hv = _grow([pb.h, pb.hu, pb.hv], nx, ny, i0, j0)
    return big


@pytest.fixture(scope="module")
def oracle_run(oracle_lib):
    pb = _problem()
    orc = oracle_lib.Oracle.from_problem(pb)
    return orc.forward_adjoint([pb.h.copy(), pb.hu.copy(), pb.hv.copy()], STEPS, _weights(pb))


def test_front_crosses_blocks(oracle_run):
    pb, UN = _problem(), oracle_run[0]
    before, after = (np.unique(np.flatnonzero(h > 0) // NX // 16) for h in (pb.h, UN[0]))
    assert after.max() >= before.max() + 2 and len(after) < NY // 16
    edge = UN[0].reshape(NY, NX)
    assert not edge[:2].any() and not edge[-2:].any()      # (the embedding needs that)
    assert not edge[:, :2].any() and not edge[:, -2:].any()
    inside = (_weights(pb)[0] * UN[0]).sum() / (25.0 * UN[0].sum())
    assert 0.2 < inside < 0.9 and _weights(pb)[0][pb.h > 0].max() == 0.0


@pytest.mark.parametrize("tile", [(0, 0), (64, 4), (32, 8), (16, 16)])
@pytest.mark.parametrize("nx,ny,i0,j0", MESHES)
def test_front_into_new_blocks(oracle_run, nx, ny, i0, j0, tile):
    _say(f"case front {nx}x{ny} tile {tile}")
    pb = _embedded(_problem(), nx, ny, i0, j0)
    w = _grow(_weights(_problem()), nx, ny, i0, j0)
    UN, dts, lam_ref, _ = oracle_run
    UN, lam_ref = _grow(UN, nx, ny, i0, j0), _grow(lam_ref.reshape(3, -1), nx, ny, i0, j0)
    for k, graph in ((9, 0), (9, 1), (1, 0)):
        with Simulation(pb, checkpoint_every=k, use_graph=graph, tile_x=tile[0],
                        tile_y=tile[1]) as sim:
            for rep in range(2):  # the second sweep starts from the first one's buffers
                sim.set_state(pb.h, pb.hu, pb.hv)
                sim.run()
                assert np.array_equal(sim.dt_record(), dts), (k, graph, rep)
                assert np.array_equal(sim.get_state(), UN), (k, graph, rep)
                for _ in range(2):
                    lam, _ = sim.dual_solver(w, want_dphi=bool(rep))
                    assert np.array_equal(lam, lam_ref), (k, graph, rep)


def test_a_tile_is_left_alone_by_its_own_mark(oracle_lib):
    """Each tile's workgroup decides by the mark of its own tile: where a block
    of the buffer a pass writes still holds an earlier run's cells in one of its
    four tiles, that tile is written and the other three are left alone, however
    far their neighbours have come.  (A decision by the block's whole word would
    also write the other three, or not, by who is first.)"""
    nx, ny = 256, 96
    _say("case a tile's own mark")

    def pile(i, j):  # 2 x 2 cells at rest: one step on they reach one cell around
        pb = analytic_problem(nx, ny, 5.0, slope_x_deg=20.0, phi_int=33.0, phi_bed=16.0, nsteps=2)
        h = np.zeros((ny, nx))
        h[j:j + 2, i:i + 2] = 2.0
        return h.reshape(-1)

    z = np.zeros(nx * ny)
    # inside the second tile of a block; in a block with none of those around it
    here, there = pile(150, 49), pile(30, 9)
    pb = analytic_problem(nx, ny, 5.0, slope_x_deg=20.0, phi_int=33.0, phi_bed=16.0, nsteps=2)
    short = []
    with Simulation(pb, checkpoint_every=1, tile_x=64, tile_y=4, use_graph=0) as sim:
        for first in (there, here):
            w = np.stack([np.ones(nx * ny), z, z])
            sim.set_state(first, z, z)
            sim.run(2)
            sim.dual_solver(w)
            sim.set_state(there, z, z)
            sim.instrument(True)
            sim.run(1)
            sim.dual_solver(w)
            _, launches, _, cells = sim.instrumentation()
            sim.instrument(False)
            assert launches[1] == launches[2] == 1
            short.append(cells)
    assert short[1][1] - short[0][1] == 64 * 4   # update
    assert short[1][2] - short[0][2] == 64 * 4   # reverse step


@pytest.mark.parametrize("precision", [_lib.TG_FP32, _lib.TG_MIXED, _lib.TG_FWD64_ADJ32])
@pytest.mark.parametrize("nx,ny,i0,j0", MESHES)
def test_front_in_fp32_modes(nx, ny, i0, j0, precision):
    """The FP32 reverse sweeps, whose marks leave tiles alone, equal their own
    single reverse steps from uploaded states, which have no marks, bit for bit:
    a cell left unwritten under a mark that says +0.0 would keep an earlier
    step's lambda."""
    _say(f"case fp32 front {nx}x{ny} precision {precision}")
    pb = _embedded(_problem(), nx, ny, i0, j0)
    w = _grow(_weights(_problem()), nx, ny, i0, j0)
    with Simulation(pb, precision=precision, checkpoint_every=9) as sim:
        for _ in range(2):  # the second time over the buffers of the first
            sim.set_state(pb.h, pb.hu, pb.hv)
            sim.run()
            got = [sim.dual_solver(w, want_dphi=d)[0] for d in (False, True)]
        dts = sim.dt_record()
        with Simulation(pb, precision=precision, max_steps=STEPS) as one:
            lam = w
            for s in range(STEPS - 1, -1, -1):
                one.set_state(*sim.trajectory_state(s))
                lam = one.adjoint_step(s, dts[s], lam)
    assert np.isfinite(lam).all() and np.abs(lam).max() > 1.0
    for g in got:
        assert np.array_equal(g, lam)
