"""GPU: the steps at the sizes where their tiles end -- members of one
tile less, equal and more than each tile shape, the thinnest ones, whole rows
of boundary cells -- and on both sides of the line between a workgroup per
tile (1024 tiles) and the tile list, against the oracle.  Bar: states, dt and
lambda bit-identical (every product and sum in the reference's order), a step's
bed-friction gradient to 1e-12 of the absolute sum of its terms lambda .
dU/dphi (each is rounded some 30 times and they are added in another order); the
FP32 modes' bars stand at their tests."""
import sys

import numpy as np
import pytest

from discrete_adjoint_amd import _lib
from discrete_adjoint_amd.solver import Simulation
from helpers import analytic_problem, paraboloid

pytestmark = pytest.mark.gpu

SIZES = [(2, 2), (3, 2), (2, 5), (15, 17), (16, 16), (17, 15), (33, 8), (31, 9), (63, 5), (64, 4),
         (65, 3), (66, 33), (130, 70)]


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _problem(nx, ny, seed):
    rng = np.random.default_rng(seed)
    L, W = nx * 10.0, ny * 10.0
    pb = analytic_problem(nx, ny, 10.0, slope_x_deg=22.0, slope_y_deg=4.0,
                          h=paraboloid(0.5 * L, 0.5 * W, 0.45 * L + 5.0, 0.45 * W + 5.0, 6.0),
                          phi_int=32.0, phi_bed=18.0, nsteps=4, curv=(1e-3, -5e-4))
    n = pb.n
    pb.h *= rng.uniform(0.2, 1.0, n)
    pb.h[rng.uniform(size=n) < 0.15] = 0.0          # void cells inside the flow
    thin = rng.uniform(size=n) < 0.1
    pb.h[thin] = 1e-4 * rng.choice([0.5, 1.0, 1.5], thin.sum())   # below, at and above tiny
    pb.hu = pb.h * rng.normal(scale=9.0, size=n)    # sub- and supercritical faces
    pb.hv = pb.h * rng.normal(scale=9.0, size=n)
    still = rng.uniform(size=n) < 0.1
    pb.hu[still] = pb.hv[still] = 0.0
    return pb


def _terms(orc, pb, s, dt, lam):
    """The absolute sum of a reverse step's gradient terms."""
    return np.abs(lam * orc.dstep_dphi([pb.h, pb.hu, pb.hv], s, dt)).sum()


@pytest.mark.parametrize("tile", [(64, 4), (32, 8), (16, 16)])
@pytest.mark.parametrize("nx,ny", SIZES + [(513, 512)])
def test_reverse_step_at_tile_edges(oracle_lib, nx, ny, tile):
    _say(f"case reverse step {nx}x{ny} tile {tile}")
    pb = _problem(nx, ny, 100 * nx + ny)
    orc = oracle_lib.Oracle.from_problem(pb)
    rng = np.random.default_rng(nx + ny)
    lam = rng.normal(size=(3, pb.n)) * np.where(rng.uniform(size=pb.n) < 0.2, 0.0, 1.0)
    with Simulation(pb, max_steps=64, tile_x=tile[0], tile_y=tile[1]) as sim:
        for s, dt in ((3, 0.03), (60, 0.05)):
            ref, dphi = orc.adjoint_step([pb.h, pb.hu, pb.hv], s, dt, lam, want_dphi=True)
            got, g = sim.adjoint_step_grad(s, dt, lam)
            assert np.array_equal(got, np.asarray(ref).reshape(3, -1)), s
            assert np.array_equal(sim.adjoint_step(s, dt, lam), got), s
            assert abs(g - dphi) <= 1e-12 * _terms(orc, pb, s, dt, lam), s


@pytest.mark.parametrize("tile", [(0, 0), (64, 4), (32, 8), (16, 16)])
@pytest.mark.parametrize("nx,ny", SIZES + [(512, 512), (513, 512)])
def test_forward_steps_at_tile_edges(oracle_lib, nx, ny, tile):
    _say(f"case forward steps {nx}x{ny} tile {tile}")
    pb = _problem(nx, ny, 7 * nx + ny)
    if nx * ny > 100000:  # mostly empty, so that tiles are skipped, dry and wet
        j, i = np.divmod(np.arange(pb.n), nx)
        away = np.hypot(i - nx // 2, j - ny // 2) > 60
        pb.h[away] = pb.hu[away] = pb.hv[away] = 0.0
    orc = oracle_lib.Oracle.from_problem(pb)
    U = [pb.h.copy(), pb.hu.copy(), pb.hv.copy()]
    with Simulation(pb, max_steps=8, tile_x=tile[0], tile_y=tile[1]) as sim:
        for s in range(3):
            dt, _ = orc.step(U, s)
            assert sim.step().dt == dt, s
            for x, y in zip(sim.get_state(), U):
                assert np.array_equal(x, y) and np.array_equal(np.signbit(x), np.signbit(y)), s
        # the same steps as a run (clock and reduction cells start afresh),
        # then single steps on from it
        sim.set_state(pb.h, pb.hu, pb.hv)
        sim.run(2)
        sim.step()
        for x, y in zip(sim.get_state(), U):
            assert np.array_equal(x, y)


def test_reverse_sweep_on_both_launches(oracle_lib):
    """A sweep over 1024 tiles and one over more, checkpoints and recompute:
    lambda bit-identical to the oracle's, the gradient to rtol 1e-12."""
    for nx in (512, 513):
        _say(f"case reverse sweep {nx}x512")
        pb = _problem(nx, 512, nx)
        j, i = np.divmod(np.arange(pb.n), nx)
        away = np.hypot(i - nx // 2, j - 256) > 40
        pb.h[away] = pb.hu[away] = pb.hv[away] = 0.0
        w = pb.box_weights((nx * 2.0, nx * 6.0, 1500.0, 3500.0))
        orc = oracle_lib.Oracle.from_problem(pb)
        _, dts, lam_ref, dphi_ref = orc.forward_adjoint([pb.h.copy(), pb.hu.copy(), pb.hv.copy()],
                                                        5, w, want_dphi=True)
        for graph in (0, 1):
            with Simulation(pb, max_steps=5, checkpoint_every=2, use_graph=graph) as sim:
                sim.run(5)
                assert np.array_equal(sim.dt_record(), dts)
                lam, dphi = sim.dual_solver(w, want_dphi=True)
                assert np.array_equal(lam, lam_ref), (nx, graph)
                assert dphi == pytest.approx(dphi_ref, rel=1e-12), (nx, graph)


@pytest.mark.parametrize("thin", [0.1, 0.5])
@pytest.mark.parametrize("tile", [(64, 4), (32, 8), (16, 16)])
@pytest.mark.parametrize("nx,ny", SIZES + [(513, 512)])
def test_fp32_reverse_step_at_tile_edges(oracle_lib, nx, ny, tile, thin):
    """The FP32 gather and the FP64 pass over the cells next to a thin layer
    (eight lanes each or, where most cells are such, a thread each), on both
    launches, over void, thin and boundary cells.
    Bar: 1e-4 in norm, the one the sweeps of this mode are held to -- some
    hundred FP32 roundings of terms of the result's own size, with the cells
    whose 1/h is largest gathered in FP64.  A second step in a row reads the
    counts the first emptied."""
    _say(f"case fp32 reverse step {nx}x{ny} tile {tile} thin {thin}")
    pb = _problem(nx, ny, 11 * nx + ny)
    if thin > 0.1:
        more = np.random.default_rng(nx * ny).uniform(size=pb.n) < thin
        pb.h[more], pb.hu[more], pb.hv[more] = 5e-4, 3e-3, -2e-3
    if nx * ny > 100000:
        j, i = np.divmod(np.arange(pb.n), nx)
        away = np.hypot(i - nx // 2, j - ny // 2) > 60
        pb.h[away] = pb.hu[away] = pb.hv[away] = 0.0
    orc = oracle_lib.Oracle.from_problem(pb)
    rng = np.random.default_rng(nx + ny)
    lam = rng.normal(size=(3, pb.n)) * np.where(rng.uniform(size=pb.n) < 0.2, 0.0, 1.0)
    with Simulation(pb, max_steps=64, tile_x=tile[0], tile_y=tile[1],
                    precision=_lib.TG_FWD64_ADJ32) as sim:
        for s, dt in ((3, 0.03), (60, 0.05)):
            ref, dphi = orc.adjoint_step([pb.h, pb.hu, pb.hv], s, dt, lam, want_dphi=True)
            ref = np.asarray(ref).reshape(3, -1)
            got, g = sim.adjoint_step_grad(s, dt, lam)
            assert np.linalg.norm(got - ref) <= 1e-4 * np.linalg.norm(ref), s
            assert np.array_equal(sim.adjoint_step(s, dt, lam), got), s
            assert abs(g - dphi) <= 1e-4 * _terms(orc, pb, s, dt, lam), s


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("nx,ny", [(66, 33), (513, 512)])
def test_reverse_step_of_a_lambda_that_is_not_finite(oracle_lib, nx, ny, value):
    """An infinite or undefined entry of lambda^{s+1} (an adjoint that has
    overflowed) reaches every cell with h != 0 that the reference's full 3 x 3
    products carry it to: 0 * inf is not a zero that may be left out.  Void
    cells are +0.0 whatever lambda^{s+1} is."""
    _say(f"case reverse step {nx}x{ny} lambda {value}")
    pb = _problem(nx, ny, nx)
    if nx > 100:
        j, i = np.divmod(np.arange(pb.n), nx)
        away = np.hypot(i - nx // 2, j - ny // 2) > 40
        pb.h[away] = pb.hu[away] = pb.hv[away] = 0.0
    orc = oracle_lib.Oracle.from_problem(pb)
    rng = np.random.default_rng(nx + ny)
    on = pb.h != 0.0
    with Simulation(pb, max_steps=64) as sim:
        for k in range(3):
            lam = rng.normal(size=(3, pb.n))
            lam[k, rng.choice(np.flatnonzero(on), 5, replace=False)] = value
            lam[k, np.flatnonzero(on)[[0, -1]]] = value
            lam[k, [0, nx - 1, pb.n - 1]] = value   # the member's corners
            ref, _ = orc.adjoint_step([pb.h, pb.hu, pb.hv], 60, 0.05, lam)
            ref = np.where(on, ref, 0.0)
            assert 0 < np.count_nonzero(~np.isfinite(ref)) < 200
            for got in (sim.adjoint_step(60, 0.05, lam), sim.adjoint_step_grad(60, 0.05, lam)[0]):
                bad = np.argwhere((got != ref) & ~(np.isnan(got) & np.isnan(ref)))
                assert len(bad) == 0, (k, len(bad), bad[:3], got[tuple(bad[0])], ref[tuple(bad[0])])


@pytest.mark.parametrize("tile", [(64, 4), (32, 8), (16, 16)])
@pytest.mark.parametrize("nx,ny", [(66, 33), (513, 512)])
def test_fp32_gradient_term_of_one_cell(oracle_lib, nx, ny, tile):
    """lambda^{s+1} in one cell only: its gradient term alone, at the corners and
    edges of the tiles and of the member and next to thin cells, so that no term
    of a cell or of a face beyond the tile can be lost in a sum over all.
    Bar: 1e-4 of the term's three products, some hundred FP32 roundings each with
    up to ten times their size cancelling between the faces; every one of them
    far above it."""
    _say(f"case fp32 gradient of one cell {nx}x{ny} tile {tile}")
    pb = _problem(nx, ny, 3 * nx + ny)
    i0, j0 = (0, 0) if nx < 100 else (tile[0] * (256 // tile[0]), 256)
    if nx > 100:
        j, i = np.divmod(np.arange(pb.n), nx)
        away = np.hypot(i - i0, j - j0) > 80
        pb.h[away] = pb.hu[away] = pb.hv[away] = 0.0
    orc = oracle_lib.Oracle.from_problem(pb)
    at = [(i0 + a * tile[0] + di, j0 + b * tile[1] + dj)
          for a, b in ((0, 0), (1, 1)) for di in (0, tile[0] - 1) for dj in (0, tile[1] - 1)]
    at += [(0, 0), (nx - 1, 0), (0, ny - 1), (nx - 1, ny - 1)] if nx < 100 else []
    cells = [j * nx + i for i, j in at if i < nx and j < ny]
    thin = np.flatnonzero((pb.h > 0) & (pb.h < 1e-3))
    cells += [c + 1 for c in thin[::max(1, len(thin) // 6)] if c + 1 < pb.n]
    checked = 0
    with Simulation(pb, max_steps=64, tile_x=tile[0], tile_y=tile[1],
                    precision=_lib.TG_FWD64_ADJ32) as sim:
        for c in cells:
            lam = np.zeros((3, pb.n))
            lam[:, c] = 1.0, -0.7, 0.4
            _, dphi = orc.adjoint_step([pb.h, pb.hu, pb.hv], 60, 0.05, lam, want_dphi=True)
            _, g = sim.adjoint_step_grad(60, 0.05, lam)
            terms = _terms(orc, pb, 60, 0.05, lam)
            assert abs(g - dphi) <= 1e-4 * terms, (c % nx, c // nx, g, dphi)
            checked += abs(dphi) > 1e-2 * terms > 0
    assert checked >= 6
