"""The stage kernel (fuse modes -1 and 2: a whole RK stage by tiles) against
the separate gradient, edge and update passes (mode 0) and the per-edge pass
(mode 1): the same bits, at the sizes where its tiles begin and end, and from
whatever reads the primitives that it does not keep in memory."""
import numpy as np
import pytest

from cfd2d import batch, native, renumber
from cfd2d import case as cases

pytestmark = pytest.mark.gpu

MODES = (0, 1, 2, None)


def _same(outs):
    for o in outs[1:]:
        for a, b in zip(outs[0], o):
            assert np.array_equal(a, b, equal_nan=True)


def _run(solver, mode, steps):
    solver.fuse_gradient(mode)
    solver.run(steps)
    return solver.state(), solver.flags(), np.array(solver.status())


# 40 cells are one tile; 42 two; 160 four; 40 960 the last size of 40-cell
# tiles; above, tiles grow up to what a workgroup can stage
@pytest.mark.parametrize("nx,ny", [(1, 1), (2, 1), (5, 4), (7, 3), (16, 5), (160, 128), (161, 128), (300, 290)])
@pytest.mark.parametrize("opts", [dict(), dict(limiter="MINMOD", gradient="LSQ", flux="HLLC", rk_stages=3),
                                  dict(viscous=True, flux="LAX", rk_stages=3)], ids=["plain", "limited", "viscous"])
def test_tile_sizes(nx, ny, opts):
    case = cases.shock_tube(nx, ny, seed=3, **opts)
    outs = []
    for mode in MODES:
        s = native.GpuSolver(case)
        outs.append(_run(s, mode, 3))
        s.close()
    _same(outs)


@pytest.mark.parametrize("make", [
    lambda: cases.periodic_pulse(2, seed=2), lambda: cases.periodic_pulse(3, seed=2),
    lambda: renumber.renumber_case(cases.periodic_pulse(48, seed=2), "random", seed=5)[0],
    # the general Riemann solver (not gamma = 1.4), the Roe flux, a steady
    # spectral time step, bounds that flag cells in three-stage steps
    lambda: cases.bump_channel(12, gam_flux=1.6, limiter="NONE"),
    lambda: cases.bump_channel(12, flux="ROE", gradient="LSQ", rk_stages=3),
    lambda: cases.bump_channel(21, steady=True, cfl_mode="SPECTRAL", flux="LAX"),
    lambda: cases.shock_tube(40, 6, seed=4, rk_stages=3, p_max=0.9, p_min=0.55),
    lambda: cases.shock_tube(40, 6, seed=4, mild=False, max_newton=200, limiter="MINMOD"),
], ids=["periodic2", "periodic3", "shuffled", "gamma16", "roe", "steady", "bounds", "sod"])
def test_families(make):
    case = make()
    outs = []
    for mode in MODES:
        s = native.GpuSolver(case)
        outs.append(_run(s, mode, 6))
        s.close()
    _same(outs)


def test_primitives_refreshed():
    """What reads the primitives after steps of the stage kernel sees the
    state's: diagnostics, wall force, time step, the implicit fill, a change of
    mode, a recorded run, the adjoint, the autotuner."""
    case = cases.bump_channel(11, flux="LAX", gradient="LSQ", limiter="NONE", rk_stages=3, outlet="BOUND_OUTLET")
    calls = [lambda s, m: s.gradients(), lambda s, m: s.edge_fluxes(), lambda s, m: s.residual(),
             lambda s, m: np.array(s.wall_force(m)), lambda s, m: s.implicit_assemble(steady=True, cfl=2.0)[2],
             lambda s, m: (s.calc_tau(), s.tau()[1])[1]]
    for call in calls:
        outs = []
        for mode in MODES:
            s = native.GpuSolver(case)
            mask = s.edge_mask("bump")
            _run(s, mode, 4)
            outs.append((call(s, mask),))
            s.close()
        _same(outs)
    outs = []
    for first, then in ((0, 0), (2, 0), (2, 1), (0, 2), (None, 1)):
        s = native.GpuSolver(case)
        mask = s.edge_mask("bump")
        s.fuse_gradient(first)
        s.run(3)
        s.fuse_gradient(then)
        s.run(3, graph=True)
        s.run(3, graph=True)
        J, gU, gb = s.adjoint(5, mask, 2)
        outs.append((s.state(), np.array(s.wall_force(mask)), np.array(J), gU, gb))
        s.close()
    _same(outs)
    s = native.GpuSolver(case)
    _run(s, 2, 4)
    before = s.state(), np.array(s.wall_force(s.edge_mask("bump"))), s.residual()
    s.run(2)
    s.set_state(before[0])
    s.autotune(2)
    _same([before, (s.state(), np.array(s.wall_force(s.edge_mask("bump"))), s.residual())])
    s.close()


def test_batch_tiles_do_not_mix_cases():
    """Overlapping channels in one batch: each case's cells, alone, give the same bits."""
    cs = [cases.bump_channel(ny, mach=m, seed=5 + ny, limiter="NONE") for ny, m in ((5, 0.4), (9, 0.8), (4, 1.5))]
    b = batch.BatchSolver(cs)
    b.run(5)
    for c, U in zip(cs, b.states()):
        s = native.GpuSolver(c)
        s.run(5)
        assert np.array_equal(U, s.state())
        s.close()
    b.close()


@pytest.mark.parametrize("flux", ["HLLC", "GODUNOV"])
@pytest.mark.parametrize("make", [
    lambda **k: cases.shock_tube(1, 1, seed=3, gradient="LSQ", rk_stages=3, **k),
    lambda **k: cases.shock_tube(2, 1, seed=3, **k), lambda **k: cases.shock_tube(7, 3, seed=3, rk_stages=3, **k),
    lambda **k: cases.shock_tube(161, 128, seed=3, gradient="LSQ", **k),
    lambda **k: cases.shock_tube(300, 290, seed=3, **k),
    lambda **k: cases.periodic_pulse(3, seed=2, **dict(k, viscous=False, gradient="GREEN_GAUSS")),
    lambda **k: cases.bump_channel(11, gradient="LSQ", limiter="NONE", outlet="BOUND_OUTLET", **k),
], ids=["2", "4", "42", "41k", "174k", "periodic", "bump"])
def test_adjoint_tiles(make, flux):
    """The reverse of HLLC and Godunov by tiles against the passes that form the
    cells' (P, G) adjoints in memory, as the geometry adjoint runs them: the
    same sums in another order.  4 steps of 3 stages and some 400 roundings per
    value and stage give 5e-13; ten times that for cancellation, and twice for
    the two sides."""
    s = native.GpuSolver(make(flux=flux))
    U = s.state()
    mask = (np.random.default_rng(1).random(s.mesh.ne) < 0.2).astype(np.int32)
    mask[0] = 1
    outs = []
    for adjoint in (s.adjoint, s.adjoint_geometry):
        s.set_state(U)
        outs.append(adjoint(4, mask, 2)[:3])
    assert abs(outs[0][0] - outs[1][0]) <= 1e-11 * abs(outs[1][0])
    if s.nc > 2:  # of the two cells' edges the mask has a vertical one, without lift
        assert np.abs(outs[1][1]).max() > 0
    for a, b in zip(outs[0][1:], outs[1][1:]):
        assert np.all(np.abs(a - b) <= 1e-11 * np.abs(b).max(initial=0.0))
    s.close()
