"""
The persistent sheet's tiles at their edges: sheets whose sizes leave one
column, one row or a few lanes in the last tile, each tile height, and
conductance fields, in double precision against the CPU oracle bit for bit
and in single precision against the one-step grid driver.
"""
import numpy as np
import pytest

import myokit_amd as myokit
from tests.helpers import Scenario, run_both

pytestmark = pytest.mark.gpu

# widths with 1, 8 and 64 cells in the last tile column; heights with one
# row in the last tile row of each tile height, and a sheet of one tile
SHAPES = [(65, 33), (72, 17), (128, 9), (40, 20)]


def _scenario(shape, field, rl=True):
    nx, ny = shape
    rng = np.random.default_rng(nx + 7 * ny)
    g = None
    if field:
        gx = rng.uniform(2, 12, (ny, nx - 1))
        gy = rng.uniform(2, 12, (ny - 1, nx))
        gx[:, nx // 2] = 0.0
        g = (gx, gy)
    return Scenario('lr1991', shape, rl=rl, dt=0.01, gx=9.5, gy=6.0,
                    paced=(4, ny, 0, 0), conductance_field=g)


@pytest.mark.parametrize('shape', SHAPES)
@pytest.mark.parametrize('field', [False, True])
def test_fp64_sheet_edges_bit_exact(shape, field):
    P, O = run_both(_scenario(shape, field), 4.0, myokit.DOUBLE_PRECISION)
    assert P['sim'].engine_driver() == 'sheet'
    assert P['sim'].tuning()['sheet_cpt'] == 1
    np.testing.assert_array_equal(P['V'], O['V'])
    np.testing.assert_array_equal(P['state'], O['state'])


@pytest.mark.parametrize('cpt', [1, 2, 4])
@pytest.mark.parametrize('field', [False, True])
def test_fp32_every_tile_height_equals_grid(cpt, field):
    # the same operations in the same order in every driver and tile height
    for shape in SHAPES:
        V = []
        for kw in ({'driver': 'sheet', 'sheet_cpt': cpt}, {'driver': 'grid'}):
            s = _scenario(shape, field, rl=False).product(32)
            s.set_tuning(**kw)
            b = s.run_block(3.0, ['membrane.V'], log_interval=0.5)
            assert s.engine_driver() == kw['driver']
            V.append((b['membrane.V'], np.array(s.state())))
        np.testing.assert_array_equal(V[0][0], V[1][0])
        np.testing.assert_array_equal(V[0][1], V[1][1])


@pytest.mark.parametrize('shape', SHAPES)
@pytest.mark.parametrize('cpt', [1, 2, 8])
def test_reverse_sheet_edges_equal_one_step_kernel(shape, cpt):
    # double precision: the loss and the field gradients bit for bit, the
    # conductances' (whose terms are grouped by tile) to 1e-12
    from myokit_amd.adjoint import TissueAdjoint
    nx, ny = shape
    res = []
    for sheet in (1, 0):
        s = _scenario(shape, False).product(64)
        s.set_field('ina.gNa', np.linspace(14, 18, nx * ny).reshape(ny, nx))
        s.set_tuning(adjoint_cpt=cpt)
        s.set_engine_option('adj_sheet', sheet)
        adj = TissueAdjoint(s, [(0, 0), (nx - 1, ny - 1)],
                            checkpoint_every=23)
        target = np.full((adj.n_steps(0.6), 2), -40.0)
        loss, g, dgx, dgy = adj.loss_and_gradient(0.6, target)
        kind = adj.reverse_kernel()[0]
        assert (kind == 'sheet') == bool(sheet), kind
        res.append((loss, g['ina.gNa'].copy(), dgx, dgy))
    assert res[0][0] == res[1][0]
    np.testing.assert_array_equal(res[0][1], res[1][1])
    assert res[0][2] == pytest.approx(res[1][2], rel=1e-12)
    assert res[0][3] == pytest.approx(res[1][3], rel=1e-12)


@pytest.mark.parametrize('field', [False, True])
@pytest.mark.parametrize('shape', [(1009, 601), (601, 1021)])
def test_fp32_two_steps_per_launch_equal_one(shape, field):
    # large sheets on the grid driver: a run that logs every step takes
    # single steps, one that logs every 5 or never takes pairs and odd ones
    out = []
    for every in (1, 5, 1000):
        s = _scenario(shape, field).product(32)
        s.set_tuning(driver='grid')
        b = s.run_block(0.21, ['membrane.V'], log_interval=every * 0.01)
        assert s.engine_driver() == 'grid'
        # 21 steps: one launch each where all log; the first alone and ten
        # pairs where none but the first does
        launches = s.engine_timing()['launches']
        assert launches == {1: 21, 5: launches, 1000: 11}[every]
        assert every != 5 or 13 <= launches <= 15
        out.append((b['membrane.V'][::5 // min(every, 5)], np.array(s.state())))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
    np.testing.assert_array_equal(out[0][1], out[2][1])


@pytest.mark.parametrize('shape,prec,row', [
    ((40, 20), 32, 6), ((40, 20), 64, 10), ((200, 97), 32, 6),
    ((257, 257), 64, 8)])
@pytest.mark.parametrize('field', [False, True])
def test_rows_too_close_for_a_sheet_launch(shape, prec, row, field):
    # rows every `row` steps take a launch each (the first row's step one),
    # closer ones one per step; equal results
    dt = 1.0 / 128          # times are exact
    for every, steps in ((row, 6 * row + 1), (row - 1, 6 * row - 5)):
        out = []
        for driver in ('auto', 'grid'):
            s = _scenario(shape, field).product(prec)
            s.set_tuning(driver=driver)
            s.set_step_size(dt)
            b = s.run_block(steps * dt, ['membrane.V'],
                            log_interval=every * dt)
            if driver == 'auto':
                assert s.engine_driver() == 'sheet'
                assert s.engine_timing()['launches'] == (
                    1 + 6 if every == row else steps)
            out.append((b['membrane.V'], np.array(s.state())))
        for a, b in zip(*out):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize('shape,field,driver', [
    ((600, 600), False, 'grid'), ((600, 600), True, 'grid'),
    ((301, 217), True, 'sheet')])
def test_sheet_tiles_that_spill_leave_the_grid_driver(shape, field, driver):
    # 16 states in double precision: with 4 cells per thread the sheet kernel
    # keeps half its registers in scratch memory; asked for, it runs
    nx, ny = shape
    out = []
    for d in ('auto', 'sheet'):
        s = myokit.SimulationOpenCL(
            myokit.load_model('tests/data/dn-1985-normalised.mmt'),
            myokit.pacing.blocktrain(1000, 2), ncells=shape, precision=64)
        s.set_step_size(0.005)
        s.set_paced_cells(4, ny, 0, 0)
        if field:
            s.set_conductance_field(np.full((ny, nx - 1), 2.0),
                                    np.full((ny - 1, nx), 1.5))
        else:
            s.set_conductance(2.0, 1.5)
        s.set_tuning(driver=d)
        b = s.run_block(0.1, ['membrane.V'], log_interval=0.06)
        assert s.engine_driver() == (driver if d == 'auto' else 'sheet')
        out.append((b['membrane.V'], np.array(s.state())))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize('waves', [1, 2, 3])
def test_tile_follows_a_given_register_budget(waves):
    # 1,024 tiles of 64 x 4 cells need the rule's four waves: a smaller budget
    # takes larger tiles, so that the driver asked for is not refused
    s = _scenario((512, 512), False).product(64)
    s.set_tuning(driver='sheet', sheet_waves=waves)
    s.run_block(0.2, ['membrane.V'], log_interval=1)
    assert s.engine_driver() == 'sheet'
