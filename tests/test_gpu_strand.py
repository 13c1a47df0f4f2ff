"""
The strand driver (lines of cells and uncoupled cells, each step shared by
four waves) at the edges of its tiles: one tile, one cell more, tiles of 32
and 48 cells with a short last one, runs that end on, before and after an
exchange. Double precision against the CPU oracle bit for bit, single
precision against the drivers that compute a whole cell per thread.
"""
import numpy as np
import pytest

import myokit_amd as myokit
from myokit_amd._err import DeviceError
from tests.helpers import Scenario, run_both

pytestmark = pytest.mark.gpu

DT = 0.005


def _scenario(n, field=False, rl=False, model='lr1991'):
    rng = np.random.default_rng(n)
    g = (rng.uniform(2, 12, n - 1), None) if field else None
    return Scenario(model, n, rl=rl, dt=DT, gx=9.5, paced=(4, 1, 0, 0),
                    conductance_field=g)


@pytest.mark.parametrize('n,field,rl', [
    (1, False, False), (2, False, False), (64, False, True),
    (65, False, False), (97, True, False), (161, True, True),
    (200, False, False)])
def test_fp64_bit_exact(n, field, rl):
    P, O = run_both(_scenario(n, field, rl), 6.0, myokit.DOUBLE_PRECISION,
                    log_interval=0.25)
    assert P['sim'].engine_driver() == 'strand'
    np.testing.assert_array_equal(P['V'], O['V'])
    np.testing.assert_array_equal(P['state'], O['state'])


def test_fp64_other_model_and_uncoupled():
    P, O = run_both(_scenario(70, model='br1977'), 4.0,
                    myokit.DOUBLE_PRECISION)
    assert P['sim'].engine_driver() == 'strand'
    np.testing.assert_array_equal(P['state'], O['state'])
    rng = np.random.default_rng(0)
    sc = Scenario('lr1991', 131, diffusion=False, dt=DT,
                  events=((1, 0, 0.5, 1000, 0),),
                  fields={'ina.gNa': 16 * rng.uniform(0.5, 2, 131)})
    P, O = run_both(sc, 4.0, myokit.DOUBLE_PRECISION)
    assert P['sim'].engine_timing()['launches'] == 2
    np.testing.assert_array_equal(P['V'], O['V'])
    np.testing.assert_array_equal(P['state'], O['state'])


def _run(s, steps, rows):
    v = [s.run_block(k * DT, ['membrane.V', 'ica.ICa', 'membrane.i_diff'],
                     log_interval=rows * DT) for k in steps]
    return [np.concatenate([b[q] for b in v]) for q in
            ('membrane.V', 'ica.ICa', 'membrane.i_diff')] \
        + [np.array(s.state())]


# 8,192 cells are 256 tiles of 32, one more makes 171 of 48; 49,152 cells are
# 1,024 tiles of 48, one more takes another driver
@pytest.mark.parametrize('n', [33, 64, 96, 513, 8192, 8193, 49152, 49153])
@pytest.mark.parametrize('rl', [False, True])
def test_fp32_equals_grid_across_run_lengths(n, rl):
    out = []
    for driver in ('auto' if n > 49152 else 'strand', 'grid'):
        # (asked for, the driver takes short batches too)
        s = _scenario(n, rl=rl).product(32)
        s.set_tuning(driver=driver)
        out.append(_run(s, (1, 15, 16, 17, 40, 33), 7))
        assert s.engine_driver() == (
            'grid' if driver == 'grid' or n > 49152 else 'strand')
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize('n', [64, 65, 49152, 49153])
def test_fp32_uncoupled_equals_cells(n):
    out = []
    for driver in ('auto', 'cells'):
        rng = np.random.default_rng(1)
        s = myokit.SimulationOpenCL(
            myokit.load_model('example'), myokit.pacing.blocktrain(1000, 0.5),
            ncells=n, diffusion=False)
        s.set_step_size(DT)
        s.set_field('ina.gNa', 16 * rng.uniform(0.5, 2, n))
        s.set_tuning(driver=driver)
        b = s.run_block(1.0, ['membrane.V', 'ica.ICa'], log_interval=0.2)
        # (the name of the layout, whichever kernel runs: one launch up to
        # the last row and one after it, or one per row)
        assert s.engine_driver() == 'cells'
        rows = len(b['time'])
        assert s.engine_timing()['launches'] == (
            2 if driver == 'auto' and n <= 49152 else rows + 1)
        out.append([b['membrane.V'], b['ica.ICa'], np.array(s.state())])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize('n', [40, 200])
def test_nan_ends_the_run_where_other_drivers_do(n):
    # a NaN in cell 0 at the second log row: the same rows, time and state
    out = []
    for driver in ('auto', 'grid'):
        s = _scenario(n).product(32)
        s.set_tuning(driver=driver)
        st = np.array(s.state()).reshape(n, -1)
        st[0, 7] = -1e-3        # log of a negative concentration
        s.set_state(st.reshape(-1))
        d = s.run(2.0, log=['membrane.V', 'engine.time'], log_interval=0.1,
                  report_nan=False)
        out.append((np.asarray(d['engine.time']),
                    np.asarray(d['0.membrane.V']), np.array(s.state())))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    assert len(out[0][0]) < 20 and np.isnan(out[0][2]).any()


def _nan_run(s, driver, st, rows=4):
    """The columns of a run of 10 ``rows`` steps from state ``st`` with a row
    every ``rows``, and the state it leaves."""
    s.set_tuning(driver=driver)
    s.reset()
    s.set_state(st.reshape(-1))
    d = s.run(10 * rows * DT, log=['membrane.V', 'ica.ICa', 'engine.time'],
              log_interval=rows * DT, report_nan=False)
    return [np.asarray(v) for v in d.values()] + [np.array(s.state())]


# a NaN in cell 0 that the first of the launch's rows finds, on lines of many
# tiles (the largest with several per CU) and on uncoupled cells, each after
# a run whose rows fill the log buffer
@pytest.mark.parametrize('n,coupled', [
    (65, True), (1000, True), (8193, True), (30000, True), (64, False),
    (1000, False), (49152, False)])
def test_nan_in_the_first_row(n, coupled):
    sc = _scenario(n) if coupled else Scenario(
        'lr1991', n, diffusion=False, dt=DT, events=((1, 0, 0.5, 1000, 0),))
    s = sc.product(32)
    st = np.array(s.state()).reshape(n, -1)
    bad = st.copy()
    bad[0] = np.nan
    out = []
    for driver in ('strand', 'grid') if coupled else ('auto', 'cells'):
        _nan_run(s, driver, st)
        out.append(_nan_run(s, driver, bad))
    assert len(out[0]) == 2 * n + 2
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    assert all(len(a) == 1 for a in out[0][:-1])
    assert np.isnan(out[0][-1]).any() and np.isfinite(out[0][-1][-8:]).all()


def test_exchange_timeout_of_the_repeated_steps_is_reported():
    # the steps up to a NaN's row are taken again: if a wait of theirs times
    # out (no polls allowed; the first launch has them all), the state is not
    # the run's, and the run must say so
    n = 1000
    s = _scenario(n).product(32)
    st = np.array(s.state()).reshape(n, -1)
    st[0, 7] = -1e-3
    _nan_run(s, 'strand', st, 20)
    s.set_engine_option('repeat_spins', 0)
    with pytest.raises(DeviceError, match='timed out'):
        _nan_run(s, 'strand', st, 20)
    s.set_engine_option('repeat_spins', 1 << 20)
    d = _nan_run(s, 'strand', st, 20)
    assert len(d[0]) == 2 and np.isnan(d[-1]).any()


@pytest.mark.parametrize('driver', ['strand', 'sheet', 'chain'])
def test_exchange_tags_start_again_before_they_overflow(driver):
    # the tags go on from run to run; near 2^31 the words are cleared and
    # they start again, in the first launch, a later one or a later run
    def make():
        if driver == 'chain':
            s = Scenario('lr1991', 300, connections=[
                (i, i + 1, 9.5) for i in range(299)],
                paced_list=[0, 1]).product(32)
        else:
            s = _scenario(300 if driver == 'strand' else (30, 20)).product(32)
        s.set_tuning(driver=driver)
        s.run_block(20 * DT, ['membrane.V'], log_interval=DT * 10)
        return s

    def go(s):
        b = [s.run_block(k * DT, ['membrane.V'], log_interval=DT * 20)
             ['membrane.V'] for k in (60, 90, 40)]
        assert s.engine_driver() == driver
        return np.concatenate(b)
    want = go(make())
    for left in (5, 50, 100, 150, 300):
        s = make()
        s.set_engine_option('step_tags', 2 ** 31 - 1 - left)
        np.testing.assert_array_equal(go(s), want)


@pytest.mark.parametrize('n,prec,least', [
    (200, 32, 24), (200, 64, 8), (1000, 32, 6), (1000, 64, 5), (20000, 32, 6),
    (64, 32, 1)])
def test_batches_too_short_for_a_cooperative_launch(n, prec, least):
    # a run's last row ends a batch, the steps after it are another one: with
    # a row at the first step only, one step and then steps - 1
    for steps in (least, least + 1):
        out = []
        for driver in ('auto', 'strand'):
            s = _scenario(n).product(prec)
            s.set_tuning(driver=driver)
            b = s.run_block(steps * DT, ['membrane.V'], log_interval=1000)
            assert s.engine_driver() == 'strand' and len(b['time']) == 1
            one = driver == 'strand' or steps > least or least == 1
            # the other driver's launches: one per step, of mk_block (up to
            # 512 cells) one per batch
            assert s.engine_timing()['launches'] == (
                min(steps, 2) if one or n <= 512 else steps)
            out.append((b['membrane.V'], np.array(s.state())))
        for a, b in zip(*out):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize('n', [16384, 16385])
def test_uncoupled_cells_of_a_model_that_splits_badly(n):
    # a model whose four groups share much of the work (nearly twice the cell
    # step in all) takes one tile per CU, then one thread per cell
    out = []
    for driver in ('auto', 'cells'):
        s = myokit.SimulationOpenCL(
            myokit.load_model('tests/data/dn-1985-normalised.mmt'),
            myokit.pacing.blocktrain(1000, 0.5), ncells=n, diffusion=False)
        s.set_step_size(DT)
        s.set_tuning(driver=driver)
        b = s.run_block(20 * DT, ['membrane.V'], log_interval=5 * DT)
        # one launch for the batch of all rows and one for the steps after
        # the last, or one per row
        rows = len(b['time'])
        assert s.engine_timing()['launches'] == (
            2 if driver == 'auto' and n == 16384 else rows + 1)
        out.append([b['membrane.V'], np.array(s.state())])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


def test_launches_grow_with_the_run():
    # a launch of the strand driver takes no more steps than the run before
    # it, at least 4,096: a NaN early in a long run does not cost the rest of
    # a full batch
    s = _scenario(65).product(32)
    s.run_block(40000 * DT, ['membrane.V'], log_interval=39999 * DT)
    # 4,096, 4,096, 8,192, 16,384 and 7,232 steps up to or past the last row,
    # which ends a batch
    assert s.engine_driver() == 'strand'
    assert s.engine_timing()['launches'] in (5, 6)
    s = _scenario(65).product(32)
    s.set_engine_option('batch_steps', 1000)
    s.run_block(4000 * DT, ['membrane.V'], log_interval=1e6)
    # the first row ends a batch of one step
    assert s.engine_timing()['launches'] == 5
