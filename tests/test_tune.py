"""
Autotuner logic without a device: candidate sets per coupling and
geometry, tuning validation, and the choice cache.
"""
import pytest

import myokit_amd as myokit
from myokit_amd import tune


def sim(ncells, **kw):
    return myokit.SimulationOpenCL(myokit.load_model('example'),
                                   myokit.pacing.blocktrain(1000, 2),
                                   ncells=ncells, **kw)


def test_candidates_by_coupling():
    c = tune.candidates(sim((256, 256)))
    drivers = {x['driver'] for x in c}
    assert drivers == {'block', 'grid', 'sheet'}
    sheet = [x for x in c if x['driver'] == 'sheet']
    assert {x['sheet_cpt'] for x in sheet} <= set(
        myokit_amd_choices()) and all(x['block_threads'] == 256
                                      for x in sheet)
    c = tune.candidates(sim(100))
    assert {x['driver'] for x in c} == {'block', 'grid'}
    c = tune.candidates(sim(100, diffusion=False))
    assert {x['driver'] for x in c} == {'cells', 'grid'}
    s = sim(10)
    s.set_connections([(i, i + 1, 1.0) for i in range(9)])
    c = tune.candidates(s)
    assert {x['driver'] for x in c} == {'block', 'grid', 'chain'}
    from myokit_amd import _kernelgen
    assert all(x['chain_cpt'] in _kernelgen.CHAIN_CPT_CHOICES
               for x in c if x['driver'] == 'chain')
    for x in tune.candidates(sim((64, 64), precision=64)):
        if x['driver'] == 'sheet':
            assert x['sheet_cpt'] in (2, 4)
    g64 = {x['grid_waves'] for x in tune.candidates(
        sim((64, 64), precision=64)) if x['driver'] == 'grid'}
    assert g64 == {0, 4, 5, 6}
    assert {x['grid_waves'] for x in tune.candidates(sim((64, 64)))
            if x['driver'] == 'grid'} == {0}


def myokit_amd_choices():
    from myokit_amd import _kernelgen
    return _kernelgen.SHEET_CPT_CHOICES


def test_set_tuning_validation():
    s = sim(50)
    assert s.tuning()['driver'] == 'auto'
    with pytest.raises(ValueError):
        s.set_tuning(block_threads=100)
    with pytest.raises(ValueError):
        s.set_tuning(sheet_cpt=3)
    with pytest.raises(ValueError):
        s.set_tuning(sheet_waves=0)
    with pytest.raises(ValueError):
        s.set_tuning(driver='fast')
    with pytest.raises(ValueError):
        s.set_tuning(adjoint_waves=9)
    with pytest.raises(ValueError):
        s.set_tuning(chain_cpt=3)
    with pytest.raises(ValueError):
        s.set_tuning(chain_waves=9)
    with pytest.raises(ValueError):
        s.set_tuning(adjoint_cpt=3)
    with pytest.raises(ValueError):
        s.set_tuning(grid_waves=9)
    s.set_tuning(driver='grid', block_threads=128, sheet_cpt=8,
                 sheet_waves=3, adjoint_waves=4, chain_cpt=1, chain_waves=6,
                 adjoint_cpt=4, grid_waves=5)
    t = s.tuning()
    assert t == {'driver': 'grid', 'block_threads': 128, 'sheet_cpt': 8,
                 'sheet_waves': 3, 'adjoint_waves': 4, 'chain_cpt': 1,
                 'chain_waves': 6, 'adjoint_cpt': 4, 'grid_waves': 5}


def test_cache_round_trip(tmp_path, monkeypatch):
    monkeypatch.setenv(tune.CACHE_ENV, str(tmp_path / 'tune.json'))
    s = sim((32, 32))
    assert tune.apply_cached(s) is None
    cfg = {'driver': 'grid', 'block_threads': 512}
    tune._store(tune._key(s), cfg)
    t = sim((32, 32))
    assert tune.apply_cached(t) == cfg
    assert t.tuning()['block_threads'] == 512
    # another geometry or precision has its own entry
    assert tune.apply_cached(sim((32, 16))) is None
    assert tune.apply_cached(sim((32, 32), precision=64)) is None


def test_tuned_kernel_source_has_tile_shape():
    from myokit_amd import _kernelgen
    from myokit_amd.simulation import _prepare_cell_model
    cm = _prepare_cell_model(myokit.load_model('example'), rl=True,
                             diffusion=True, fields=[], quantities=[])
    src = _kernelgen.generate_kernel(cm, 32, 1, tile_cpt=8, tile_waves=3)
    assert '#define MK_SCPT 8' in src and '#define MK_SWAVES 3' in src
    with pytest.raises(ValueError):
        _kernelgen.generate_kernel(cm, 32, 1, tile_cpt=16)


def test_grid_register_budget_in_kernel_source():
    # waves per SIMD -> workgroups per CU of the grid driver's launch
    # bounds (4 SIMDs per CU): 5 waves of 256-thread workgroups is 5 per
    # CU, of 1024-thread workgroups 1; 0 leaves the bound to the compiler
    from myokit_amd import _kernelgen
    from myokit_amd.simulation import _prepare_cell_model
    cm = _prepare_cell_model(myokit.load_model('example'), rl=True,
                             diffusion=True, fields=[], quantities=[])
    for threads, waves, blocks in ((256, 5, 5), (128, 4, 8), (1024, 5, 1),
                                   (256, 0, 0)):
        src = _kernelgen.generate_kernel(cm, 64, 1, threads,
                                         grid_budget=waves)
        assert '#define MK_GBLOCKS %d' % blocks in src
    with pytest.raises(ValueError):
        _kernelgen.generate_kernel(cm, 64, 1, grid_budget=9)


def test_sheet_tiles_follow_the_size():
    # the fewest cells per thread whose tiles are all sure to be resident:
    # 64 x 4 cpt cells each, 256 CUs times the waves of the budget
    from myokit_amd import _kernelgen as k
    for prec, one, two in ((32, 1536, 1280), (64, 1024, 768)):
        assert k.sheet_waves(prec, 1) * 256 == one
        assert k.sheet_waves(prec, 2) * 256 == two
        # one column of tiles, exactly full and one row more
        assert k.sheet_cpt(prec, (64, 4 * one)) == 1
        assert k.sheet_cpt(prec, (64, 4 * one + 1)) == 2
        assert k.sheet_cpt(prec, (1, 8 * two)) == 2
        assert k.sheet_cpt(prec, (65, 4 * two + 1)) == 4
        assert k.sheet_cpt(prec, (5000, 5000)) == 4
        assert k.sheet_cpt(prec) == 1
        # large cell models keep the wider register budget
        assert k.sheet_waves(prec, 1, 30) == k.sheet_waves(prec, 4, 30) \
            == k.sheet_waves(prec, 4)
    assert sim((100, 70)).tuning()['sheet_cpt'] == 1
    # a register budget that is given counts in place of the rule's
    s = sim((600, 600))
    assert s.tuning()['sheet_cpt'] == 1
    for waves, cpt in ((3, 2), (2, 4), (6, 1)):
        s.set_tuning(sheet_waves=waves)
        assert s.tuning()['sheet_cpt'] == cpt
    assert sim((1024, 1024)).tuning()['sheet_cpt'] == 4


def test_reverse_sheet_tiles_follow_the_size():
    from myokit_amd import _kernelgen as k
    for prec, most in ((32, 512), (64, 256)):
        assert k.adjoint_sheet_waves(prec) * 256 == most
        assert k.adjoint_sheet_cpt(prec) == 1
        assert k.adjoint_sheet_cpt(prec, (64, 4 * most)) == 1
        assert k.adjoint_sheet_cpt(prec, (1000, 1)) == 1
        assert k.adjoint_sheet_cpt(prec, (1000,)) == 0
    assert k.adjoint_sheet_cpt(64, (64, 1025)) == 0
    assert k.adjoint_sheet_cpt(32, (64, 2049)) == 2
    assert k.adjoint_sheet_cpt(32, (65, 2049)) == 0
    assert k.adjoint_sheet_cpt(32, (1024, 1024)) == 8
    assert k.adjoint_sheet_cpt(32, (1025, 1024)) == 0
    # the tiles of 8 cells per thread are the faster from 900,000 cells on
    assert k.adjoint_sheet_cpt(32, (960, 960)) == 8
    assert k.adjoint_sheet_cpt(32, (960, 896)) == 0
    # 0 leaves the persistent kernel out of the text
    s = sim((800, 800), rl=True)
    assert s.tuning()['adjoint_cpt'] is None
    cm = k.CellModel(s._model, s._bound_variables, s._rl_states, [], [])
    src = k.generate_kernel(cm, 32, 1, adjoint=True, adjoint_cpt=0)
    assert '#define MK_ADJ_SHEET 0' in src
