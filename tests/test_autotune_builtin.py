"""The tuner offers the library's built-in choice of every knob whose named values leave a path that
the built-in choice may take (the split integration of few rays, shared direct sums and wide series
tiles have no value of their own), so a tuned call is never slower than an untuned one for want of
it; and a saved record that lacks a candidate is timed again."""
import json

import pytest

from radiobear_amd import autotune


@pytest.fixture
def timed(monkeypatch):
    """Times by launch shape: 1 ms for the built-in choice, 2 ms for a named one."""
    seen = []

    def run(launch):
        seen.append(dict(launch))

    def time_call(fn, reps=3, warmup=1):
        fn()
        return 2.0 if any(seen[-1].values()) else 1.0
    monkeypatch.setattr(autotune, 'time_call', time_call)
    monkeypatch.setattr(autotune, '_cache', {})
    return run


@pytest.mark.parametrize('knob', ['alpha_k', 'int_unroll', 'int_map', 'alpha_split', 'far_split', 'tan_split'])
def test_builtin_choice_is_a_candidate(timed, knob):
    launch, rec = autotune.tune(knob, 'few rays', timed)
    assert rec['best'] == 0 and launch == {knob: 0}


def test_integration_knobs_together(timed):
    launch, _ = autotune.tune_all(('int_unroll', 'int_map'), 'few rays', timed)
    assert launch == {'int_unroll': 0, 'int_map': 0}


def test_saved_record_without_a_candidate(timed, tmp_path):
    path = str(tmp_path / 'tuned.json')
    autotune.tune('int_map', 'shape', timed, path=path)
    with open(path) as fp:
        disk = json.load(fp)
    key, = disk
    assert autotune.tune('int_map', 'shape', None, path=path)[1] == disk[key]   # held: nothing is run
    autotune._cache.clear()
    del disk[key]['ms']['0']
    disk[key]['best'] = 2
    with open(path, 'w') as fp:
        json.dump(disk, fp)
    assert autotune.tune('int_map', 'shape', timed, path=path)[1]['best'] == 0
    assert autotune.tune('int_map', 'shape', timed, path=path, candidates=(1, 2))[1]['best'] == 0   # (as before)
