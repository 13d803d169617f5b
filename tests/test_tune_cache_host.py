"""The tuned-shape cache: entries of another kernel generation are not used, the
committed defaults stand in, and stored entries come back.  (No device.)"""
import json

import pytest

from qradient_amd import autotune


@pytest.fixture
def cache(tmp_path, monkeypatch):
    monkeypatch.setenv('QRADIENT_AMD_TUNE_CACHE', str(tmp_path / 'tune.json'))
    return tmp_path / 'tune.json'


def test_entries_of_another_generation_are_not_used(cache):
    k = autotune.key('mcclean', 21, 7, 'complex64', 'cnot')
    old = {'kmax': 11, 'cmin': 3, 'r_fwd': 4, 'r_rev': 4}
    cache.write_text(json.dumps({k: old}))
    assert autotune.lookup(k) is None
    cache.write_text(json.dumps({k: old, 'kernels': autotune.KERNELS - 1}))
    assert autotune.lookup(k) is None
    new = {'kmax': 12, 'cmin': 2, 'r_fwd': 4, 'r_rev': 4}
    autotune._store(k, new)
    assert autotune.lookup(k) == new
    other = autotune.qaoa_key(20, 8, 512, 'complex64')
    assert autotune.lookup(other) == json.load(open(autotune.DEFAULTS_PATH))[other]
    assert json.loads(cache.read_text())['kernels'] == autotune.KERNELS


def test_default_shape_is_the_untuned_tile():
    for n, dtype, kmax, cmin in ((14, 'complex64', 11, 2), (19, 'complex128', 11, 2), (20, 'complex64', 12, 2),
                                 (22, 'complex128', 12, 2), (23, 'complex64', 12, 2), (23, 'complex128', 12, 3),
                                 (30, 'complex64', 12, 3)):
        s = autotune.default_shape(n, dtype)
        assert (s['kmax'], s['cmin']) == (kmax, cmin), (n, dtype)
