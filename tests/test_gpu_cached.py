"""The cache modes of the two-stage kernels (which pointwise accesses carry
the non-temporal hint) leave every result as it is: fields and SGT series of
runs in modes 1..3 equal those in mode 0 bit for bit, claimed and one block
per tile, and a batch's, whose mode follows its runs' sizes together."""
import numpy as np
import pytest

import awpsgt
from test_gpu_batch import _make

pytestmark = pytest.mark.gpu


def _done(d, storage, monkeypatch, mode, **env):
    monkeypatch.setenv("AWP_SCHEME", "split")
    monkeypatch.setenv("AWP_CACHED", mode)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    r = _make(d, storage)
    for k in env:
        monkeypatch.delenv(k)
    r.step(r.p.nt)
    r.synchronize()
    return r


def _same(a, b):
    assert np.array_equal(a.sgt(), b.sgt())
    for f in ("u1", "v1", "w1", "xx", "yy", "zz", "xy", "xz", "yz", "r1", "r2", "r3", "r4", "r5", "r6"):
        k = 2 if f in ("u1", "v1", "w1", "zz", "xz", "yz") else 0
        assert np.array_equal(a.field(f, k), b.field(f, k)), f


@pytest.mark.parametrize("storage", [awpsgt.AWP_STORAGE_FP32, awpsgt.AWP_STORAGE_MIXED])
@pytest.mark.parametrize("mode", ["1", "2", "3"])
def test_cache_modes_are_bit_identical(case_dirs, storage, mode, monkeypatch):
    d = case_dirs["g7_random_edges"][0]
    ref = _done(d, storage, monkeypatch, "0")
    for env in ({}, {"AWP_CLAIM": "2", "AWP_TILE_Y": "8"}, {"AWP_O32V": "1", "AWP_KC": "5"}):
        r = _done(d, storage, monkeypatch, mode, **env)
        _same(r, ref)
        r.close()
    ref.close()


@pytest.mark.parametrize("storage", [awpsgt.AWP_STORAGE_FP32, awpsgt.AWP_STORAGE_MIXED])
def test_batch_in_its_own_mode(case_dirs, storage, monkeypatch):
    dirs = [case_dirs[n][0] for n in ("g1_fx_layered", "g6_surface_zz")]
    refs = [_done(d, storage, monkeypatch, "0") for d in dirs]
    runs = [_make(d, storage) for d in dirs]
    with awpsgt.Batch(runs) as b:
        b.step(runs[0].p.nt)
    for r, ref in zip(runs, refs):
        _same(r, ref)
        r.close()
        ref.close()
