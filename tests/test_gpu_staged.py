"""The staged two-stage kernels (neighbours through LDS, 64 x 8 tiles) give
the bits of the kernels without LDS: fields, SGT series and trace of runs
whose sizes meet the edges of a tile (one column or row over and under, the
two ghost layers across a tile's edge) and of a z chunk (of 3 and 4 levels,
one chunk, a short last one), in every cache mode, with body and surface
sources; and of a batch of runs of different sizes, whose chunks follow the
tiles of all."""
import numpy as np
import pytest

import awpsgt
import cases
from test_gpu_batch import _make

pytestmark = pytest.mark.gpu

FIELDS = ("u1", "v1", "w1", "xx", "yy", "zz", "xy", "xz", "yz", "r1", "r2", "r3", "r4", "r5", "r6")
STORAGE = [awpsgt.AWP_STORAGE_FP32, awpsgt.AWP_STORAGE_MIXED]
# nx, ny, nz, levels a chunk, igreen, source, cache mode
SHAPES = [(64, 8, 24, None, 1, (64, 8, 5), "0"), (65, 9, 25, "4", 6, (65, 9, 1), "1"),
          (63, 23, 26, "3", 2, (1, 8, 3), "2"), (126, 16, 24, None, 5, (64, 16, 1), "3"),
          (127, 17, 31, "9", 3, (65, 9, 31), "0"), (129, 33, 24, "12", 4, (128, 1, 1), "2"),
          (130, 31, 25, "7", 6, (1, 31, 1), "3")]


def _case(d, nx, ny, nz, igreen, src):
    spec = cases.RunSpec(nx=nx, ny=ny, nz=nz, dh=200.0, dt=0.01, nt=15, igreen=igreen, src=src, nd=3, sigma=0.03,
                         t0=0.05, ntiskp_sgt=5)
    media = awpsgt.inputs.layered_media(nx, ny, nz, [700.0, 1500.0, 2500.0])
    media *= np.random.default_rng(nx).uniform(0.95, 1.05, media.shape).astype(np.float32)
    pts = awpsgt.inputs.random_cordfile_points(60, 5, (1, nx), (1, ny), (1, nz))
    cases.write_case(str(d), spec, media, pts)
    return str(d)


def _equal(a, b):
    assert np.array_equal(a.sgt(), b.sgt())
    assert np.array_equal(a.trace()[0], b.trace()[0])
    for f in FIELDS:
        k = 2 if f in ("u1", "v1", "w1", "zz", "xz", "yz") else 0
        assert np.array_equal(a.field(f, k), b.field(f, k)), f


@pytest.mark.parametrize("storage", STORAGE)
@pytest.mark.parametrize("nx,ny,nz,kc,igreen,src,mode", SHAPES)
def test_staged_equals_plain(nx, ny, nz, kc, igreen, src, mode, storage, tmp_path, monkeypatch):
    monkeypatch.setenv("AWP_SCHEME", "split")
    d = _case(tmp_path, nx, ny, nz, igreen, src)
    runs = []
    for staged in ("0", "1"):
        monkeypatch.setenv("AWP_STAGED", staged)
        if staged == "1":
            monkeypatch.setenv("AWP_CACHED", mode)
            if kc:
                monkeypatch.setenv("AWP_KC", kc)
        r = _make(d, storage)
        assert (r.scheme()[1] == 8) == (staged == "1")
        r.step(8)
        r.step(r.p.nt)
        r.synchronize()
        runs.append(r)
    assert np.any(runs[0].field("xx") != 0) and np.all(np.isfinite(runs[0].field("xx")))
    _equal(*runs)
    for r in runs:
        r.close()


@pytest.mark.parametrize("storage", STORAGE)
def test_staged_batch(storage, tmp_path, monkeypatch):
    monkeypatch.setenv("AWP_SCHEME", "split")
    dirs = [_case(tmp_path / str(n), *SHAPES[n][:3], *SHAPES[n][4:6]) for n in (1, 4, 6)]
    monkeypatch.setenv("AWP_STAGED", "0")
    refs = [_make(d, storage) for d in dirs]
    for r in refs:
        r.step(r.p.nt)
        r.synchronize()
    monkeypatch.setenv("AWP_STAGED", "1")
    runs = [_make(d, storage) for d in dirs]
    with awpsgt.Batch(runs) as b:
        assert b.launch()[0] == 8
        b.step(7)
        b.step(runs[0].p.nt)
    for a, r in zip(runs, refs):
        _equal(a, r)
        a.close()
        r.close()
