"""The scheme and launch shape a batch takes from its runs."""
import numpy as np
import pytest

import awpsgt
from test_gpu_batch import _make
from test_gpu_staged import _case, _equal

pytestmark = pytest.mark.gpu


def _runs(tmp_path, sizes, storage=awpsgt.AWP_STORAGE_FP32):
    return [_make(_case(tmp_path / str(n), *q, 1 + n % 3, (q[0] // 2, q[1] // 2, 5)), storage)
            for n, q in enumerate(sizes)]


def test_fused_batch_of_two_stage_runs(tmp_path, monkeypatch):
    """Small FP32 runs step two-stage by themselves; a fused batch of them
    takes the fused step's default shape, not their two-stage tiles."""
    runs, refs = (_runs(tmp_path, [(70, 34, 40), (48, 40, 32), (130, 25, 24)]) for _ in range(2))
    assert not any(r.scheme()[0] for r in runs)
    monkeypatch.setenv("AWP_BATCH_SCHEME", "fused")
    with awpsgt.Batch(runs) as b:
        assert b.fused() and b.launch()[:2] == (11, 3)
        b.step(6)
        b.step(runs[0].p.nt)
    for r, ref in zip(runs, refs):
        ref.step(ref.p.nt)
        ref.synchronize()
        _equal(ref, r)
        r.close()
        ref.close()


@pytest.mark.parametrize("storage", [awpsgt.AWP_STORAGE_FP32, awpsgt.AWP_STORAGE_MIXED])
def test_two_stage_batch_of_fused_runs(storage, tmp_path, monkeypatch):
    """The other way round: the shape a two-stage run of the sizes has."""
    sizes = [(70, 34, 40), (48, 40, 32), (130, 25, 24)]
    monkeypatch.setenv("AWP_SCHEME", "split")
    refs = _runs(tmp_path, sizes, storage)
    with awpsgt.Batch(refs) as b:
        want = b.launch()
        b.step(refs[0].p.nt)
    monkeypatch.setenv("AWP_SCHEME", "fused")
    runs = _runs(tmp_path, sizes, storage)
    monkeypatch.setenv("AWP_BATCH_SCHEME", "split")
    with awpsgt.Batch(runs) as b:
        assert not b.fused() and b.launch() == want
        b.step(7)
        b.step(runs[0].p.nt)
    for r, ref in zip(runs, refs):
        _equal(ref, r)
        r.close()
        ref.close()


def test_batch_scheme_by_all_runs_sizes(tmp_path, monkeypatch):
    """FP32 runs too small to step fused by themselves make a fused batch
    when they hold 25M points together; not below, and not where a run was
    put on the two-stage step."""
    sizes = [(300, 300, 100), (300, 280, 110), (250, 260, 120)]     # 9.0 + 9.24 + 7.8M
    runs = _runs(tmp_path, sizes)
    refs = _runs(tmp_path, sizes)
    assert not any(r.scheme()[0] for r in runs)
    with awpsgt.Batch(runs[:2]) as b:
        assert not b.fused()
    with awpsgt.Batch(runs) as b:
        assert b.fused() and b.launch()[:2] == (11, 3)
        b.step(7)
    for r in refs:
        r.set_scheme(False)
    with awpsgt.Batch(refs) as b:
        assert not b.fused()
        b.step(7)
    for r, ref in zip(runs, refs):
        for f in ("u1", "xx", "yz", "r1", "r6"):
            assert np.array_equal(r.field(f), ref.field(f)), f
        r.close()
        ref.close()


@pytest.mark.parametrize("scheme", ["fused", "split"])
def test_tuner_tries_the_shape_it_was_given(scheme, tmp_path, monkeypatch, capfd):
    """Tuning a batch that is on its default shape times that shape too (the
    staged two-stage tiles, the FP32 fused step with its z chunks)."""
    sizes = [(70, 34, 56), (48, 40, 32), (130, 25, 24)]
    refs = _runs(tmp_path, sizes)
    monkeypatch.setenv("AWP_STAGED", "1")
    runs = _runs(tmp_path, sizes)
    monkeypatch.setenv("AWP_BATCH_SCHEME", scheme)
    monkeypatch.setenv("AWP_TUNE_LOG", "1")
    with awpsgt.Batch(runs) as b:
        ty, pf, chunks = b.launch()
        assert (ty, pf) == ((11, 3) if scheme == "fused" else (8, 1))
        capfd.readouterr()
        b.tune(1)
        tried = [ln.split() for ln in capfd.readouterr().err.splitlines() if ln.startswith("awp_batch_tune first")]
        assert len(tried) > 20
        if scheme == "fused":
            # scheme, grid, "ty", rows, "xw", waves, "pf/unroll", depth, "chunks", chunks
            assert ["fused", "persistent", "ty", "11", "xw", "1", "pf/unroll", "3", "chunks", str(chunks)] in \
                [t[2:12] for t in tried]
        else:
            # staged: form 3; a run's chunks from the levels a chunk, at least 8 each
            kcs = [int(t[11]) for t in tried if t[2] == "two-stage" and t[13] == "3"]
            assert any(min((56 + kc // 2) // kc, 56 // 8) == chunks for kc in kcs)
        b.step(runs[0].p.nt)
    for r, ref in zip(runs, refs):
        ref.step(ref.p.nt)
        ref.synchronize()
        _equal(ref, r)
        r.close()
        ref.close()
