"""Two levels per barrier of the mixed fused step on 64 x 11 tiles where the
level pair meets the free surface: where the pair (nz, nz + 1) falls in one
group (nz - kb even, kb the chunk's first level), the velocity images at
nz + 1 wait for level nz behind a barrier of their own.  (FP32 takes another
body on these tiles.)"""
import numpy as np
import pytest

import awpsgt
from test_gpu_batch import _make
from test_gpu_staged import _case, _equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("claim", ["0", "2"])
@pytest.mark.parametrize("nz,kc,chunks", [(33, "40", 1), (33, "12", 3), (34, "40", 1), (34, "12", 3), (34, "17", 2),
                                          (35, "18", 2)])
def test_mixed_pairs_meet_the_free_surface(nz, kc, chunks, claim, tmp_path, monkeypatch):
    d = _case(tmp_path, 70, 30, nz, 1, (35, 15, 6))
    monkeypatch.setenv("AWP_SCHEME", "split")
    ref = _make(d, awpsgt.AWP_STORAGE_MIXED)
    for k, v in (("SCHEME", "fused"), ("TILE_Y", "11"), ("PF", "3"), ("KC", kc), ("CLAIM", claim)):
        monkeypatch.setenv("AWP_" + k, v)
    r = _make(d, awpsgt.AWP_STORAGE_MIXED)
    assert r.scheme() == (True, 11, chunks)
    for x in (ref, r):
        x.step(9)
        x.step(x.p.nt)
        x.synchronize()
    assert np.any(ref.field("w1", 2)[-2] != 0)
    _equal(ref, r)
    ref.close()
    r.close()
