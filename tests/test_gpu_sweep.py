"""The FP32 fused step on 64 x 11 tiles (neighbours through LDS, one wait a
level) gives the bits of the two-stage kernels: fields, SGT series and trace
of runs whose sizes meet the edges of a tile (one row or column over and
under, the halo rows and columns and their ghost layers in the next tile) and
of a z chunk (one, two, a short last one), one block per tile and claimed."""
import numpy as np
import pytest

import awpsgt
from test_gpu_batch import _make
from test_gpu_staged import _case, _equal

pytestmark = pytest.mark.gpu

# nx, ny, nz, levels a chunk, igreen, source
SHAPES = [(64, 11, 24, None, 1, (64, 11, 5)), (65, 12, 33, "17", 6, (65, 12, 1)), (63, 23, 48, "16", 2, (1, 11, 17)),
          (66, 10, 40, "20", 5, (64, 10, 1)), (126, 22, 37, "19", 3, (65, 12, 19)), (130, 34, 50, "25", 4, (128, 1, 1)),
          (128, 45, 32, "16", 1, (66, 34, 16))]


@pytest.mark.parametrize("claim", ["0", "2"])
@pytest.mark.parametrize("nx,ny,nz,kc,igreen,src", SHAPES)
def test_sweep_equals_two_stage(nx, ny, nz, kc, igreen, src, claim, tmp_path, monkeypatch):
    d = _case(tmp_path, nx, ny, nz, igreen, src)
    runs = []
    for scheme in ("split", "fused"):
        monkeypatch.setenv("AWP_SCHEME", scheme)
        if scheme == "fused":
            monkeypatch.setenv("AWP_CLAIM", claim)
            if kc:
                monkeypatch.setenv("AWP_KC", kc)
        r = _make(d, awpsgt.AWP_STORAGE_FP32)
        assert r.scheme()[0] == (scheme == "fused") and (scheme == "split" or r.scheme()[1] == 11)
        r.step(8)
        r.step(r.p.nt)
        r.synchronize()
        runs.append(r)
    assert np.any(runs[0].field("xx") != 0)
    _equal(*runs)
    for r in runs:
        r.close()
