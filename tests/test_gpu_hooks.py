"""The source and trace work the two-stage kernels do between the steps of
one awp_step call (a run with one source) against the separate source kernel,
which does it after the last step of every call: a run stepped in one call
equals the same run stepped one step per call, bit for bit, in fields, SGT
series and trace -- body forces and surface sources, sources on the grid's
edges, on the last lane of a wave and the first of the next, on the traced
node, and two sources (which keep the separate kernel)."""
import numpy as np
import pytest

import awpsgt
import cases
from test_gpu_batch import _make

pytestmark = pytest.mark.gpu

NX, NY, NZ, ND = 70, 23, 27, 8
TRACED = (ND + 2, ND + 2, NZ + 1 - (ND + 2))   # as a source position (depth 1 is k = NZ)


@pytest.mark.parametrize("storage", [awpsgt.AWP_STORAGE_FP32, awpsgt.AWP_STORAGE_MIXED])
@pytest.mark.parametrize("igreen,src,o32v", [(1, (1, 1, 1), "0"), (1, (NX, NY, NZ), "1"), (2, (64, 12, 9), "0"),
                                             (3, (65, 5, 4), "0"), (3, TRACED, "1"), (2, TRACED, "0"),
                                             (4, (NX, 1, 1), "0"), (5, (1, NY, 1), "1"),
                                             (6, (64, NY, 1), "0")])
def test_one_call_equals_single_steps(igreen, src, o32v, storage, tmp_path, monkeypatch):
    monkeypatch.setenv("AWP_SCHEME", "split")
    monkeypatch.setenv("AWP_O32V", o32v)
    spec = cases.RunSpec(nx=NX, ny=NY, nz=NZ, dh=200.0, dt=0.01, nt=30, igreen=igreen, src=src, nd=ND, sigma=0.03,
                         t0=0.1, ntiskp_sgt=5)
    media = awpsgt.inputs.layered_media(NX, NY, NZ, [700.0, 1500.0, 2500.0])
    pts = awpsgt.inputs.random_cordfile_points(40, 5, (1, NX), (1, NY), (1, NZ))
    cases.write_case(str(tmp_path), spec, media, pts)
    runs = [_make(str(tmp_path), storage) for _ in range(2)]
    if src == TRACED and igreen == 2:
        # two sources on the traced node
        for r in runs:
            xyz, stf = awpsgt.read_source(str(tmp_path) + "/source", 1, r.p.nst)
            r.set_source(np.concatenate([xyz, xyz]), np.concatenate([stf, 0.5 * stf]))
            r.init()
    a, b = runs
    a.step(11)
    a.step(a.p.nt)
    for _ in range(b.p.nt):
        b.step(1)
    for r in runs:
        r.synchronize()
    assert a.progress() == b.progress() == (30, 6)
    assert np.any(a.field("u1") != 0)
    assert np.array_equal(a.sgt(), b.sgt())
    assert np.array_equal(a.trace()[0], b.trace()[0])
    assert src != TRACED or np.all(a.trace()[0][5:, igreen - 1] != 0)
    for f in ("u1", "v1", "w1", "xx", "yy", "zz", "xy", "xz", "yz", "r1", "r6"):
        k = 2 if f in ("u1", "v1", "w1", "zz", "xz", "yz") else 0
        assert np.array_equal(a.field(f, k), b.field(f, k)), f
    for r in runs:
        r.close()
