"""SGT output larger than the pinned staging buffer (several pieces, several
host threads): sgt(), the raw file, the RWG-order file and the FP16 file with
its reader agree with one another and with the formats' rules, with dropped
points at the ends and inside the pieces and a partial last buffer."""
import os

import numpy as np
import pytest

import awpsgt
import cases
from test_gpu_batch import _make

pytestmark = pytest.mark.gpu

NX, NY, NZ, NT, WS = 48, 40, 32, 45, 20      # 45 samples: two full buffers of 20, five dropped


@pytest.fixture(scope="module")
def finished(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("out"))
    spec = cases.RunSpec(nx=NX, ny=NY, nz=NZ, dh=200.0, dt=0.01, nt=NT, igreen=3, src=(24, 20, 4), nd=8, sigma=0.03,
                         t0=0.12, ntiskp_sgt=1, write_step=WS)
    media = awpsgt.inputs.layered_media(NX, NY, NZ, [700.0, 1500.0, 2500.0])
    n = 40000
    rng = np.random.default_rng(4)
    pts = np.stack([rng.integers(1, m + 1, n) for m in (NX, NY, NZ)], -1)
    # beyond the far x face: dropped.  The first, the last two, a run across
    # the first piece's end and every 977th
    drop = np.r_[0, 1, n - 2, n - 1, 15520:15560, 0:n:977]
    pts[drop, 0] = NX + 1
    cases.write_case(d, spec, media, pts)
    r = _make(d, awpsgt.AWP_STORAGE_FP32)
    r.step(NT)
    r.synchronize()
    keep = np.ones(n, bool)
    keep[drop] = False
    yield r, pts, keep, d
    r.close()


def _raw(sgt, keep):
    """the raw file's bytes by its rules: NT_OUT samples a series, full
    buffers only, zeros for dropped points, cut after the last kept point"""
    nt_out = NT // WS * WS
    out = np.where(keep[:, None, None], sgt[:, :, :nt_out], np.float32(0))
    return out[:np.flatnonzero(keep)[-1] + 1]


def test_sgt_pieces(finished):
    r, pts, keep, _ = finished
    sgt = r.sgt()
    assert sgt.nbytes > 2 * (16 << 20)
    assert np.all(sgt[~keep] == -1.0)      # never sampled
    # points on the same node hold the same series wherever they lie
    node = {}
    for n in np.flatnonzero(keep):
        node.setdefault(tuple(pts[n]), []).append(n)
    twins = [v for v in node.values() if len(v) > 1 and v[-1] - v[0] > 20000]
    assert len(twins) > 50
    for v in twins:
        assert np.array_equal(sgt[v[0]], sgt[v[-1]])
    assert np.any(sgt[keep][:, :, -1] != 0)


def test_files_agree(finished, tmp_path):
    r, _, keep, _ = finished
    want = _raw(r.sgt(), keep)
    raw, rwg, half = (os.path.join(str(tmp_path), f) for f in ("raw", "rwg", "half"))
    r.write_sgt_file(raw)
    assert np.array_equal(np.fromfile(raw, dtype=np.float32), want.reshape(-1))
    for z in (False, True):
        r.write_sgt_file_rwg(rwg, z)
        x = want * np.float32(-2.0) if z else want.copy()
        x = x[:, [1, 0, 2, 3, 5, 4]]
        x[:, 4:] *= np.float32(-1.0)
        got = np.fromfile(rwg, dtype=np.float32).reshape(-1, 6, want.shape[2])
        # the reformatter takes complete records
        assert np.array_equal(got, x[:len(got)]) and len(got) >= len(x) - 1
    r.write_sgt_file_fp16(half)
    whole = awpsgt.read_sgt16(half)
    nt_out = want.shape[2]
    assert whole.shape == (len(keep), 6, nt_out)
    full = np.zeros_like(whole)
    full[:len(want)] = want
    # 11-bit rounding under each series' power of two
    peak = np.abs(full).max(axis=2, keepdims=True)
    assert np.all(np.abs(whole - full) <= peak * 2.0 ** -11)
    for first, count in ((0, len(keep)), (3, 12345), (len(keep) - 1, 1)):
        part = awpsgt.read_sgt16_points(half, first, count, nt_out)
        assert np.array_equal(part, whole[first:first + count])
        y = awpsgt.read_sgt16_points(half, first, count, nt_out, 2)
        x = np.float32(-2.0) * whole[first:first + count][:, [1, 0, 2, 3, 5, 4]]
        x[:, 4:] *= np.float32(-1.0)
        assert np.array_equal(y, x)
