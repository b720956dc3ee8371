"""Decoding the compact FP16 SGT file: every FP16 value, in every output
layout, is its FP32 value times the series' scale, also for a caller whose
floating-point mode flushes subnormal numbers to zero (a program linked with
-ffast-math, torch.set_flush_denormal(True))."""
import os
import struct

import numpy as np
import pytest
import torch

import awpsgt

SCALE = (1.0, 0.5, 2.0 ** 20, 2.0 ** -60, 1.0, 4.0)
RWG = (1, 0, 2, 3, 5, 4)     # input component of each RWG output component


@pytest.fixture(scope="module")
def every_code(tmp_path_factory):
    """An FP16 file of 8 points x 6 components, each series all 65536 codes
    in another order (3 MB: the reader takes more than one thread)."""
    path = os.path.join(str(tmp_path_factory.mktemp("sgt16")), "half")
    codes = np.stack([np.roll(np.arange(65536, dtype=np.uint16), 1021 * s) for s in range(48)])
    hdr = struct.pack("<8s5IfI", b"AWPSGT16", 1, 8, 6, 65536, 1, 0.01, 65536)
    with open(path, "wb") as f:
        f.write(hdr.ljust(64, b"\0"))
        np.tile(np.array(SCALE, np.float32), 8).tofile(f)
        codes.tofile(f)
    # every value here and its product with a scale is a normal FP32 or zero,
    # an infinity or a NaN: exact in FP32
    with np.errstate(invalid="ignore"):
        val = codes.view(np.float16).astype(np.float32).reshape(8, 6, 65536) * np.array(SCALE, np.float32)[:, None]
    return path, val


@pytest.mark.parametrize("flush", [False, True])
def test_every_half(every_code, flush):
    path, val = every_code
    rwg = val[:, RWG].copy()
    rwg[:, 4:] *= np.float32(-1.0)
    want = [val, val[2:7], rwg[2:7], np.float32(-2.0) * rwg[2:7]]
    if flush and not torch.set_flush_denormal(True):
        pytest.skip("this CPU has no flush mode")
    try:
        got = [awpsgt.read_sgt16(path)] + [awpsgt.read_sgt16_points(path, 2, 5, 65536, n) for n in range(3)]
    finally:
        torch.set_flush_denormal(False)
    for w, g in zip(want, got):
        assert np.array_equal(np.isnan(w), np.isnan(g))
        ok = ~np.isnan(w)
        assert np.array_equal(w[ok].view(np.uint32), g[ok].view(np.uint32))   # signs of zeros too
