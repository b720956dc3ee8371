"""How SGT output reaches the host: through pinned memory where there is any,
through pageable memory where it is refused.  A child process whose
hipHostMalloc goes through a counting stand-in, which can refuse, checks that
every reader and writer gives the same bytes both ways."""
import os
import subprocess
import sys

import numpy as np
import pytest

import awpsgt
import cases
from conftest import REPO

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
static int refuse, calls;
static int (*real)(void **, size_t, unsigned);
int shim_open(const char *lib)
{
    void *h = dlopen(lib, RTLD_LAZY | RTLD_NOLOAD);
    real = h ? (int (*)(void **, size_t, unsigned))dlsym(h, "hipHostMalloc") : NULL;
    return real != NULL;
}
void shim_refuse(int on) { refuse = on; }
int shim_calls(void) { return calls; }
int hipHostMalloc(void **p, size_t n, unsigned flags)
{
    ++calls;
    return refuse || !real ? 2 : real(p, n, flags);   /* 2: hipErrorOutOfMemory */
}
"""

CHILD = r"""
import ctypes, os, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)   # before the library that calls it
for p in (%r, %r, %r, %r):
    sys.path.insert(0, p)
import numpy as np
import awpsgt
from test_gpu_parity import _inputs

awpsgt.lib()
hip = [ln.split()[-1] for ln in open("/proc/self/maps") if "libamdhip64" in ln][0]
assert shim.shim_open(hip.encode())

def make(d):
    p, media, xyz, stf, pts = _inputs(d)
    r = awpsgt.Run(p)
    r.set_media(media)
    r.set_source(xyz, stf)
    r.set_sgt_points(pts)
    r.init()
    r.step(r.p.nt)
    r.synchronize()
    return r

def outputs(r, d):
    out = [r.sgt().tobytes()]
    for name, write in (("raw", r.write_sgt_file), ("rwg", lambda f: r.write_sgt_file_rwg(f, True)),
                        ("half", r.write_sgt_file_fp16)):
        f = os.path.join(d, name)
        write(f)
        out.append(open(f, "rb").read())
    return out
"""


def _child(tmp_path, body, *args):
    src, lib = os.path.join(str(tmp_path), "shim.c"), os.path.join(str(tmp_path), "shim.so")
    open(src, "w").write(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", lib, src, "-ldl"], check=True)
    here = [REPO, os.path.join(REPO, "cybershake-core_amd"), os.path.join(REPO, "tests", "golden"),
            os.path.join(REPO, "tests")]
    r = subprocess.run([sys.executable, "-c", CHILD % tuple(here) + body, lib] + list(args), stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
    return r.stdout


def _case(d, npts):
    spec = cases.RunSpec(nx=48, ny=40, nz=32, dh=200.0, dt=0.01, nt=45, igreen=3, src=(24, 20, 4), nd=8, sigma=0.03,
                         t0=0.12, ntiskp_sgt=1, write_step=20)
    media = awpsgt.inputs.layered_media(48, 40, 32, [700.0, 1500.0, 2500.0])
    rng = np.random.default_rng(6)
    pts = np.stack([rng.integers(1, m + 1, npts) for m in (48, 40, 32)], -1)
    pts[[0, npts // 3, npts - 1], 0] = 49      # dropped
    cases.write_case(d, spec, media, pts)
    return d


def test_pinned_memory_refused(tmp_path):
    """77 MB of output: every call falls back to pageable memory, and a
    later run of the process takes pinned memory again."""
    d = _case(str(tmp_path), 72000)
    _child(tmp_path, r"""
shim.shim_refuse(1)
r = make(sys.argv[2])
a = outputs(r, sys.argv[2])
n = shim.shim_calls()
assert n >= 1
shim.shim_refuse(0)
q = make(sys.argv[2])
b = outputs(q, sys.argv[2])
assert shim.shim_calls() == n + 1      # one buffer, kept for the run's later reads
assert a == b and len(a[0]) == 72000 * 6 * 45 * 4 and any(a[0])
""", d)


def test_threads_share_a_run(tmp_path):
    """Four threads read and write one finished run at the same time, more
    than once: each gets the bytes a thread alone gets."""
    from concurrent.futures import ThreadPoolExecutor
    from test_gpu_batch import _make
    d = _case(str(tmp_path), 36000)
    r = _make(d, awpsgt.AWP_STORAGE_FP32)
    r.step(r.p.nt)
    r.synchronize()

    def job(kind, n):
        f = os.path.join(d, "%s%d" % (kind, n))
        if kind == "sgt":
            return r.sgt().tobytes()
        if kind == "rwg":
            r.write_sgt_file_rwg(f)
        else:
            (r.write_sgt_file if kind == "raw" else r.write_sgt_file_fp16)(f)
        return open(f, "rb").read()

    kinds = ["sgt", "raw", "rwg", "half"]
    want = {k: job(k, 99) for k in kinds}
    q = _make(d, awpsgt.AWP_STORAGE_FP32)      # a run that has made no buffer yet
    q.step(q.p.nt)
    q.synchronize()
    for x in (r, q):
        r = x
        with ThreadPoolExecutor(4) as ex:
            got = list(ex.map(lambda n: (kinds[n % 4], job(kinds[n % 4], n)), range(16)))
        for k, b in got:
            assert b == want[k], k
        x.close()


def test_small_output_makes_no_pinned_buffer(tmp_path):
    """A run whose output is read once, 2 to 26 MB of it, makes no pinned
    buffer (which costs more than it saves there); one that reads 64 MB in
    all makes one, once."""
    small, large = (_case(os.path.join(str(tmp_path), n), k) for n, k in (("small", 2000), ("large", 24000)))
    _child(tmp_path, r"""
r = make(sys.argv[2])
a = outputs(r, sys.argv[2])
assert len(a[0]) == 2000 * 6 * 45 * 4 and shim.shim_calls() == 0
r = make(sys.argv[3])
a = [r.sgt() for k in range(2)]
assert a[0].nbytes == 24000 * 6 * 45 * 4 and shim.shim_calls() == 0
a += [r.sgt() for k in range(3)]
assert shim.shim_calls() == 1
assert all(np.array_equal(a[0], b) for b in a) and np.any(a[0] != 0)
""", small, large)


def test_writers_into_a_pipe(tmp_path):
    """The RWG-order and FP16 writers go from start to end, so a pipe takes
    them: the same bytes as the file."""
    import threading
    from test_gpu_batch import _make
    d = _case(str(tmp_path), 9000)
    r = _make(d, awpsgt.AWP_STORAGE_FP32)
    r.step(r.p.nt)
    r.synchronize()
    for n, write in enumerate((r.write_sgt_file_rwg, lambda f: r.write_sgt_file_rwg(f, True), r.write_sgt_file_fp16)):
        plain, pipe = (os.path.join(d, "%s%d" % (k, n)) for k in ("plain", "pipe"))
        write(plain)
        os.mkfifo(pipe)
        got = []
        t = threading.Thread(target=lambda: got.append(open(pipe, "rb").read()), daemon=True)
        t.start()
        write(pipe)
        t.join(20)
        want = open(plain, "rb").read()
        assert got and got[0] == want and len(want) > 1000000
    r.close()
