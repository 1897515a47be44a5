"""The engine's pinned readback buffer: where the HIP runtime cannot give it, and
where it grows while a server's launch runs.  A process of its own loads a shim
ahead of the library whose hipHostMalloc can be told to ask for more than there
is, so that the call fails in the runtime, and which counts the frees of pinned
memory between a graph launch and the wait for its stream."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
static void* runtime(const char* name) {
    return dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD), name);
}
int allocs = 0, last_flags = 0;
int fail_allocs = 0;  /* allocations still to fail */
int hipHostMalloc(void** p, size_t n, unsigned flags) {
    int (*real)(void**, size_t, unsigned) = (int (*)(void**, size_t, unsigned))runtime("hipHostMalloc");
    allocs++;
    last_flags = flags;
    return real(p, fail_allocs > 0 && fail_allocs-- ? (size_t)1 << 60 : n, flags);
}
static void* volatile launched = 0;  /* the stream of a graph launch not waited for yet */
int frees = 0, frees_in_launch = 0;
int hipGraphLaunch(void* graph, void* stream) {
    launched = stream;
    return ((int (*)(void*, void*))runtime("hipGraphLaunch"))(graph, stream);
}
int hipStreamSynchronize(void* stream) {
    int rc = ((int (*)(void*))runtime("hipStreamSynchronize"))(stream);
    if (stream == launched) launched = 0;
    return rc;
}
int hipHostFree(void* p) {
    frees++;
    if (launched) frees_in_launch++;
    return ((int (*)(void*))runtime("hipHostFree"))(p);
}
"""

HEAD = r"""
import ctypes as C, sys
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
C.CDLL("libamdhip64.so.7", mode=C.RTLD_GLOBAL)
import numpy as np
import fastmd_amd as fmd
from conftest import KG_LJ, pos4_of
def desc(n, seed=1):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = g * 1.1 + rng.uniform(0.0, 0.1, (n, 3))
    return fmd.Desc(pos4_of(x), max(1.1 * m + 0.2, 9.0), KG_LJ, vel=rng.standard_normal((n, 3)), seed=seed)
def var(name):
    return C.c_int.in_dll(shim, name)
"""


def _run(tmp_path, script):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", str(so), str(src), "-ldl"], check=True)
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([ROOT, os.path.join(ROOT, "tests")]))
    env["LD_LIBRARY_PATH"] = os.pathsep.join(filter(None, ["/opt/rocm/lib", env.get("LD_LIBRARY_PATH")]))
    r = subprocess.run([sys.executable, "-c", HEAD + script, str(so)], env=env, timeout=100,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    print(r.stdout, flush=True)
    assert r.returncode == 0 and "\nok" in "\n" + r.stdout


def test_a_refused_buffer_is_the_readback_s_error_only(tmp_path):
    _run(tmp_path, r"""
e = fmd.Engine(0)
var("fail_allocs").value = 1
s = e.add(desc(300))          # the buffer is refused here, which nothing needs yet
assert var("fail_allocs").value == 0
e.step(s, 5)
assert e.steps_done(s) == 5
var("fail_allocs").value = 1
try:
    e.state(s)
    raise SystemExit("the readback did not report it")
except fmd.FmdError as x:
    assert x.code == fmd.api.ERR_NOMEM, x
e.step(s, 5)
p, v, im = e.state(s)         # there is memory again
assert np.isfinite(p).all() and e.steps_done(s) == 10
e.close()
print("ok")
""")


def test_the_buffer_is_of_every_device(tmp_path):
    """A thread that reads an engine may have another device current (the flag is
    hipHostMallocPortable)."""
    _run(tmp_path, r"""
e = fmd.Engine(0)
s = e.add(desc(300))
e.state(s)
assert var("allocs").value == 1 and var("last_flags").value & 1
e.close()
print("ok")
""")


def test_growth_beside_a_launch_frees_nothing_until_it_ends(tmp_path):
    _run(tmp_path, r"""
import time
s = fmd.Server(0)
a = s.submit(desc(300), 60000)
while s.stats()["graph_launches"] < 20:
    time.sleep(0.002)
before = var("allocs").value
jobs = [s.submit(desc(n, n), 40) for n in (9000, 20000, 60000)]
while any(s.poll(j) not in (2, 3) for j in jobs):
    time.sleep(0.002)
running = s.poll(a) == 1
s.drain()
for j, n in zip([a] + jobs, (300, 9000, 20000, 60000)):
    r = s.result(j, state=True)
    assert r["status"] == 0 and np.isfinite(r["pos4"]).all() and len(r["pos4"]) == n
print("grown", var("allocs").value - before, "freed", var("frees").value, "beside a launch", var("frees_in_launch").value)
assert running and var("allocs").value > before and var("frees").value > 0
assert var("frees_in_launch").value == 0
s.close()
print("ok")
""")
