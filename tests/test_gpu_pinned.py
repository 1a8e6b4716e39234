"""When the simulator's pinned buffers for large reads are allocated, and reads without them.
A library loaded before the simulator's stands in for hipHostMalloc: it counts the large
allocations, and refuses them when told to."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#include <cstddef>
#include <dlfcn.h>
extern "C" {
int large = 0, refuse = 0;
int hipHostMalloc(void** p, size_t n, unsigned f) {
    if (n >= (1u << 20)) {
        ++large;
        if (refuse) return 2;       // hipErrorOutOfMemory
    }
    void* h = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
    if (!h) h = dlopen("libamdhip64.so", RTLD_LAZY | RTLD_NOLOAD);
    auto real = h ? (int (*)(void**, size_t, unsigned))dlsym(h, "hipHostMalloc") : nullptr;
    return real ? real(p, n, f) : 1;
}
}
"""

CHILD = r"""
import ctypes, sys
sys.path.insert(0, sys.argv[2])
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
large, refuse = ctypes.c_int.in_dll(shim, "large"), ctypes.c_int.in_dll(shim, "refuse")
import numpy as np
from mgbrain_amd import native as N
from mgbrain_amd import workloads as W
def sim(m):
    n = 3000
    rng = np.random.default_rng(4)
    src, tar = rng.integers(0, n, m, dtype=np.int32), rng.integers(0, n, m, dtype=np.int32)
    w = rng.random(m, dtype=np.float32)
    s = N.Simulator.from_arrays([N.LIF] * n, [0.0] * n, W.lifb_consts(), src, tar, w, np.full(m, np.float32(1e-3)),
                                weight_format=N.WF_F32)
    return s, w[np.argsort(src, kind="stable")]
refuse.value = int(sys.argv[3])
s, want = sim((1 << 22) + 1)                     # 16 MiB a read
before = large.value
at = []
for _ in range(6):
    assert np.array_equal(s.weights(), want)
    at.append(large.value - before)
s.close()
t, want = sim(1 << 24)                           # 64 MiB
before = large.value
assert np.array_equal(t.weights(), want)
t.close()
print(at, large.value - before)
"""


@pytest.mark.parametrize("refuse,want", [(0, "[0, 0, 0, 2, 2, 2] 2"), (1, "[0, 0, 0, 1, 1, 1] 1")])
def test_large_reads(tmp_path, refuse, want):
    """The buffers come when the reads reach 64 MiB together; refused, reads go on without."""
    print(f"case: reads of 16 and 64 MiB, pinned memory refused={refuse}", flush=True)
    src, so = tmp_path / "shim.cpp", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-shared", "-fPIC", "-o", str(so), str(src), "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-c", CHILD, str(so), ROOT, str(refuse)], stdout=subprocess.PIPE,
                       stderr=subprocess.PIPE, text=True, timeout=90)
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip() == want
