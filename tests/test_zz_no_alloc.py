"""qed_lanczos_gs_noalloc, the Lanczos ground state that allocates no device memory (its
vectors and partial sums live in a fixed device array of the library), against
qed_lanczos_gs on the same sectors and start vectors: three calls in a row on sectors of
decreasing size (the array keeps the previous call's contents), one of them on the fused
Lanczos product; the error for a sector beyond the array's limit; and the runtime's allocating
calls, counted."""
import os
import subprocess
import sys

import numpy as np
import pytest

from tests import models as TM

pytestmark = pytest.mark.gpu

LIMIT = 1 << 21


def _run(entry, S, x0, max_iter=400):
    from pyqcm_amd import _lib
    from pyqcm_amd._lib import DeviceArray
    psi = DeviceArray.from_host(x0)
    E0 = np.zeros(1)
    nit = np.zeros(1, np.int32)
    a = np.zeros(max_iter + 2)
    b = np.zeros(max_iter + 2)
    _lib.call(entry, S.h, 1e-12, max_iter, psi.ptr, _lib.dp(E0), _lib.ip(nit), _lib.dp(a), _lib.dp(b))
    n = int(nit[0])
    out = (float(E0[0]), n, a[:n].copy(), b[:n].copy(), psi.to_host())
    psi.free()
    return out


def test_noalloc_lanczos_matches_lanczos_gs(gpu_lib):
    from pyqcm_amd.sector import Sector
    cases = [
        # 3x4 Hubbard, N=12 Sz=0: D = 924^2 = 853,776 (rows shorter than 4096: ELL kernel)
        (TM.square(3, 4, tp=-0.3, U=8.0, mu=4.0), 6, 6),
        # 4x4 Hubbard, 8 up + 1 down: D = 12870 * 16 = 205,920 (fused Lanczos product)
        (TM.square(4, 4, tp=-0.3, U=8.0, mu=4.0), 8, 1),
        # 3x3 Hubbard, 5 up + 4 down: D = 126^2 = 15,876
        (TM.square(3, 3, tp=-0.3, U=8.0, mu=4.0), 5, 4),
    ]
    rng = np.random.default_rng(41)
    for (m, vals), nup, ndn in cases:
        S = Sector(m.L, nup, ndn, m.flat(vals))
        assert S.dim <= LIMIT
        x0 = rng.standard_normal(S.dim)
        x0 /= np.linalg.norm(x0)
        ref = _run("qed_lanczos_gs", S, x0)
        got = _run("qed_lanczos_gs_noalloc", S, x0)
        print("L=%d (%d, %d) D=%d: E0 %.14f / %.14f, iterations %d / %d, max|dpsi| %.1e"
              % (m.L, nup, ndn, S.dim, ref[0], got[0], ref[1], got[1], np.abs(ref[4] - got[4]).max()),
              flush=True)
        assert got[1] == ref[1]
        assert abs(got[0] - ref[0]) <= 1e-12 * abs(ref[0])
        np.testing.assert_allclose(got[2], ref[2], rtol=1e-12, atol=1e-12)
        np.testing.assert_allclose(got[3], ref[3], rtol=1e-12, atol=1e-12)
        assert np.abs(got[4] - ref[4]).max() <= 1e-10
        S.close()


def test_noalloc_lanczos_rejects_large_sector(gpu_lib):
    from pyqcm_amd import _lib
    from pyqcm_amd._lib import DeviceArray
    from pyqcm_amd.sector import Sector
    m, vals = TM.square(4, 4, tp=-0.3, U=8.0, mu=4.0)
    S = Sector(m.L, 7, 6, m.flat(vals))  # D = 11440 * 8008 > 2^21
    assert S.dim > LIMIT
    psi = DeviceArray(8).zeros()  # never touched: the size check comes first
    E0 = np.zeros(1)
    nit = np.zeros(1, np.int32)
    with pytest.raises(RuntimeError, match="exceeds the scratch limit of 2097152"):
        _lib.call("qed_lanczos_gs_noalloc", S.h, 1e-12, 10, psi.ptr, _lib.dp(E0), _lib.ip(nit), None, None)
    psi.free()
    S.close()


COUNTER = r"""
#include <dlfcn.h>
#include <cstddef>
#include <cstdio>
#include <cstdlib>
static int count = 0;
static void* real(const char* name) {
  static void* lib = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_LOCAL);
  void* f = lib ? dlsym(lib, name) : nullptr;
  if (!f) { fprintf(stderr, "no %s\n", name); exit(3); }
  return f;
}
#define COUNT(name, params, args) \
  extern "C" int name params { ++count; return ((int(*) params)real(#name)) args; }
COUNT(hipMalloc, (void** p, size_t n), (p, n))
COUNT(hipMallocAsync, (void** p, size_t n, void* s), (p, n, s))
COUNT(hipHostMalloc, (void** p, size_t n, unsigned f), (p, n, f))
COUNT(hipFree, (void* p), (p))
COUNT(hipHostFree, (void* p), (p))
COUNT(hipEventCreate, (void** e), (e))
COUNT(hipEventCreateWithFlags, (void** e, unsigned f), (e, f))
COUNT(hipEventDestroy, (void* e), (e))
COUNT(hipStreamCreateWithFlags, (void** s, unsigned f), (s, f))
extern "C" int counted() { return count; }
"""

CALLS = r"""
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
import numpy as np
from pyqcm_amd import _lib
from tests import models as TM
from tests.test_zz_no_alloc import _run
from pyqcm_amd.sector import Sector
from pyqcm_amd._lib import DeviceArray
_lib.call("qed_init", 0)
made = 0
for (m, vals), nup, ndn in [(TM.square(2, 3, U=4.0, mu=2.0), 3, 3), (TM.square(4, 4, tp=-0.3, U=8.0, mu=4.0), 8, 1)]:
    S = Sector(m.L, nup, ndn, m.flat(vals))
    x0 = np.random.default_rng(1).standard_normal(S.dim)
    psi = DeviceArray.from_host(x0 / np.linalg.norm(x0))
    E0, nit = np.zeros(1), np.zeros(1, np.int32)
    before = stub.counted()
    _lib.call("qed_lanczos_gs_noalloc", S.h, 1e-12, 400, psi.ptr, _lib.dp(E0), _lib.ip(nit), None, None)
    made += stub.counted() - before
print("outside", before, "inside", made, flush=True)
"""


def test_noalloc_lanczos_makes_no_runtime_objects(gpu_lib, tmp_path):
    """In a process of its own the runtime's allocating calls are counted (their names are
    resolved to a counting library first): none from the first call on, where pinned memory or
    events made on demand would show."""
    src, so = tmp_path / "count.cpp", tmp_path / "libcount.so"
    src.write_text(COUNTER)
    subprocess.check_call(["g++", "-O1", "-shared", "-fPIC", str(src), "-o", str(so), "-ldl"])
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", CALLS, str(so)], cwd=root, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, (r.stdout, r.stderr)
    _, outside, _, inside = r.stdout.split()[-4:]
    assert int(outside) > 0 and int(inside) == 0, r.stdout
