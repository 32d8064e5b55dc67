"""Plan creation reports a failing device query instead of quietly doing without the
launches that need its answer, and leaves no error behind for the next launch to report.
Runs without a GPU: the few HIP functions that plan creation calls are taken from a small
stand-in library, loaded ahead of the real one in a process of its own."""

import shutil
import subprocess
import sys

import pytest

STAND_IN = r"""
#include <stdlib.h>
#include <string.h>
static int pending, blocks = 3;
static int fail(const char *what, int code) {
  const char *f = getenv("FAIL_IN");
  if (f && !strcmp(f, what)) return pending = code;
  return 0;
}
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipDeviceGetAttribute(int *v, int a, int d) { *v = 10; return fail("attribute", 101); }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int t, size_t s) {
  *n = blocks++;
  return fail("occupancy", 98);
}
int hipMalloc(void **p, size_t n) { *p = malloc(n); return 0; }
int hipFree(void *p) { free(p); return 0; }
int hipGetSymbolAddress(void **p, const void *s) { *p = 0; return 0; }
int hipGetLastError(void) { int e = pending; pending = 0; return e; }
int pending_error(void) { return pending; }
"""

PROGRAM = r"""
import ctypes, sys
hip = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
from scratch_wadge_amd import _lib
L = _lib.load()
h = ctypes.c_void_p()
rc = L.wadges_plan_create(ctypes.byref(h), 2, 3, 12, 4, 1.4, 1.0)
print("rc", rc, "handle", bool(h.value), "pending", hip.pending_error(), "hip", L.wadges_last_hip_error())
if rc == 0:
    a, b = ctypes.c_int(), ctypes.c_int()
    assert L.wadges_plan_wide_limits(h, ctypes.byref(a), ctypes.byref(b)) == 0
    print("limits", a.value, b.value)
    assert L.wadges_plan_wide_limits(None, ctypes.byref(a), ctypes.byref(b)) == -1
    assert L.wadges_plan_wide_limits(h, None, ctypes.byref(b)) == -1
    assert L.wadges_plan_destroy(h) == 0
"""


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    if not shutil.which("gcc"):
        pytest.skip("gcc not available")
    d = tmp_path_factory.mktemp("hip")
    (d / "hip.c").write_text(STAND_IN)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(d / "standin.so"), str(d / "hip.c")], check=True)
    return str(d / "standin.so")


def create(stand_in, fail_in):
    import os
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, "-c", PROGRAM, stand_in], capture_output=True, text=True, cwd=root,
                         env={**os.environ, "FAIL_IN": fail_in}, timeout=120)
    assert res.returncode == 0, res.stderr[-2000:]
    return res.stdout.split("\n")


def test_limits_follow_the_occupancy(stand_in):
    out = create(stand_in, "nothing")
    # 10 CUs, 3 blocks of one element and 4 of two
    assert out[0] == "rc 0 handle True pending 0 hip 0" and out[1] == "limits 20 80"


@pytest.mark.parametrize("query,code", [("attribute", 101), ("occupancy", 98)])
def test_failing_query_is_reported(stand_in, query, code):
    assert create(stand_in, query)[0] == f"rc -3 handle False pending 0 hip {code}"
