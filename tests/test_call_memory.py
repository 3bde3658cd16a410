"""What calls leave in a context's memory cache: a second process whose device memory is counted and limited (a
host library loaded ahead of the framework's takes hipMalloc, hipFree and hipMemGetInfo and passes them on)."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
size_t live, limit = (size_t)1 << 40, left = (size_t)64 << 30;
static struct { void *p; size_t n; } blocks[4096];
static void *hip(const char *name) {
  void *h = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
  return h ? dlsym(h, name) : 0;
}
int hipMalloc(void **p, size_t n) {
  if (live + n > limit) return 2;
  int e = ((int (*)(void **, size_t))hip("hipMalloc"))(p, n);
  for (int i = 0; !e && i < 4096; ++i)
    if (!blocks[i].p) {
      blocks[i].p = *p;
      blocks[i].n = n;
      live += n;
      break;
    }
  return e;
}
int hipFree(void *p) {
  for (int i = 0; p && i < 4096; ++i)
    if (blocks[i].p == p) {
      live -= blocks[i].n;
      blocks[i].p = 0;
      break;
    }
  return ((int (*)(void *))hip("hipFree"))(p);
}
int hipMemGetInfo(size_t *f, size_t *t) {
  *f = left;
  *t = (size_t)288 << 30;
  return 0;
}
"""
CHILD = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path[:0] = [sys.argv[2], sys.argv[3]]
import numpy as np
from andromeda_amd import api
from test_lsqr_shapes import _system
cell = lambda name: ctypes.c_size_t.in_dll(shim, name)
live, MB = lambda: cell("live").value, 1 << 20
def solve(ctx, n):
    A, b = _system(n, n, 1)
    X, _ = ctx.lsqr_dense(A, b, eps=1e-12)
    assert np.linalg.norm(A @ X - b) < 1e-9 * np.linalg.norm(b)
def csr(n, fill):
    A = _system(n, n, 1)[0]
    A[:, : n - fill] *= np.eye(n)[:, : n - fill]
    i, j = np.nonzero(A)
    ia = np.concatenate([[1], 1 + np.cumsum(np.bincount(i, minlength=n))]).astype(np.int64)
    a, b, x = A[i, j], A @ np.ones(n), np.zeros(n)
    ja = (j + 1).astype(np.int32)
    q = api.lsqr_precon(n, n, ia, ja, a)
    r = api.lsqr_solve(n, n, ia, ja, a, q, b, x, eps=1e-12)
    assert r["ierr"] == 0 and np.abs(x - 1.0).max() < 1e-8
"""


def run(tmp_path, body):
    src, lib = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src), "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-c", CHILD + body, str(lib), os.path.dirname(HERE), HERE],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-500:] + r.stderr[-2000:]


@pytest.mark.gpu
def test_gpu_cache_leaves_room(tmp_path):
    """With little device memory free a new allocation empties the cache."""
    run(tmp_path, """
grown = []
for left in (64 << 30, 1 << 30):
    cell("left").value = left
    with api.Context(0) as ctx:
        n0 = live()
        solve(ctx, 1000)
        solve(ctx, 2000)
        grown.append(live() - n0)
assert grown[1] < grown[0] - 7 * MB, grown
""")


@pytest.mark.gpu
def test_gpu_large_dense_matrix_goes_back(tmp_path):
    """A matrix of 200 MB: the driver has it again when the call returns, and the small ones stay."""
    run(tmp_path, """
with api.Context(0) as ctx:
    solve(ctx, 300)
    n0 = live()
    solve(ctx, 300)
    assert live() == n0
    solve(ctx, 5000)
    assert live() - n0 < 40 * MB, live() - n0
""")


@pytest.mark.gpu
def test_gpu_csr_behind_a_larger_one(tmp_path):
    """36.9 MB of device memory: a CSR whose dense copy, 24 MB, and staging fit them alone, behind another
    whose staging and workspaces, 14 MB, the cache holds."""
    run(tmp_path, """
cell("limit").value = 36900000
csr(1000, 1000)
csr(1700, 570)
n0 = live()
api.lsqr_forget()
assert n0 - live() >= 8 * 1700 * 1712
""")
