"""What the Krylov solves allocate when device memory is short, with a HIP runtime that only keeps books
(tests/fake_hip): buffers a solve cannot do without come before the optional ones of the multigrid
preconditioner, and a call that failed leaves nothing half done behind."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

SRC = os.path.join(ROOT, "tests", "fake_hip", "fake_hip.cpp")
LIB = os.path.join(ROOT, "jax-cpfem_amd", "cpfem_amd", "libcpfem_hip.so")

# Runs in a process of its own: the library's HIP symbols have to bind to the stand-in.
CHILD = r'''
import ctypes, importlib.util, os, sys
import numpy as np
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_used.restype = ctypes.c_size_t
fake.fake_limit.argtypes = [ctypes.c_size_t]
fake.fake_mallocs.restype = ctypes.c_int64
spec = importlib.util.spec_from_file_location("native", sys.argv[2])
N = importlib.util.module_from_spec(spec)
spec.loader.exec_module(N)
L = N.load_library()

n = 10
ax = np.arange(n + 1.0)
Z, Y, X = np.meshgrid(ax, ax, ax, indexing="ij")
points = np.ascontiguousarray(np.stack([X.ravel(), Y.ravel(), Z.ravel()], axis=1))
k, j, i = (v.ravel() for v in np.meshgrid(*[np.arange(n)] * 3, indexing="ij"))
node = lambda a, b, c: a + (n + 1) * (b + (n + 1) * c)
cells = np.ascontiguousarray(np.stack([node(i + a, j + b, k + c) for a, b, c in
    ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))], axis=1).astype(np.int32))
dirs = np.ascontiguousarray(np.tile(np.array([1.0, -1.0, 0.0]) / 2 ** 0.5, (12, 1)))
nrms = np.ascontiguousarray(np.tile(np.array([1.0, 1.0, 1.0]) / 3 ** 0.5, (12, 1)))
v = np.zeros(3 * len(points))
mat = np.zeros(81 * len(v))

def create():
    ctx = ctypes.c_void_p()
    mesh = N.CpfemMesh(len(points), len(cells), points.ctypes.data, cells.ctypes.data)
    slip = N.CpfemSlip(12, dirs.ctypes.data, nrms.ctypes.data)
    assert L.cpfem_create(ctypes.byref(mesh), ctypes.byref(slip), ctypes.byref(ctx)) == 0, L.cpfem_last_error()
    return ctx

def solve(ctx, multigrid, precision=0):
    info = N.CpfemSolveInfo()
    args = (ctx, None, mat.ctypes.data, v.ctypes.data, v.ctypes.data, 1e-10, 1e-10, 1)
    if multigrid:
        return L.cpfem_solve_mg(*args, precision, ctypes.byref(info))
    return L.cpfem_solve(*args, 1, precision, ctypes.byref(info))

def sizes(precision):
    """Bytes of the Krylov vectors and of the multigrid buffers."""
    ctx = create()
    a = fake.fake_used()
    assert solve(ctx, False, precision) == 0
    b = fake.fake_used()
    solve(ctx, True, precision)  # kernels that do nothing report no progress: only its memory matters
    c = fake.fake_used()
    L.cpfem_destroy(ctx)
    assert 0 < b - a < c - b
    return b - a, c - b
'''

ORDER = CHILD + r'''
for precision in (0, 1):
    krylov, multigrid = sizes(precision)
    ctx = create()
    base = fake.fake_used()
    fake.fake_limit(base + multigrid + 1024)  # room for either, not for both
    rc = solve(ctx, True, precision)
    assert rc == 0, (precision, rc, L.cpfem_last_error())
    assert fake.fake_used() == base + krylov, (fake.fake_used() - base, krylov, multigrid)
    fake.fake_limit(2 ** 62)
    L.cpfem_destroy(ctx)
print("done")
'''

RETRY = CHILD + r'''
krylov, _ = sizes(0)
for part in (0.02, 0.3, 0.7, 0.95):
    ctx = create()
    base = fake.fake_used()
    fake.fake_limit(base + int(part * krylov))
    assert solve(ctx, False) == N.EHIP, L.cpfem_last_error()
    fake.fake_limit(2 ** 62)
    assert solve(ctx, False) == 0
    assert fake.fake_used() == base + krylov, (part, fake.fake_used() - base, krylov)
    count = fake.fake_mallocs()
    assert solve(ctx, False) == 0 and fake.fake_mallocs() == count
    L.cpfem_destroy(ctx)
    assert fake.fake_used() == 0
print("done")
'''


DIRECT = CHILD + r'''
def direct(ctx):
    info = N.CpfemSolveInfo()
    return L.cpfem_solve_direct(ctx, None, mat.ctypes.data, v.ctypes.data, v.ctypes.data, 0, ctypes.byref(info))

ctx = create()
base = fake.fake_used()
assert direct(ctx) == 0, L.cpfem_last_error()
whole = fake.fake_used() - base
L.cpfem_destroy(ctx)
for part in (0.01, 0.5, 0.9, 0.999):
    ctx = create()
    fake.fake_limit(base + int(part * whole))
    assert direct(ctx) == N.EHIP
    fake.fake_limit(2 ** 62)
    assert direct(ctx) == 0, L.cpfem_last_error()
    assert fake.fake_used() == base + whole, (part, fake.fake_used() - base, whole)
    L.cpfem_destroy(ctx)
    assert fake.fake_used() == 0
print("done")
'''


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    if not os.path.exists(LIB):
        pytest.skip("libcpfem_hip.so not built")
    out = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-o", out, SRC], check=True)
    return out


def _run(script, fake):
    native = os.path.join(ROOT, "jax-cpfem_amd", "cpfem_amd", "_native.py")
    r = subprocess.run([sys.executable, "-c", script, fake, native], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("done"), r.stdout + r.stderr


def test_krylov_vectors_come_before_multigrid_buffers(fake):
    _run(ORDER, fake)

def test_a_failed_allocation_is_made_up_for_by_the_next_call(fake):
    _run(RETRY, fake)


def test_a_failed_direct_solve_is_made_up_for_by_the_next_call(fake):
    _run(DIRECT, fake)
