"""The hand-written reverse product of a point (cp_reverse.hpp) against the forward-mode one
(cp_dual.hpp), one input direction at a time, both compiled for the CPU and run at the same
converged stress: both slip-system counts, rate exponents down to m = 1, latent hardening with and
without blocks, resistances below, at and above saturation, rotations that are scaled or sheared,
points without slip, missing cotangents and masked groups.

Both are exact derivatives of the same map, so they differ by rounding: a few hundred operations on
terms that 1/m (50) and the 6 x 6 system's condition (up to 1e3) amplify, 1e-11 of a group's norm;
the bound is ten times that."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT
from helpers import FCC_304, random_states, slip_table

SRC = os.path.join(ROOT, "tests", "cpu_point", "reverse_check.cpp")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rc") / "libreverse_check.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", out, SRC], check=True)
    return ctypes.CDLL(out)


@pytest.mark.parametrize("table,N", [("slip_fcc12.txt", 12), ("slip_bcc24.txt", 24)])
@pytest.mark.parametrize("xm,gss_a,self_block,mode,mask", [
    (0.02, 2.0, 1, "plain", 31), (0.05, 1.0, 0, "scaled", 31), (0.02, 2.2, 1, "sheared", 31), (1.0, 2.0, 1, "plain", 31),
    (0.02, 2.0, 1, "saturated", 31), (0.02, 1.0, 0, "rest", 31), (0.02, 2.0, 0, "no history cotangents", 31),
    (0.05, 2.0, 1, "plain", 5), (0.05, 2.0, 1, "plain", 26)])
def test_reverse_matches_forward(lib, table, N, xm, gss_a, self_block, mode, mask):
    from oracle import cp_local
    rng = np.random.default_rng(5)
    Q = 24
    H, Fp, g, slip, quat = random_states(Q, N, rng, table=table, cap=1.3)
    R = cp_local.rot_mat_from_quat(quat)
    if mode == "scaled":
        R = 1.01 * R
    if mode == "sheared":
        R = R + 1e-3 * rng.normal(size=R.shape)
    mat = np.tile([xm, gss_a] + [FCC_304[k] for k in ("h", "t_sat", "r", "C11", "C12", "C44")], (Q, 1))
    if mode == "saturated":
        g[: Q // 2, ::2] = mat[0, 3]
        g[Q // 2:, 1::2] = 1.1 * mat[0, 3]
    if mode == "rest":
        H, Fp = np.zeros_like(H), np.broadcast_to(np.eye(3), Fp.shape).copy()
    tab = slip_table(table)
    d = tab[:, 3:6] / np.linalg.norm(tab[:, 3:6], axis=1)[:, None]
    n = tab[:, 0:3] / np.linalg.norm(tab[:, 0:3], axis=1)[:, None]
    cots = [rng.normal(size=(Q, 9)), rng.normal(size=(Q, 9)), 50 * rng.normal(size=(Q, 9)), rng.normal(size=(Q, N)),
            100 * rng.normal(size=(Q, N))]
    keep = [np.ascontiguousarray(x, dtype=float) for x in (H, Fp, g, R, mat, d, n)]
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    tail = [p(c) for c in cots[:3]] + ([None, None] if mode == "no history cotangents" else [p(c) for c in cots[3:]])
    got = []
    for reverse in (0, 1):
        out = np.full((Q, 35 + N), -7.0)
        lib.reverse_check(N, reverse, ctypes.c_int64(Q), *[p(a) for a in keep], ctypes.c_double(1e-3), ctypes.c_double(0.5),
                          self_block, mask, *tail, p(out))
        got.append(out)
    fwd, rev = got
    assert np.isfinite(fwd).all()
    for bit, (a, b) in zip((1, 2, 4, 8, 8, 16), ((0, 9), (9, 18), (18, 18 + N), (18 + N, 23 + N), (23 + N, 26 + N), (26 + N, 35 + N))):
        if not mask & bit:
            assert (rev[:, a:b] == -7.0).all() and (fwd[:, a:b] == -7.0).all()
            continue
        scale = np.linalg.norm(fwd[:, a:b], axis=1, keepdims=True)
        err = np.abs(rev[:, a:b] - fwd[:, a:b]) / (scale + 1e-300)
        assert err.max() <= 1e-10, (mode, bit, a, err.max())
