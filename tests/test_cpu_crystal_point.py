"""The crystal-frame form of the local Newton (cp_crystal.hpp), compiled for the CPU, against the
general form (cp_point.hpp) over what its dispatch accepts: both slip-system counts, rate
exponents on both sides of 1, scaled rotations, latent hardening with and without blocks, a
plastic history, saturated and over-saturated resistances, an iteration cap; and over what it
leaves to the general form.

The two differ by rounding: the local tolerance 1e-8 on stresses of order 100 lets the
quadratically converging iterates differ by a few 1e-11 of them, and a slip rate by 1/m times
that."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT
from helpers import FCC_304, random_states, slip_table

SRC = os.path.join(ROOT, "tests", "cpu_point", "crystal_check.cpp")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("cc") / "libcrystal_check.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", out, SRC], check=True)
    L = ctypes.CDLL(out)
    L.crystal_check.restype = ctypes.c_int64
    return L


def _inputs(table, N, Q, seed, xm, scale=None):
    from oracle import cp_local
    rng = np.random.default_rng(seed)
    tab = slip_table(table)
    d = tab[:, 3:6] / np.linalg.norm(tab[:, 3:6], axis=1)[:, None]
    n = tab[:, 0:3] / np.linalg.norm(tab[:, 0:3], axis=1)[:, None]
    H, Fp, g, slip, q = random_states(Q, N, rng, table=table)
    R = cp_local.rot_mat_from_quat(q)
    if scale is not None:
        R = R * scale
    mat = np.tile([xm] + [FCC_304[k] for k in ("gss_a", "h", "t_sat", "r", "C11", "C12", "C44")], (Q, 1))
    return [np.ascontiguousarray(x, dtype=float) for x in (H, Fp, g, slip, R, mat, d, n)]


def _run(lib, ins, N, crystal, self_block=1, max_iter=250, dt=0.5):
    Q = len(ins[0])
    o = dict(S=np.zeros((Q, 6)), P=np.zeros((Q, 9)), A=np.zeros((Q, 81)), gn=np.zeros((Q, N)), sn=np.zeros((Q, N)),
             it=np.zeros(Q, np.int32), st=np.zeros(Q, np.int32))
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    used = lib.crystal_check(N, crystal, ctypes.c_int64(Q), *[p(a) for a in ins], ctypes.c_double(1e-3 * dt),
                             ctypes.c_double(1e-8), 5, max_iter, self_block, *[p(a) for a in o.values()])
    return o, used


def _same(c, g, ins, xm):
    scale = np.linalg.norm(g["S"], axis=1).max()
    assert np.abs(c["S"] - g["S"]).max() <= 1e-10 * scale
    assert np.abs(c["P"] - g["P"]).max() <= 1e-10 * scale
    rel = np.linalg.norm(c["A"] - g["A"], axis=1) / np.linalg.norm(g["A"], axis=1)
    assert rel.max() <= 1e-9 * max(1.0, 0.1 / xm)
    inc = np.abs(g["sn"] - ins[3])
    np.testing.assert_allclose(c["sn"], g["sn"], rtol=0, atol=1e-10 / xm * inc.max() + 1e-18)
    np.testing.assert_allclose(c["gn"], g["gn"], rtol=1e-12)
    np.testing.assert_array_equal(c["st"], g["st"])
    assert np.mean(c["it"] == g["it"]) >= 0.98


@pytest.mark.parametrize("table,N,xm,block", [("slip_fcc12.txt", 12, 0.02, 1), ("slip_bcc24.txt", 24, 0.02, 1),
                                              ("slip_bcc12.txt", 12, 0.1, 0), ("slip_fcc12.txt", 12, 0.5, 1),
                                              ("slip_bcc24.txt", 24, 2.0, 0)])
@pytest.mark.parametrize("scale", [None, 0.75, 1.02])
def test_crystal_form_matches_the_general_form(lib, table, N, xm, block, scale):
    ins = _inputs(table, N, 400, 11, xm, scale)
    if xm > 1.0:  # a rate exponent below 1 has no slope at zero stress; keep the increments small
        ins[2][:] *= 1e3
    ins[2][::7] *= 4.0  # resistances beyond t_sat
    ins[2][::11, ::2] = FCC_304["t_sat"]
    c, used = _run(lib, ins, N, 1, block)
    g, _ = _run(lib, ins, N, 0, block)
    assert used == 400
    _same(c, g, ins, xm)


def test_iteration_cap_and_bad_history_set_the_same_status(lib):
    ins = _inputs("slip_fcc12.txt", 12, 200, 5, 0.02)
    ins[2][17, 3] = np.nan
    ins[0][40:44] = 0.0  # unstrained points: sound, a NaN, a zero and an infinite resistance
    ins[1][40:44] = np.eye(3)
    ins[2][41:44, 5] = np.nan, 0.0, np.inf
    for cap in (1, 3, 250):
        c, _ = _run(lib, ins, 12, 1, max_iter=cap)
        g, _ = _run(lib, ins, 12, 0, max_iter=cap)
        np.testing.assert_array_equal(c["st"], g["st"])
        assert (cap == 250) == (np.count_nonzero(c["st"]) == 3)
        np.testing.assert_array_equal(np.isnan(c["P"]), np.isnan(g["P"]))


def test_other_points_keep_the_general_form(lib):
    """m = 1, a sheared R, moduli that are not positive definite and slip directions out of their
    planes: the general form's results bit for bit."""
    for change in ("m", "R", "C", "d"):
        ins = _inputs("slip_fcc12.txt", 12, 50, 8, 1.0 if change == "m" else 0.05)
        if change == "m":
            ins[2][:] *= 1e3
        if change == "R":
            ins[4][:, 0, 1] += 1e-9
        if change == "C":
            ins[5][:, 7] *= -1.0
        if change == "d":
            ins[6][3] += 1e-9
        c, used = _run(lib, ins, 12, 1, max_iter=5)
        g, _ = _run(lib, ins, 12, 0, max_iter=5)
        assert used == 0
        for k in c:
            np.testing.assert_array_equal(c[k], g[k])
