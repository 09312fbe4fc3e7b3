"""The Cholesky kernels' own source on the host, one fiber per lane
(tests/emulation), the waves in a given order between the workgroup's barriers
and the lanes of a wave in a given order between its cross-lane operations.
An order and its reverse put every pair of waves (lanes) both ways round, so
accesses that no barrier orders show as another result.  Oracle: numpy's
Cholesky; tolerances as in test_gpu_potrf.py."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CLANG = "/opt/rocm/llvm/bin/clang++"
EPS = np.finfo(float).eps
FORWARD = list(range(8))


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("emulation") / "potrf.so")
    src = os.path.join(HERE, "emulation", "potrf.cpp")
    subprocess.run([CLANG, "-std=c++17", "-O1", "-mfma", "-ffp-contract=off", "-w", "-fPIC", "-shared", "-I",
                    os.path.join(HERE, "emulation"), src, "-o", out], check=True)
    lib = ctypes.CDLL(out)

    def factor(A, order=FORWARD, lanes_reversed=False, mode=1, rb4=False):
        n = len(A)
        L, W, cond = np.asfortranarray(A).copy(order="F"), np.zeros((n, n), order="F"), np.zeros(n // 64)
        dp = ctypes.POINTER(ctypes.c_double)
        p = lambda x: x.ctypes.data_as(dp)
        st = lib.emu_factor(p(L), p(W), p(cond), n, mode, (ctypes.c_int * 8)(*order), int(lanes_reversed), int(rb4))
        return np.tril(L), W, cond, st

    return factor


def spd(n):
    X = np.random.default_rng(n).uniform(size=(n, 3))
    return 0.9 * np.exp(-np.sum(np.abs(X[:, None, :] - X[None, :, :]), axis=2) / 0.3) + 0.1 * np.eye(n)


def graded(n):
    """estimates 64 max|L| max|L^-1| past the refinement threshold of 1e4 in every block"""
    D = 10.0 ** (-3.0 * (np.arange(n) % 64) / 63.0)
    return spd(n) * np.outer(D, D)


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a[:3], b[:3])) and a[3] == b[3]


@pytest.mark.parametrize("n,make", [(64, spd), (128, spd), (128, graded), (192, spd)])
def test_order_of_waves_does_not_matter(emu, n, make):
    A = make(n)
    ref = emu(A)
    assert ref[3] == 0
    L, _, cond, _ = ref
    assert np.all((cond > 1e4) == (make is graded))
    scale = np.sqrt(np.outer(np.diag(A), np.diag(A)))
    assert np.max(np.abs(A - L @ L.T) / scale) <= 256 * (n + 1) * EPS
    for order in (FORWARD[::-1], [1, 0, 3, 2, 5, 4, 7, 6], [4, 5, 6, 7, 0, 1, 2, 3]):
        assert same(emu(A, order), ref), order
    assert same(emu(A, FORWARD, rb4=True), ref)


@pytest.mark.parametrize("n,make", [(64, spd), (128, graded), (192, spd)])
def test_order_of_lanes_does_not_matter(emu, n, make):
    A = make(n)
    ref = emu(A)
    assert ref[3] == 0
    assert same(emu(A, lanes_reversed=True), ref)


@pytest.mark.parametrize("exponent", [0, -600, 600])
@pytest.mark.parametrize("make", [spd, graded])
def test_condition_estimate_at_any_scale(emu, make, exponent):
    # 64 max|L_kk| max|L_kk^-1| of what was stored, in 64 bits; a scaling by an
    # even power of two scales the factor exactly, so the same blocks refine
    n = 128
    L0, W0, _, _ = emu(make(n))
    L, W, cond, st = emu(make(n) * 2.0 ** exponent)
    assert st == 0
    assert np.array_equal(L, L0 * 2.0 ** (exponent // 2)) and np.array_equal(W, W0 * 2.0 ** (-exponent // 2))
    for k in range(n // 64):
        b = slice(64 * k, 64 * k + 64)
        assert cond[k] == 64 * np.max(np.abs(L[b, b])) * np.max(np.abs(W[b, b]))


@pytest.mark.parametrize("make", [spd, graded])
def test_rows_of_16_and_of_64(emu, make):
    # two block columns per square and three row blocks below the first
    A = make(320)
    ref = emu(A)
    assert ref[3] == 0
    assert same(emu(A, FORWARD[::-1], lanes_reversed=True, rb4=True), ref)
