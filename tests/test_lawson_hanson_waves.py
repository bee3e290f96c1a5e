"""k_nnls_lh lane by lane on the CPU (tests/waves): what passes between the
two waves of a block is ordered by block barriers whichever wave runs first,
and no LDS access is misaligned or out of range. Every case's weights equal
the oracle's bit for bit."""
from __future__ import annotations

import ctypes
import re
import shutil
import struct
import subprocess
from pathlib import Path

import numpy as np
import pytest

from kvc_data import normal, uniform
from kvc_harness import load_oracle

HERE = Path(__file__).resolve().parent
KERNELS = HERE.parent / "kv-compact_amd" / "csrc" / "kvc_kernels.hip"


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("waves")
    m = re.search(r"^constexpr int LH_PMAX.*?(?=^// Right-hand side entry)", KERNELS.read_text(), re.S | re.M)
    assert m, "k_nnls_lh not found"
    # (the one register constraint by the host's name)
    (d / "lawson_hanson.inc").write_text(m.group(0).replace('"+v"(me)', '"+r"(me)'))
    exe = d / "lawson_hanson"
    b = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-w", "-ffp-contract=off", "-fsanitize=undefined",
                        "-fno-sanitize-recover=undefined", f"-I{d}", str(HERE / "waves" / "lawson_hanson.cpp"),
                        "-o", str(exe)], capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-3000:]
    return exe


def weights(model, waves, first, M, b, cap):
    """The kernel's weights, clamped as k_beta_log does, and its redo flag."""
    n = M.shape[1]
    ata, atb = np.zeros((n, n), np.float32), np.zeros(n, np.float32)
    with np.errstate(over="ignore"):
        for q in range(M.shape[0]):   # sums in row order, as k_ls_build's
            ata = ata + M[q][:, None] * M[q][None, :]
            atb = atb + M[q] * b[q]
    r = subprocess.run([str(model)], input=struct.pack("<4i", waves, first, n, cap) + ata.tobytes() + atb.tobytes(),
                       capture_output=True, timeout=300)
    assert r.returncode == 0, r.stderr.decode()[-3000:]
    assert len(r.stdout) == 4 * n + 8
    status, redo = struct.unpack("<2i", r.stdout[4 * n:])
    assert status == 0
    return np.maximum(np.frombuffer(r.stdout[:4 * n], np.float32), np.float32(1e-12)), redo


def oracle(M, b, cap):
    w = np.zeros(M.shape[1], np.float32)
    f = load_oracle().dll.orc_nnls_lh
    f.argtypes, f.restype = [ctypes.c_void_p] * 3 + [ctypes.c_int] * 3, None
    f(M.ctypes.data, b.ctypes.data, w.ctypes.data, M.shape[0], M.shape[1], cap)
    return w


def system(m, n, seed, form=""):
    M = np.exp(normal(seed, (m, n))).astype(np.float32)
    if form == "apart":    # nearly orthogonal columns: every variable enters and stays
        M = (M * 0.02 + 3.0 * np.eye(m, n)).astype(np.float32)
    if form == "repeat":   # ties, and sub-problems that are singular but for the 1e-10
        M[:, 1::2] = M[:, 0::2][:, :n // 2]
    if form == "huge":     # a column whose own weight comes out 0: the set empties at once
        M[:, n // 2] = np.float32(1e20)
    b = (M.sum(1) * ((1.5 if form == "apart" else 0.5) + uniform(seed + 1, m))).astype(np.float32)
    if form == "huge":
        b = np.ones(m, np.float32)
    return np.ascontiguousarray(M), b


# Passive sets of odd and even size (the step's parity picks the offer), one
# variable, sets past 64 (both waves have rows), caps that end a loop early.
CASES = [(6, 1, 3, 200, ""), (4, 3, 5, 200, ""), (9, 7, 11, 200, ""), (16, 13, 13, 60, ""), (12, 24, 17, 40, ""),
         (8, 12, 19, 40, "repeat"), (3, 5, 23, 7, "huge"), (72, 71, 31, 200, "apart")]


@pytest.mark.parametrize("first", [0, 1])
@pytest.mark.parametrize("m,n,seed,cap,form", CASES)
def test_two_waves_in_either_order(model, m, n, seed, cap, form, first):
    M, b = system(m, n, seed, form)
    w, _ = weights(model, 2, first, M, b, cap)
    assert np.array_equal(w.view(np.uint32), oracle(M, b, cap).view(np.uint32))


@pytest.mark.parametrize("m,n,seed,cap,form", CASES)
def test_one_wave(model, m, n, seed, cap, form):
    M, b = system(m, n, seed, form)
    w, redo = weights(model, 1, 0, M, b, cap)
    assert redo == (form == "apart")   # (a set past 64 is left to the two waves)
    if not redo:
        assert np.array_equal(w.view(np.uint32), oracle(M, b, cap).view(np.uint32))
