"""GPU parity of the register LU's two variants and of non-finite inputs.

The LU runs unmasked (multiplier 0 for the rows off the elimination) and
sends a system to the masked variant when its input holds -0 or a
non-finite entry, or when a final entry is non-finite. KVC_LU_MASKED=1 sends
every system to the masked variant, so both are checked against the oracle
on the same cases. Non-finite K / V entries reach the LU through the scores
and exercise the fallback itself; NaN results are compared by position (the
GPU and the x86 oracle may produce different NaN bit patterns), every other
value bit for bit.
"""
from __future__ import annotations

import numpy as np
import pytest

from kvc_data import CASE_BY_NAME, beta_variant, kv_cache, make_case, nonfinite_variant, nonfinite_variant_names, snapkv_queries
from kvc_harness import case_params, kc, load_oracle, run_case

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.fixture(scope="module")
def gpu():
    lib = kc.load_product()
    if not lib.dll.kv_compact_hip_available():
        pytest.fail("no usable GPU for the GPU test tier")
    return lib


@pytest.fixture(scope="module")
def orc():
    return load_oracle()


def same_nan(x, y, what):
    x = np.ascontiguousarray(x, np.float32)
    y = np.ascontiguousarray(y, np.float32)
    nx, ny = np.isnan(x), np.isnan(y)
    assert np.array_equal(nx, ny), f"{what}: NaN positions differ"
    assert np.array_equal(bits(x[~nx]), bits(y[~ny])), f"{what}: values differ"


def same(a, b):
    assert a.t == b.t
    assert np.array_equal(a.indices, b.indices), "indices"
    same_nan(a.beta, b.beta, "beta")
    same_nan(a.C_v, b.C_v, "C_v")
    for k in ("avg_cosine_sim", "avg_mse", "avg_agreement"):
        same_nan(np.float32(a.stats[k]), np.float32(b.stats[k]), k)


@pytest.mark.parametrize("name", ["cfg1_small", "cfg2_small_nodiv", "beta_clamped", "refine2_beta", "count",
                                  "tiny_T3", "dv_ne_dk", "prefix"])
def test_masked_variant_parity(gpu, orc, name, monkeypatch):
    monkeypatch.setenv("KVC_LU_MASKED", "1")
    c = CASE_BY_NAME[name]
    print(f"[case] masked {name}", flush=True)
    inp = make_case(c)
    same(run_case(gpu, c, inp), run_case(orc, c, inp))


def test_masked_variant_clamped_ls_chunks(gpu, orc, monkeypatch):
    """Clamped-LS beta (the LU also solves the mass fit) at 256 kept keys per chunk."""
    monkeypatch.setenv("KVC_LU_MASKED", "1")
    c, K, V, Q, nq = beta_variant("pgd_chunk")
    T, H, d = c["T"], c["H"], c["d"]
    print("[case] masked pgd_chunk", flush=True)
    a = gpu.compact(K, V, Q, T, nq, H, d, d, case_params(gpu, c, T))
    b = orc.compact(K, V, Q, T, nq, H, d, d, case_params(orc, c, T))
    same(a, b)


@pytest.mark.parametrize("pgd", [0, 1])
@pytest.mark.parametrize("name", nonfinite_variant_names())
def test_nonfinite_inputs(gpu, orc, name, pgd):
    c, K, V, Q, nq = nonfinite_variant(name)
    T, H, d = c["T"], c["H"], c["d"]
    extra = dict(skip_beta=0, nnls_method=1) if pgd else {}
    print(f"[case] nonfinite {name} pgd={pgd}", flush=True)
    a = gpu.compact(K, V, Q, T, nq, H, d, d, case_params(gpu, c, T, **extra))
    b = orc.compact(K, V, Q, T, nq, H, d, d, case_params(orc, c, T, **extra))
    same(a, b)


# The substitution that spreads a system over eight waves (grids of at most
# one block per CU): unknown counts around its groups of eight rows and blocks
# of four entries, column counts around its 64 lanes.
SUBST_EDGES = [(1, 32), (2, 40), (3, 64), (4, 72), (5, 130), (8, 32), (9, 64), (31, 96), (33, 64), (64, 256), (127, 40),
               (129, 64), (201, 72), (253, 64), (254, 130), (255, 64), (256, 128)]


@pytest.mark.parametrize("n,d", SUBST_EDGES)
def test_substitution_wide_edges(gpu, orc, n, d):
    check_substitution(gpu, orc, n, d)


# The same with the one wave per 64 columns that larger grids take.
@pytest.mark.parametrize("n,d", SUBST_EDGES)
def test_substitution_one_wave_edges(gpu, orc, n, d, monkeypatch):
    monkeypatch.setenv("KVC_SUBST_WIDE", "0")
    check_substitution(gpu, orc, n, d)


def check_substitution(gpu, orc, n, d):
    T = 2 * n
    K, V = kv_cache(T, 2, d, 61, channel_scale=True)
    nq = min(T, 24)
    Q = snapkv_queries(K, nq, 61)
    print(f"[subst] n={n} d={d}", flush=True)
    a = gpu.compact(K, V, Q, T, nq, 2, d, d, gpu.params(target_ratio=0.5, chunk_size=-1))
    b = orc.compact(K, V, Q, T, nq, 2, d, d, orc.params(target_ratio=0.5, chunk_size=-1))
    assert a.t == b.t == n and np.array_equal(a.indices, b.indices)
    assert np.array_equal(a.C_v.view(np.uint32), b.C_v.view(np.uint32)), "C_v"


# Systems with skipped pivots: equal keys make M exactly singular, and the beta
# fit's ridge of 1e-10 is lost beside its entries. One system (all of the
# grid), several chunks, and column counts past one block of 64.
@pytest.mark.parametrize("T,H,d,nq,chunk,ratio", [
    (6, 1, 32, 4, -1, 0.5), (40, 2, 64, 9, -1, 0.5), (130, 1, 130, 40, -1, 0.5), (256, 2, 64, 24, -1, 0.5),
    (400, 1, 128, 64, -1, 0.5), (512, 2, 96, 32, -1, 0.5), (3000, 2, 64, 32, 300, 0.4)])
def test_skipped_pivots(gpu, orc, T, H, d, nq, chunk, ratio):
    K, V = kv_cache(T, H, d, 71)
    K[1::2] = K[0::2][:T // 2]
    Q = snapkv_queries(K, nq, 71)
    print(f"[skip] T={T} H={H} d={d} nq={nq} chunk={chunk}", flush=True)
    par = dict(target_ratio=ratio, chunk_size=chunk, skip_beta=0, nnls_method=1)
    a = gpu.compact(K, V, Q, T, nq, H, d, d, gpu.params(**par))
    b = orc.compact(K, V, Q, T, nq, H, d, d, orc.params(**par))
    assert a.t == b.t and np.array_equal(a.indices, b.indices)
    assert np.array_equal(a.beta.view(np.uint32), b.beta.view(np.uint32)), "beta"
    assert np.array_equal(a.C_v.view(np.uint32), b.C_v.view(np.uint32)), "C_v"


# Skipped pivots in the value refit, many columns a system: without its ridge a
# pair of equal keys gives a pivot that cancels exactly. At most 256 unknowns
# (columns past one block of 64), then the blocked elimination: full panels,
# narrower ones with sizes that are no multiple of four, and the sizes whose
# back substitution does not fit LDS 64 columns at a time; with and without
# skipped pivots, and the beta fit's single column beside them.
@pytest.mark.parametrize("T,H,d,nq,pairs", [
    (6, 1, 130, 4, 1), (130, 1, 130, 40, 1), (512, 2, 96, 32, 1), (514, 1, 40, 40, 1), (700, 2, 40, 64, 1),
    (1042, 1, 130, 400, 1), (1042, 1, 130, 24, 1), (1160, 1, 64, 33, 1), (1202, 1, 72, 64, 1), (1042, 1, 130, 400, 0),
    (1178, 1, 64, 200, 0)])
def test_skipped_pivots_values(gpu, orc, T, H, d, nq, pairs):
    K, V = kv_cache(T, H, d, 71)
    if pairs:
        K[1::2] = K[0::2][:T // 2]
    Q = snapkv_queries(K, nq, 71)
    print(f"[skip] values T={T} H={H} d={d} nq={nq} pairs={pairs}", flush=True)
    for par in (dict(skip_beta=1, ridge=0.0 if pairs else 1e-6), dict(skip_beta=0, nnls_method=1)):
        par.update(target_ratio=0.5, chunk_size=-1)
        a = gpu.compact(K, V, Q, T, nq, H, d, d, gpu.params(**par))
        b = orc.compact(K, V, Q, T, nq, H, d, d, orc.params(**par))
        # a skipped pivot's values are exactly 0
        assert not par["skip_beta"] or (b.C_v == 0).all(-1).any() == bool(pairs)
        assert a.t == b.t == T // 2 and np.array_equal(a.indices, b.indices)
        assert np.array_equal(a.beta.view(np.uint32), b.beta.view(np.uint32)), "beta"
        assert np.array_equal(a.C_v.view(np.uint32), b.C_v.view(np.uint32)), "C_v"
