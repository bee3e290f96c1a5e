"""GPU parity of the beta fit (api.cpp:812-831) against the oracle.

beta = logf(max(1e-12, w)) with w from the clamped unconstrained least
squares (nnls_method 1, math.h:683-757) or Lawson-Hanson NNLS (nnls_method 0,
math.h:283-452) on M = exp_scores[:, sel], b = row sums. beta then shifts the
compacted softmax, so C_v and the statistics depend on it too; everything
must match bit for bit. Lawson-Hanson on chunks keeping more than 256 keys
is refused (KV_COMPACT_E_UNSUPPORTED).
"""
from __future__ import annotations

import numpy as np
import pytest

from kvc_data import beta_variant, beta_variant_names, kv_cache, snapkv_queries
from kvc_harness import case_params, kc, load_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    lib = kc.load_product()
    if not lib.dll.kv_compact_hip_available():
        pytest.fail("no usable GPU for the GPU test tier")
    return lib


@pytest.fixture(scope="module")
def orc():
    return load_oracle()


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


@pytest.mark.parametrize("name", beta_variant_names())
def test_beta_variant(gpu, orc, name):
    c, K, V, Q, nq = beta_variant(name)
    T, H, d = c["T"], c["H"], c["d"]
    print(f"[beta] {name} T={T} H={H} d={d} params={c['params']}", flush=True)
    if name == "lh_unchunked_big_t":
        rc, _ = gpu.compact_raw(K, V, Q, T, nq, H, d, d, case_params(gpu, c, T))
        assert rc == kc.E_UNSUPPORTED
        return
    a = gpu.compact(K, V, Q, T, nq, H, d, d, case_params(gpu, c, T))
    b = orc.compact(K, V, Q, T, nq, H, d, d, case_params(orc, c, T))
    assert a.t == b.t
    assert np.array_equal(a.indices, b.indices), "indices"
    ba, bb = bits(a.beta), bits(b.beta)
    if not np.array_equal(ba, bb):
        bad = np.argwhere(ba != bb)
        raise AssertionError(f"beta differs at {len(bad)} of {ba.size}: first {bad[:3].tolist()}")
    assert np.array_equal(bits(a.C_v), bits(b.C_v)), "C_v"
    for k in ("avg_cosine_sim", "avg_mse", "avg_agreement"):
        assert np.float32(a.stats[k]).view(np.uint32) == np.float32(b.stats[k]).view(np.uint32), k


# Lawson-Hanson's register kernels: passive sets up to 64 on one wave (query
# counts up to 62 try it first; 62 queries outgrow it here), larger ones on
# two; the loop's cycles cut short at iteration caps that leave a remainder;
# few variables; repeated keys (ties and singular sub-problems); NaN.
@pytest.mark.parametrize("T,d,nq,ratio,cap,form", [
    (1280, 128, 62, 0.2, 200, "scale"), (512, 64, 62, 0.4, 67, ""), (512, 64, 64, 0.4, 200, ""),
    (400, 64, 64, 0.5, 71, ""), (512, 32, 33, 0.5, 1000, ""), (512, 32, 32, 0.5, 41, ""), (300, 32, 1, 0.5, 200, ""),
    (9, 32, 8, 0.4, 200, ""), (512, 32, 24, 0.5, 200, "repeat"), (512, 32, 64, 0.5, 200, "repeat"),
    (512, 32, 16, 0.5, 5, "nan"), (512, 32, 64, 0.5, 5, "nan")])
def test_lawson_hanson_sets(gpu, orc, T, d, nq, ratio, cap, form):
    print(f"[lh] T={T} d={d} nq={nq} cap={cap} {form}", flush=True)
    K, V = kv_cache(T, 2, d, 47, channel_scale=True)
    if form == "scale":
        K = (K * np.float32(0.7)).astype(np.float32)
    if form == "repeat":
        K[1::2] = K[0::2]
    Q = snapkv_queries(K, nq, 47)
    if form == "nan":
        K[T // 3, 3] = np.nan
    par = dict(target_ratio=ratio, skip_beta=0, nnls_method=0, nnls_max_iter=cap)
    a = gpu.compact(K, V, Q, T, nq, 2, d, d, gpu.params(**par))
    b = orc.compact(K, V, Q, T, nq, 2, d, d, orc.params(**par))
    assert np.array_equal(a.indices, b.indices), "indices"
    for k in ("beta", "C_v"):
        x, y = getattr(a, k), getattr(b, k)
        nan = np.isnan(x) & np.isnan(y)   # (a NaN's payload is not pinned)
        assert np.array_equal(bits(np.where(nan, 0, x)), bits(np.where(nan, 0, y))), k
