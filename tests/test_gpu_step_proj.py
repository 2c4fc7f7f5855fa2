"""The one-token step's split fp16 projection (stepproj.hip) against float64, through the LM head
of a model without layers over up to 64 rows: logits = RMSNorm(E[ids]) E^T, every operand known.

Bound per element as for the prefill's product (test_gpu_split_gemm.py): 3 ceil(K / 32) roundings
of a running sum of at most S = sum_k |x_k e_k|, 2^-20 S for the operands, the part left out and
the RMSNorm; the eight waves' partial sums add 8 more roundings.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from test_gpu_split_gemm import device, logits_of, reference, wide_rows  # noqa: E402,F401

pytestmark = pytest.mark.gpu


def bounded(E, ids):
    ref, bound = reference(E, ids)
    x = E[ids].astype(np.float64)
    x = np.abs(x) / np.sqrt((x * x).mean(1, keepdims=True) + 1e-5)
    return ref, bound + 8 * 2.0 ** -24 * (x @ np.abs(E.astype(np.float64)).T)


@pytest.mark.parametrize("T", [1, 16, 17, 33, 64])   # one row tile, two, two groups of two
@pytest.mark.parametrize("V,d", [
    (16, 16),        # one column tile, half a k block
    (300, 48),       # ragged columns, k tail
    (3070, 1024),    # two column tiles per workgroup from 33 rows on
    (5001, 144),     # workgroups walk column groups, ragged last group
    (4099, 1040),    # K past four blocks per wave: two passes, or eight blocks in one
    (700, 2064),     # K past eight blocks per wave: several passes
    (130, 4096),     # the longest rows
])
def test_matches_float64(device, T, V, d):   # noqa: F811
    print(f"[case] step projection T={T} V={V} d={d}", flush=True)
    r = np.random.default_rng(T + V)
    E = r.standard_normal((V, d)).astype(np.float32)
    ids = r.integers(0, V, T).astype(np.uint32)
    got = logits_of(device, E, ids)
    ref, bound = bounded(E, ids)
    ratio = float((np.abs(got - ref) / bound).max())
    rel = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
    print(f"  worst |err| / bound {ratio:.3f}, relative 2-norm {rel:.2e}")
    assert np.isfinite(got).all() and ratio <= 1.0 and rel <= 1e-6


@pytest.mark.parametrize("T", [5, 40])
def test_scales_and_non_finite(device, T):   # noqa: F811
    """Columns from 1e-30 to 1e30, single large elements, a zero column, inf, -inf and NaN; and
    rows with an element far above the others."""
    print(f"[case] step projection scales and non-finite T={T}", flush=True)
    r = np.random.default_rng(3)
    V, d = 300, 256
    E = r.standard_normal((V, d)).astype(np.float32)
    E[90:100, 11] = 1e4
    E[100:160] *= 10.0 ** np.linspace(-30, 30, 60)[:, None].astype(np.float32)
    E[160:170, 7] = 1e6
    E[170] = 0.0
    E[171, 3], E[172, 5], E[173, 9] = np.inf, -np.inf, np.nan
    E[174, 3], E[174, 4] = np.inf, -np.inf
    ids = (99 - np.arange(T)).astype(np.uint32)     # finite rows
    got = logits_of(device, E, ids)
    with np.errstate(all="ignore"):
        ref, bound = bounded(E, ids)
    fin = np.r_[0:171, 175:V]
    assert np.isfinite(got[:, fin]).all()
    ratio = float((np.abs(got - ref) / (bound + 1e-37))[:, fin].max())
    print(f"  worst |err| / bound {ratio:.3f}")
    assert ratio <= 1.0
    np.testing.assert_array_equal(np.isnan(got[:, 171:175]), np.isnan(ref[:, 171:175]))
    for c in (171, 172):
        np.testing.assert_array_equal(got[:, c], ref[:, c].astype(np.float32))


@pytest.mark.parametrize("small", ["inverse", "zero"])
@pytest.mark.parametrize("big", [1e5, 1e6, 1e8, 2.0 ** 34])
@pytest.mark.parametrize("T,V,d", [(1, 300, 768), (40, 130, 2064), (64, 3100, 1024)])
def test_wide_rows_keep_fp32_precision(device, T, V, d, big, small):   # noqa: F811
    """As in the prefill's test: one large element in a row against 1 / it, or 0, in the other
    operand's row. Outputs formed again add K / 16 terms in order and 4 levels of a tree."""
    print(f"[case] step projection wide rows T={T} V={V} d={d} big={big:g} {small}", flush=True)
    r = np.random.default_rng(d)
    E = wide_rows(r, V, d, big, 7)
    E[:V // 2, 7] = r.standard_normal(V // 2) / big if small == "inverse" else 0.0
    for ids in (r.integers(V // 2, V, T), r.integers(0, V // 2, T)):
        got = logits_of(device, E, ids.astype(np.uint32))
        ref, bound = bounded(E, ids)
        meets = np.arange(V) < V // 2 if ids[0] >= V // 2 else np.arange(V) >= V // 2
        ratio = float((np.abs(got - ref) / bound).max())
        rel = float(np.linalg.norm((got - ref)[:, meets]) / np.linalg.norm(ref[:, meets]))
        print(f"  worst |err| / bound {ratio:.3f}, relative 2-norm of large against small {rel:.2e}")
        assert np.isfinite(got).all() and ratio <= 1.0 and rel <= 1e-6


@pytest.mark.parametrize("V,d", [(300, 768), (4099, 1040), (4099, 2064), (3100, 4096)])
def test_rows_do_not_depend_on_their_batch(device, V, d):   # noqa: F811
    """A row's logits have the same bits in batches of 1 to 64, which take one or two row tiles per
    workgroup and one or several passes over K."""
    print(f"[case] step projection batches V={V} d={d}", flush=True)
    r = np.random.default_rng(d)
    E = r.standard_normal((V, d)).astype(np.float32)
    ids = r.integers(0, V, 64).astype(np.uint32)
    whole = logits_of(device, E, ids)
    for T in (1, 16, 17, 40):
        np.testing.assert_array_equal(logits_of(device, E, ids[:T]), whole[:T])
