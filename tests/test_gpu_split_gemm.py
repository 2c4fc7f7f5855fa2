"""The prefill projections' split fp16 product (gemm_h3.hip) against float64, through the LM head
of a model without layers: logits = RMSNorm(E[ids]) E^T, so every operand is known.

Bound per element, with S = sum_k |x_k e_k|: each of the 3 ceil(K / 32) matrix instructions
rounds the running sum, whose magnitude is at most S, to 2^-24; the operands are held to 2^-23
each, the product of the low parts left out is at most 2^-22 of a term, and the fp32 RMSNorm of
the rows adds at most 2^-22 (its sum of squares in pairs, rsqrt and two products). That is
(3 ceil(K / 32) 2^-24 + 2^-20) S; an element on the diagonal (all terms of one sign) comes near
it. Over the whole result the errors are random, and the relative 2-norm stays under 1e-6 (a
product of the high parts alone is 1e-4 off).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def device():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from ssmjs_amd import backend
    d = backend.Device(0)
    yield d
    d.destroy()


def logits_of(device, E, ids):
    from ssmjs_amd import backend, checkpoint
    V, d = E.shape
    cfg = {"vocabSize": V, "dModel": d, "numLayers": 0, "dState": 16, "dConv": 4, "expand": 2,
           "nHeads": 1, "nGroups": 1, "layers": []}
    m = backend.Model(device, cfg)
    dims, T = checkpoint.unpack(m.export_weights())
    T["embedding"] = E
    m.load_weights(checkpoint.pack(dims, T))
    out = m.forward(ids[None])[0]
    m.destroy()
    return out


def reference(E, ids):
    """x E^T in float64, x the fp32 RMSNorm's exact value, and the bound of its elements."""
    x = E[ids].astype(np.float64)
    x = x / np.sqrt((x * x).mean(1, keepdims=True) + 1e-5)
    E64 = E.astype(np.float64)
    K = E.shape[1]
    bound = (3 * -(-K // 32) * 2.0 ** -24 + 2.0 ** -20) * (np.abs(x) @ np.abs(E64).T)
    return x @ E64.T, bound


@pytest.mark.parametrize("T,V,d", [
    (65, 16, 32),        # the least rows; one row block of columns, one k block
    (70, 64, 1024),      # one tile: split over K, finished by the second launch
    (129, 130, 36),      # ragged in every dimension; V % 4 != 0 never splits
    (300, 1000, 100),    # K tail, ragged tiles
    (1000, 544, 256),    # 64 x 64 tiles
    (150, 8000, 1024),   # wide: 128-column tiles
    (4090, 4084, 64),    # 256 x 256 tiles, ragged edges
    (2050, 4100, 2052),  # 128 x 128 tiles, K in more than 64 blocks, K tail
    (90, 150, 4180),     # K past what the packing keeps in registers, K tail
])
def test_matches_float64(device, T, V, d):
    print(f"[case] split product T={T} V={V} d={d}", flush=True)
    r = np.random.default_rng(T + V)
    E = r.standard_normal((V, d)).astype(np.float32)
    ids = r.integers(0, V, T).astype(np.uint32)
    got = logits_of(device, E, ids)
    ref, bound = reference(E, ids)
    ratio = float((np.abs(got - ref) / bound).max())
    rel = float(np.linalg.norm(got - ref) / np.linalg.norm(ref))
    print(f"  worst |err| / bound {ratio:.3f}, relative 2-norm {rel:.2e}")
    assert np.isfinite(got).all() and ratio <= 1.0 and rel <= 1e-6


def test_scales_and_non_finite(device):
    """Rows from 1e-30 to 1e30, rows with a single large element, a zero row, and rows with
    inf, -inf or NaN: the finite columns keep the bound, the others get fp32's own inf / NaN."""
    print("[case] split product scales and non-finite", flush=True)
    r = np.random.default_rng(3)
    V, d, T = 200, 256, 100
    E = r.standard_normal((V, d)).astype(np.float32)
    E[100:160] *= 10.0 ** np.linspace(-30, 30, 60)[:, None].astype(np.float32)
    E[160:170, 7] = 1e6
    E[170] = 0.0
    E[171, 3], E[172, 5], E[173, 9] = np.inf, -np.inf, np.nan
    E[174, 3], E[174, 4] = np.inf, -np.inf
    ids = r.integers(0, 100, T).astype(np.uint32)     # finite, ordinary rows
    got = logits_of(device, E, ids)
    with np.errstate(all="ignore"):
        ref, bound = reference(E, ids)
    fin = np.r_[0:171, 175:V]
    assert np.isfinite(got[:, fin]).all()
    ratio = float((np.abs(got - ref) / (bound + 1e-37))[:, fin].max())
    print(f"  worst |err| / bound {ratio:.3f}")
    assert ratio <= 1.0
    np.testing.assert_array_equal(np.isnan(got[:, 171:175]), np.isnan(ref[:, 171:175]))
    for c in (171, 172):
        np.testing.assert_array_equal(got[:, c], ref[:, c].astype(np.float32))


def wide_rows(r, n, d, big, at):
    """n rows of unit normals, those from n / 2 on with one element of size `big` at column `at`."""
    E = r.standard_normal((n, d)).astype(np.float32)
    E[n // 2:, at] = big
    return E


@pytest.mark.parametrize("small", ["inverse", "zero"])
@pytest.mark.parametrize("big", [1e5, 1e6, 1e8, 2.0 ** 34])
@pytest.mark.parametrize("T,V,d", [(70, 64, 1024),     # split over K
                                   (300, 400, 768), (1500, 2050, 256)])
def test_wide_rows_keep_fp32_precision(device, T, V, d, big, small):
    """One large element in a row against 1 / it, or 0, in the other operand's row, so that the sum
    is made of elements far below their row's largest. Outputs formed again take the fp32 matrix
    cores' K / 4 roundings instead of the split's."""
    print(f"[case] split product wide rows T={T} V={V} d={d} big={big:g} {small}", flush=True)
    r = np.random.default_rng(d)
    E = wide_rows(r, V, d, big, 7)
    E[:V // 2, 7] = r.standard_normal(V // 2) / big if small == "inverse" else 0.0
    ids = r.integers(0, V, T).astype(np.uint32)
    got = logits_of(device, E, ids)
    ref, bound = reference(E, ids)
    per = 3 * -(-d // 32) * 2.0 ** -24 + 2.0 ** -20
    bound *= max(per, d // 4 * 2.0 ** -24 + 2.0 ** -22) / per
    ratio = float((np.abs(got - ref) / bound).max())
    meets = np.ix_(ids >= V // 2, np.arange(V) < V // 2)
    rel = float(np.linalg.norm((got - ref)[meets]) / np.linalg.norm(ref[meets]))
    print(f"  worst |err| / bound {ratio:.3f}, relative 2-norm of large against small {rel:.2e}")
    assert np.isfinite(got).all() and ratio <= 1.0 and rel <= 1e-6


def test_non_finite_in_split_slices(device):
    """inf, -inf and NaN in a product split over K: a row with one of them, and rows with inf and
    -inf in different slices, whose sum is NaN only after the slices are added."""
    print("[case] split product non-finite slices", flush=True)
    r = np.random.default_rng(5)
    T, V, d = 70, 64, 1024
    E = r.standard_normal((V, d)).astype(np.float32)
    E[60, 3], E[61, 1000], E[62, 500] = np.inf, -np.inf, np.nan
    E[63, 3], E[63, 1000] = np.inf, -np.inf
    ids = r.integers(0, 60, T).astype(np.uint32)
    x = np.sign(E[ids][:, [3, 1000]])
    got = logits_of(device, E, ids)
    ref, bound = reference(E[:60], ids)
    assert float((np.abs(got[:, :60] - ref) / bound).max()) <= 1.0
    np.testing.assert_array_equal(got[:, 60], x[:, 0] * np.inf)
    np.testing.assert_array_equal(got[:, 61], -x[:, 1] * np.inf)
    assert np.isnan(got[:, 62]).all()
    np.testing.assert_array_equal(got[:, 63], np.where(x[:, 0] == x[:, 1], np.nan, x[:, 0] * np.inf))
