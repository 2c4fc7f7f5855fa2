"""The fp32 matrix-core SSD at the session presets' Mamba-2 shapes (d_state 16 and 32, head dims in
multiples of 64) against the oracle, with the bound of the other fp32 SSD tests: 1e-4 relative
plus 2e-6 of the largest magnitude (32-term products and chunk sums in fp32)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
from oracle import oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu


def inputs(seed, B, L, H, P, G, N):
    r = np.random.default_rng(seed)
    f = lambda *s: r.standard_normal(s).astype(np.float32)   # noqa: E731
    return (f(B, L, H, P), f(B, L, H) - 3, -r.uniform(1, 16, H).astype(np.float32),
            f(B, L, G, N), f(B, L, G, N), f(H), (0.3 * r.standard_normal((B, H, P, N))).astype(np.float32))


def close(got, ref, what):
    got, ref = got.cpu().numpy().astype(np.float64), np.asarray(ref, np.float64)
    ratio = float((np.abs(got - ref) / (1e-4 * np.abs(ref) + 2e-6 * np.abs(ref).max())).max())
    print(f"  {what}: worst |err|/bound {ratio:.3f}", flush=True)
    assert np.isfinite(got).all() and ratio <= 1.0


@pytest.mark.parametrize("B,L,H,G,N,P", [
    (1, 1, 1, 1, 16, 64),        # one step, one head: one head per workgroup
    (1, 33, 3, 1, 16, 64),       # odd heads; a second chunk of one step
    (2, 100, 2, 1, 32, 64),      # 32 states, two heads per workgroup
    (1, 700, 4, 2, 16, 128),     # two groups, 128-wide heads, segments
    (1, 2000, 12, 1, 16, 128),   # the large preset
    (1, 4097, 1, 1, 32, 192),    # three 64-row parts of one head, many segments, ragged
    (1, 300, 4, 2, 64, 128),     # 64 and 128 states: heads of several 64-row parts
    (2, 130, 3, 1, 128, 128),
])
@pytest.mark.parametrize("state,clamp", [(True, False), (False, True)])
def test_matches_oracle(B, L, H, G, N, P, state, clamp):
    print(f"[case] ssd presets B={B} L={L} H={H} G={G} N={N} P={P} {state} {clamp}", flush=True)
    from ssmjs_amd import kernels
    x, dt, A, Bm, Cm, D, h0 = inputs(L + N, B, L, H, P, G, N)
    lim = (0.05, 0.2) if clamp else (0.0, float("inf"))
    ref, hT = O.ssd(x, dt, A, Bm, Cm, D, h0=h0 if state else None, return_state=True,
                    dt_min=lim[0], dt_max=lim[1])
    t = [torch.from_numpy(a).cuda() for a in (x, dt, A, Bm, Cm, D, h0)]
    out = torch.empty(B, H, P, N, device="cuda")
    y = kernels.ssd_chunk_scan(*t[:6], dt_min=lim[0], dt_max=lim[1], h0=t[6] if state else None,
                               hT=out)
    torch.cuda.synchronize()
    close(y, ref, "y")
    close(out, hT, "final state")


def test_unaligned_rows_keep_their_route():
    """Rows that are not 16-byte aligned are accepted as before (the scan over H*P channels, or
    without a workspace the sequential kernel) and agree with the matrix-core kernel."""
    print("[case] ssd presets unaligned", flush=True)
    from ssmjs_amd import kernels
    B, L, H, G, N, P = 1, 300, 4, 1, 16, 64
    x, dt, A, Bm, Cm, D, h0 = inputs(7, B, L, H, P, G, N)
    ref = O.ssd(x, dt, A, Bm, Cm, D, h0=h0)
    t = [torch.from_numpy(a).cuda() for a in (x, dt, A, Bm, Cm, D, h0)]
    wide = torch.zeros(B, L, H * P + 1, device="cuda")
    wide[:, :, 1:] = t[0].reshape(B, L, H * P)
    xs = torch.as_strided(wide, (B, L, H, P), (L * (H * P + 1), H * P + 1, P, 1), 1)
    for ws in (None, torch.empty(1, dtype=torch.uint8, device="cuda")):
        y = kernels.ssd_chunk_scan(xs, *t[1:6], h0=t[6], workspace=ws)
        torch.cuda.synchronize()
        close(y, ref, "y")


@pytest.mark.parametrize("H,N", [(4, 16), (2, 16), (2, 32)])
def test_mixer_matches_oracle(H, N):
    """A whole Mamba-2 layer (the gated output, one sum of squares per 64 channels) at head dims
    64 and 128, and a prompt short enough for the row kernel."""
    print(f"[case] preset mixer H={H} N={N}", flush=True)
    from ssmjs_amd import _lib, backend
    dev = backend.Device(0)
    cfg = {"vocabSize": 16, "dModel": 128, "numLayers": 1, "dState": N, "dConv": 4, "expand": 2,
           "nHeads": H, "nGroups": 1, "layers": [{"type": "mamba2"}]}
    m = backend.Model(dev, cfg, seed=5)
    om = O.Model(m.export_weights())
    for B, L in ((1, 65), (2, 333), (1, 20)):
        x = np.random.default_rng(L).standard_normal((B, L, 128)).astype(np.float32)
        xd = torch.from_numpy(x).cuda()
        y = torch.empty_like(xd)
        torch.cuda.synchronize()
        _lib.call("ssm_mixer_forward_device", m.handle, 0, xd.data_ptr(), y.data_ptr(), B, L)
        dev.synchronize()
        close(y, om.mixer(0, x), f"mixer B={B} L={L}")
    m.destroy()
    dev.destroy()


@pytest.mark.parametrize("B,L,H,N,P", [(1, 64, 8, 16, 64), (2, 333, 12, 16, 128), (1, 90, 4, 32, 64),
                                       (1, 64, 4, 64, 128), (1, 100, 3, 128, 192)])
def test_fast_decay_keeps_precision(B, L, H, N, P):
    """Heads whose decay reaches tens of log2 units within a chunk: y and the final state against
    float64 in the 2-norm. A step's decay and weight are a rounded exponent difference d (d 2^-24
    ln 2, at most 0.53 2^-24 after its weight 2^-d), 2^x, softplus and three products: 5 roundings
    of 2^-24, and the last 16-wide sum's few; 6e-7 together. (A running sum in fp32 loses 1.3e-6.)"""
    print(f"[case] ssd fast decay B={B} L={L} H={H} N={N} P={P}", flush=True)
    from ssmjs_amd import kernels
    x, dt, _, Bm, Cm, D, h0 = inputs(L, B, L, H, P, 1, N)
    A = -np.linspace(12, 16, H).astype(np.float32)
    dt += 1
    t = [torch.from_numpy(a).cuda() for a in (x, dt, A, Bm, Cm, D, h0)]
    out = torch.empty(B, H, P, N, device="cuda")
    y = kernels.ssd_chunk_scan(*t[:6], h0=t[6], hT=out)
    torch.cuda.synchronize()
    x, dt, A, Bm, Cm, D, h = (a.astype(np.float64) for a in (x, dt, A, Bm, Cm, D, h0))
    d = np.log1p(np.exp(dt))
    ref = np.empty_like(x)
    for i in range(L):
        h = (np.exp(d[:, i] * A)[:, :, None, None] * h +
             (d[:, i, :, None] * x[:, i])[..., None] * Bm[:, i, 0][:, None, None])
        ref[:, i] = (h * Cm[:, i, 0][:, None, None]).sum(-1) + D[:, None] * x[:, i]
    for got, want, what in ((y, ref, "y"), (out, h, "final state")):
        rel = np.linalg.norm(got.cpu().numpy() - want) / np.linalg.norm(want)
        print(f"  {what}: relative 2-norm {rel:.2e}", flush=True)
        assert rel <= 6e-7


@pytest.mark.parametrize("B,L,H,N,P", [(1, 33, 2, 16, 64), (1, 2000, 12, 16, 128),
                                       (4, 3000, 9, 32, 128)])
def test_state_in_place(B, L, H, N, P):
    """hT in the place of h0 (a session's state, as the mixer calls it): the same bits as with two
    buffers, though the last segment's workgroup may end before another segment's starts."""
    print(f"[case] ssd state in place B={B} L={L} H={H} N={N} P={P}", flush=True)
    from ssmjs_amd import kernels
    t = [torch.from_numpy(a).cuda() for a in inputs(L, B, L, H, P, 1, N)]
    hT = torch.empty_like(t[6])
    y = kernels.ssd_chunk_scan(*t[:6], h0=t[6], hT=hT)
    state = t[6].clone()
    y2 = kernels.ssd_chunk_scan(*t[:6], h0=state, hT=state)
    torch.cuda.synchronize()
    assert torch.equal(y, y2) and torch.equal(hT, state)


@pytest.mark.parametrize("P,N", [(64, 16), (128, 32), (128, 64)])
@pytest.mark.parametrize("what", [np.inf, -np.inf, np.nan])
def test_non_finite_x_stays_causal(P, N, what):
    """x inf or NaN at one step of one channel, at every place of a 16-step tile: the steps before
    it and the other channels keep the bits that they have without it, and from it on the channel
    is not finite."""
    print(f"[case] ssd non-finite x P={P} N={N} {what}", flush=True)
    from ssmjs_amd import kernels
    B, L, H = 1, 70, 2
    t = [torch.from_numpy(a).cuda() for a in inputs(N, B, L, H, P, 1, N)]
    clean = kernels.ssd_chunk_scan(*t[:6])
    x = t[0]
    for step in list(range(16)) + [31, 32, 47, 69]:
        h, p = step % H, (7 * step) % P
        keep = x[0, step, h, p].item()
        x[0, step, h, p] = what
        y = kernels.ssd_chunk_scan(x, *t[1:6])
        torch.cuda.synchronize()
        x[0, step, h, p] = keep
        assert not torch.isfinite(y[0, step:, h, p]).any()
        y[0, step:, h, p] = clean[0, step:, h, p]
        assert torch.equal(y, clean), f"step {step}"
