"""The time-sliced Mamba-1 scan (16 states, few channels) against the oracle at the edges of its
slices (16 steps), blocks (64, 128, 256 steps) and channel groups (4), over every option it
takes; 1e-4 relative plus 2e-6 of the largest magnitude (fp32 sums of 16 terms, products of up
to 16 decays)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
from oracle import oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu


def close(got, ref, what):
    got, ref = got.cpu().numpy().astype(np.float64), np.asarray(ref, np.float64)
    ratio = float((np.abs(got - ref) / (1e-4 * np.abs(ref) + 2e-6 * np.abs(ref).max())).max())
    print(f"  {what}: worst |err|/bound {ratio:.3f}", flush=True)
    assert np.isfinite(got).all() and ratio <= 1.0


@pytest.mark.parametrize("B,L,D", [
    (1, 1, 1), (2, 16, 4), (1, 17, 6),            # one slice, one step of the next, partial group
    (1, 64, 100), (1, 65, 100), (3, 128, 33),     # 4-wave blocks, the first 8-wave length
    (1, 129, 64), (1, 256, 512), (2, 300, 130),   # 16-wave blocks
    (1, 1000, 1030),                              # 8-wave blocks, tail slice of 8 steps
    (2, 333, 1500),                               # more than 512 groups: 4-wave blocks
])
@pytest.mark.parametrize("opts", ["all", "none"])
def test_matches_oracle(B, L, D, opts):
    """"all": entering and final state, gate, skip, dt bias, softplus, strided inputs; "none": raw
    dt and nothing else."""
    print(f"[case] scan slices B={B} L={L} D={D} {opts}", flush=True)
    from ssmjs_amd import kernels
    r = np.random.default_rng(L * D)
    f = lambda *s: r.standard_normal(s).astype(np.float32)   # noqa: E731
    u, z, Bm, Cm, Dk, bias = f(B, L, D), f(B, L, D), f(B, L, 16), f(B, L, 16), f(D), f(D) - 1
    dt = f(B, L, D) - 1
    A = -r.uniform(0.5, 16, (D, 16)).astype(np.float32)
    h0 = f(B, D, 16)
    dev = lambda a: torch.from_numpy(a).cuda()   # noqa: E731
    if opts == "all":
        wide = torch.zeros(B, L, D + 40, device="cuda")
        wide[:, :, :D], wide[:, :, D:D + 16], wide[:, :, D + 20:D + 36] = dev(u), dev(Bm), dev(Cm)
        hT = torch.empty(B, D, 16, device="cuda")
        y = kernels.selective_scan(wide[:, :, :D], dev(dt), dev(A), wide[:, :, D:D + 16],
                                   wide[:, :, D + 20:D + 36], dev(Dk), dev(z), dev(bias), True,
                                   h0=dev(h0), hT=hT)
        torch.cuda.synchronize()
        ref, ref_h = O.selective_scan(u, dt, A, Bm, Cm, Dk, z, bias, True, h0=h0, return_state=True)
        close(hT, ref_h, "final state")
    else:
        dt = np.abs(dt) * 0.1
        y = kernels.selective_scan(dev(u), dev(dt), dev(A), dev(Bm), dev(Cm), softplus=False)
        torch.cuda.synchronize()
        ref = O.selective_scan(u, dt, A, Bm, Cm, None, None, None, False)
    close(y, ref, "y")


@pytest.mark.parametrize("B,L,D", [(1, 300, 130),     # time slices
                                   (1, 1100, 70), (2, 2047, 600), (1, 8192, 256)])   # chunks
def test_state_in_place(B, L, D):
    """hT in the place of h0 (a session's state): the same bits as with two buffers."""
    print(f"[case] scan state in place B={B} L={L} D={D}", flush=True)
    from ssmjs_amd import kernels
    r = np.random.default_rng(L)
    dev = lambda *s: torch.from_numpy(r.standard_normal(s).astype(np.float32)).cuda()   # noqa: E731
    u, dt, Bm, Cm, h0 = dev(B, L, D), dev(B, L, D) - 1, dev(B, L, 16), dev(B, L, 16), dev(B, D, 16)
    A = -dev(D, 16).abs()
    hT, state = torch.empty_like(h0), h0.clone()
    y = kernels.selective_scan(u, dt, A, Bm, Cm, h0=h0, hT=hT)
    y2 = kernels.selective_scan(u, dt, A, Bm, Cm, h0=state, hT=state)
    torch.cuda.synchronize()
    assert torch.equal(y, y2) and torch.equal(hT, state)


@pytest.mark.parametrize("L,D,N", [(2, 5, 16), (3, 5, 16),                        # time slices
                                   (2, 4112, 16), (2, 5, 4), (2, 5, 8), (2, 5, 32),   # single pass
                                   (2, 5, 64), (2, 5, 13)])
def test_row_stride_past_the_offset_range(L, D, N):
    """Rows 72 MB apart: step 60 of a 64- or 128-step block lies 2^32 bytes and a little on, which 32-bit
    offsets would bring back between the first two rows. The outputs agree with the oracle, and
    what lies between the rows (NaN) is neither read nor written."""
    print(f"[case] scan row stride L={L} D={D} N={N}", flush=True)
    from ssmjs_amd import kernels
    B, ld = 1, 18_000_000
    assert 60 * ld * 4 - 2 ** 32 in range(4 * D, 4 * ld)
    r = np.random.default_rng(L)
    f = lambda *s: r.standard_normal(s).astype(np.float32)   # noqa: E731
    u, Bm, Cm = f(B, L, D), f(B, L, N), f(B, L, N)
    dt = np.abs(f(B, L, D)) * 0.1
    A = -r.uniform(0.5, 16, (D, N)).astype(np.float32)

    def far(a):
        buf = torch.full(((L - 1) * ld + D + 64,), float("nan"), device="cuda")
        v = torch.as_strided(buf, a.shape, (L * ld, ld, 1))
        v.copy_(torch.from_numpy(a))
        return buf, v
    (_, ud), (_, dd), (_, bd), (_, cd), (ybuf, y) = (far(a) for a in (u, dt, Bm, Cm, 0 * u))
    hT = torch.empty(B, D, N, device="cuda")
    kernels.selective_scan(ud, dd, torch.from_numpy(A).cuda(), bd, cd, softplus=False, out=y, hT=hT)
    torch.cuda.synchronize()
    ref, ref_h = O.selective_scan(u, dt, A, Bm, Cm, None, None, None, False, return_state=True)
    close(y, ref, "y")
    close(hT, ref_h, "final state")
    assert int((~torch.isnan(ybuf)).sum()) == L * D
