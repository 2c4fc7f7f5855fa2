"""The fused one-token step of Mamba-2 layers with d_state 16 and 32 against the oracle: logits and
the whole state over a few decode steps, from a prefilled state (the bound of test_gpu_model.py)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from test_gpu_model import _model, case, close, device  # noqa: E402,F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [16, 32])
@pytest.mark.parametrize("H,B", [
    (4, 1),     # head dim 64: one workgroup per head
    (2, 17),    # head dim 128: two; two row tiles with padding rows
    (32, 3),    # head dim 8: guarded rows, partial sums of 32 heads
    (1, 33),    # head dim 256
])
def test_decode_matches_oracle(device, N, H, B):   # noqa: F811
    case(f"fused Mamba-2 step N={N} H={H} B={B}")
    m, blob = _model(device, ["mamba2", "mamba2"], N=N, H=H)
    om = O.Model(blob)
    ids = np.random.default_rng(N + H).integers(0, 512, (B, 9)).astype(np.uint32)
    st, ost = m.new_state(B), om.new_state(B)
    lg, _ = st.prefill(ids[:, :5])
    close(lg, ost.prefill(ids[:, :5]), "logits")
    for t in range(5, 9):
        lg, _ = st.decode(ids[:, t])
        close(lg, ost.decode(ids[:, t]), "logits")
    close(st.read(), ost.read(), "state")
    st.destroy()
    m.destroy()
