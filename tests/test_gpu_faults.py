"""Failure handling forced from the host (ssm_set_fault_injection), as SURVEY's auxiliary plan asks:
every kernel still runs normally; the library reports the injected failure through the error
contract of the reference (src/session/session.ts:262-270,393-401; errors.ts:5-13), and the
same device and model work again once the fault is cleared.
  alloc   every device allocation fails -> SSM_ERR_OUT_OF_MEMORY ('UNKNOWN' to the session,
          which wraps model construction failures as 'UNKNOWN', session.ts:359-362)
  launch  every launch check reports a failure -> SSM_ERR_HIP ('UNKNOWN')
"""
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")
from oracle import oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu


def case(msg):
    print(f"[case] {msg}", flush=True)
    sys.stdout.flush()


@pytest.fixture
def inject():
    """Sets the library's injected fault for one test and always clears it afterwards."""
    from ssmjs_amd import _lib

    def set_kind(kind):
        _lib.call("ssm_set_fault_injection", None if kind is None else kind.encode())
    yield set_kind
    set_kind(None)


@pytest.fixture(scope="module")
def device():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from ssmjs_amd import backend
    d = backend.Device(0)
    yield d
    d.destroy()


CFG = {"vocabSize": 64, "dModel": 64, "numLayers": 2, "dState": 16, "dConv": 4, "expand": 2,
       "nHeads": 2, "layers": [{"type": "mamba1"}, {"type": "mamba2"}]}


def test_alloc_failure_then_recovery(device, inject):
    case("injected fault: alloc")
    from ssmjs_amd import _lib, backend
    inject("alloc")
    with pytest.raises(_lib.SsmError) as e:
        backend.Model(device, CFG, seed=1)
    assert e.value.status == 6 and e.value.code == "UNKNOWN"   # SSM_ERR_OUT_OF_MEMORY
    inject(None)
    m = backend.Model(device, CFG, seed=1)
    # a workspace that has to grow under the fault fails the call, not the model
    inject("alloc")
    ids = np.arange(40, dtype=np.uint32).reshape(2, 20) % 64
    with pytest.raises(_lib.SsmError) as e:
        m.forward(ids)
    assert e.value.status == 6
    inject(None)
    out = m.forward(ids)
    ref = O.Model(m.export_weights()).forward(ids)
    assert np.abs(out - ref).max() <= 1e-4 * max(1.0, np.abs(ref).max())
    m.destroy()


def test_launch_failure_then_recovery(device, inject):
    case("injected fault: launch")
    from ssmjs_amd import _lib, backend
    m = backend.Model(device, CFG, seed=2)
    ids = np.arange(30, dtype=np.uint32).reshape(1, 30) % 64
    inject("launch")
    with pytest.raises(_lib.SsmError) as e:
        m.forward(ids)
    assert e.value.status == 5 and e.value.code == "UNKNOWN"   # SSM_ERR_HIP
    assert "injected" in str(e.value)
    st = m.new_state(1)
    with pytest.raises(_lib.SsmError):
        st.prefill(ids)
    inject(None)
    device.synchronize()
    out = m.forward(ids)
    ref = O.Model(m.export_weights()).forward(ids)
    assert np.abs(out - ref).max() <= 1e-4 * max(1.0, np.abs(ref).max())
    st.destroy()
    m.destroy()


def test_failed_weight_packing_is_built_anew(device, inject):
    """A launch failure while the projections' packed weights are built (the first mixer call of
    more than 64 rows): the next call packs them from the start."""
    case("injected fault: launch, weight packing")
    from ssmjs_amd import _lib, backend
    m = backend.Model(device, CFG, seed=2)
    om = O.Model(m.export_weights())
    d = CFG["dModel"]
    x = np.random.default_rng(0).standard_normal((1, 90, d)).astype(np.float32)
    xd = torch.from_numpy(x).cuda()
    y = torch.empty_like(xd)
    torch.cuda.synchronize()
    args = ("ssm_mixer_forward_device", m.handle, 0, xd.data_ptr(), y.data_ptr(), 1, 90)
    inject("launch")
    with pytest.raises(_lib.SsmError):
        _lib.call(*args)
    inject(None)
    _lib.call(*args)
    device.synchronize()
    ref = om.mixer(0, x)
    assert np.abs(y.cpu().numpy() - ref).max() <= 1e-4 * np.abs(ref).max()
    m.destroy()


def test_failed_step_packing_is_built_anew(device, inject):
    """A launch failure while the one-token step's packed weights are built (a decode's first
    launches): the next step packs them from the start."""
    case("injected fault: launch, step weight packing")
    from ssmjs_amd import _lib, backend
    m = backend.Model(device, CFG, seed=3)
    om = O.Model(m.export_weights())
    ids = np.array([5, 9], np.uint32)
    st = m.new_state(2)
    inject("launch")
    with pytest.raises(_lib.SsmError):
        st.decode(ids)
    inject(None)
    st.reset()
    got = st.decode(ids)[0]
    ref = om.forward(ids[:, None])[:, 0]
    assert np.abs(got - ref).max() <= 1e-4 * max(1.0, np.abs(ref).max())
    m.destroy()


def test_failed_bf16_cast_is_built_anew(device, inject):
    """The same for the bf16 layer's weights (its call's first launches)."""
    case("injected fault: launch, bf16 weights")
    from ssmjs_amd import _lib, backend
    cfg = dict(CFG, dState=64, nHeads=2, layers=[{"type": "mamba2"}] * 2)
    outs = []
    for fail in (False, True):
        m = backend.Model(device, cfg, seed=4)
        x = torch.from_numpy(np.random.default_rng(0).standard_normal((1, 90, cfg["dModel"]))
                             .astype(np.float32)).cuda()
        y = torch.empty_like(x)
        torch.cuda.synchronize()
        args = ("ssm_mixer_forward_device_bf16", m.handle, 0, x.data_ptr(), y.data_ptr(), 1, 90)
        if fail:
            inject("launch")
            with pytest.raises(_lib.SsmError):
                _lib.call(*args)
            inject(None)
        _lib.call(*args)
        device.synchronize()
        outs.append(y.cpu().numpy())
        m.destroy()
    np.testing.assert_array_equal(outs[0], outs[1])


def test_failed_reload_leaves_no_old_copies(device, inject):
    """Weights loaded while every launch fails, into a model whose derived copies all exist and
    whose step is captured: the next calls (decode, long and short prefill) use the new weights."""
    case("injected fault: launch, reload")
    from ssmjs_amd import _lib, backend
    m, other = backend.Model(device, CFG, seed=5), backend.Model(device, CFG, seed=6)
    blob = other.export_weights()
    om = O.Model(blob)
    st = m.new_state(2)
    ids = np.array([5, 9], np.uint32)
    for _ in range(3):            # eager, captured, replayed
        st.reset()
        st.decode(ids)
    long_ids = (np.arange(100, dtype=np.uint32) * 7 % 64)[None]
    m.forward(long_ids)
    inject("launch")
    with pytest.raises(_lib.SsmError):
        m.load_weights(blob)
    inject(None)
    st.reset()
    for got, ref in ((st.decode(ids)[0], om.forward(ids[:, None])[:, 0]),
                     (m.forward(long_ids), om.forward(long_ids)),
                     (m.forward(long_ids[:, :20]), om.forward(long_ids[:, :20]))):
        assert np.abs(got - ref).max() <= 1e-4 * max(1.0, np.abs(ref).max())
    m.destroy()
    other.destroy()


@pytest.mark.parametrize("nth,what", [(2, "workspace"), (3, "layers"), (4, "embedding")])
def test_no_room_for_packed_operands(device, inject, nth, what):
    """A long prompt when the device has no room for the workspace with the packed activations,
    the packed weights or the packed embedding (the allocations after the ids): it runs on the
    unpacked operands and agrees with the oracle; so does the same prompt after the weights are
    loaded again, packed."""
    case(f"injected fault: one allocation, {what}")
    from ssmjs_amd import _lib, backend
    m = backend.Model(device, CFG, seed=7)
    ids = (np.arange(100, dtype=np.uint32) * 7 % 64)[None]
    ref = O.Model(m.export_weights()).forward(ids)

    def check():
        assert np.abs(m.forward(ids) - ref).max() <= 1e-4 * max(1.0, np.abs(ref).max())
    inject(f"alloc:{nth}")
    check()
    inject("alloc")
    check()                       # (the failure was met: nothing more is allocated)
    inject(None)
    m.load_weights(m.export_weights())
    check()
    m.destroy()
    m = backend.Model(device, CFG, seed=7)
    inject("alloc:1")             # the ids: no call without them
    with pytest.raises(_lib.SsmError):
        m.forward(ids)
    inject(None)
    check()
    m.destroy()


def test_session_create_reports_model_failure(inject):
    """MambaSession.create with every allocation failing: the device opens (no allocation), the
    model construction fails and the session raises SessionError('UNKNOWN') as session.ts
    does for a throwing HybridMambaModel constructor."""
    case("MambaSession.create under an injected alloc fault")
    from ssmjs_amd import ByteTokenizer, MambaSession, SessionError
    inject("alloc")
    with pytest.raises(SessionError) as e:
        MambaSession.create({"tokenizer": ByteTokenizer(256), "mambaVersion": "mamba1",
                             "modelSize": "nano"})
    assert e.value.code == "UNKNOWN"
