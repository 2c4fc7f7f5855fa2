"""The work that a program using this framework has it do, as measurable cases.

Families (the case's "kind"):
  conv_scan  causal conv1d + SiLU, then the Mamba-1 selective scan (kernel level, fp32)
  m1_layer   one Mamba-1 mixer over a prompt batch (fp32)
  m2_layer   one Mamba-2 mixer over a prompt batch, fp32 or the bf16-input variant
  ssd        the Mamba-2 SSD over a prompt batch, fp32 or bf16 inputs
  decode     one recurrent token step of a whole model: logits, greedy picks, states
  sample     sampleToken on the device over a batch of logits

`listed` names the cases, `draw` gives more of the same ranges, `prepare` makes what a program
holds before the call, `run` is one pass through the public entry points, `work` counts the
bytes and operations a pass cannot do without, `tolerance` and `exact` say what the result has
to be.
"""
from __future__ import annotations

import math

import numpy as np
import torch
import torch.nn.functional as F

from ssmjs_amd import _lib, backend, checkpoint, kernels

# Model sizes in use: the session presets (d_model, heads; d_state 16) and the wider Mamba-2
# layers of the benchmark configurations (head dim 64, d_state 64 or 128).
PRESETS = {"nano": (128, 4, 4), "small": (256, 8, 6), "medium": (512, 8, 8),
           "large": (768, 12, 12)}          # name: (d_model, n_heads, n_layers)
M2_SIZES = [(128, 4, 16), (256, 8, 16), (512, 8, 16), (768, 12, 16), (1024, 32, 64),
            (1024, 32, 128), (2048, 64, 128)]   # (d_model, n_heads, d_state)
K_CONV = 4


def listed():
    return [
        # the smallest kernel-level call: 256 tokens of one sequence, where launches count
        {"name": "conv_scan_256", "kind": "conv_scan", "B": 1, "L": 256, "D": 512, "N": 16,
         "state": False},
        # a long single prompt continuing from a carried state, ragged length, the large
        # preset's channels: few channels, many steps
        {"name": "scan_prompt_2047", "kind": "conv_scan", "B": 1, "L": 2047, "D": 1536, "N": 16,
         "state": True},
        # a session's prompt through one layer of the medium preset (batch 1)
        {"name": "m1_layer_prompt", "kind": "m1_layer", "B": 1, "L": 200, "d": 512, "N": 16},
        # batched prefill through one layer at the large preset's width
        {"name": "m1_layer_batch", "kind": "m1_layer", "B": 4, "L": 2048, "d": 768, "N": 16},
        # a 1000-token prompt through one Mamba-2 layer of the 32-head model, fp32
        {"name": "m2_layer_prompt", "kind": "m2_layer", "dtype": "f32", "B": 1, "L": 1000,
         "d": 1024, "H": 32, "N": 128},
        # batched prefill through the widest Mamba-2 layer with bf16 operands: the largest call
        {"name": "m2_layer_bf16", "kind": "m2_layer", "dtype": "bf16", "B": 8, "L": 4096,
         "d": 2048, "H": 64, "N": 128},
        # the SSD core of that layer in fp32
        {"name": "ssd_f32_batch", "kind": "ssd", "dtype": "f32", "B": 8, "L": 4096, "H": 64,
         "P": 64, "G": 1, "N": 128, "state": False},
        # one very long document, bf16 inputs
        {"name": "ssd_bf16_long", "kind": "ssd", "dtype": "bf16", "B": 1, "L": 65536, "H": 32,
         "P": 64, "G": 1, "N": 128, "state": False},
        # the large preset's Mamba-2 heads (128 wide, 16 states) over a prompt that continues
        # from a carried state
        {"name": "ssd_preset", "kind": "ssd", "dtype": "f32", "B": 1, "L": 2000, "H": 12,
         "P": 128, "G": 1, "N": 16, "state": True},
        # serving: one token for each of 64 cached sequences (8 of the 24 layers of the 32-head
        # model: the states still exceed the last-level cache)
        {"name": "decode_m2_64", "kind": "decode", "layer": "mamba2", "B": 64, "d": 1024,
         "H": 32, "N": 128, "layers": 8, "V": 32000},
        # a session's own token step: the large preset, batch 1
        {"name": "decode_m1_1", "kind": "decode", "layer": "mamba1", "B": 1, "d": 768, "H": 12,
         "N": 16, "layers": 12, "V": 32000},
        # sampled serving: the draw for 64 sequences
        {"name": "sample_64", "kind": "sample", "rows": 64, "n": 32000, "topK": 50, "topP": 0.9,
         "temperature": 0.8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["conv_scan", "m1_layer", "m2_layer", "m2_layer", "ssd", "ssd", "decode",
                       "decode", "sample"])
    if kind == "conv_scan":
        B = rng.randint(1, 4)
        D = rng.choice([256, 512, 1024, 1536, 4 * rng.randint(32, 400)])
        return {"kind": kind, "B": B, "L": _log_int(rng, 64, 4096 // B), "D": D,
                "N": rng.choice([16, 16, 16, 8, 32]), "state": rng.random() < 0.5}
    if kind == "m1_layer":
        B = rng.randint(1, 4)
        d = rng.choice([p[0] for p in PRESETS.values()])
        return {"kind": kind, "B": B, "L": _log_int(rng, 16, 2048), "d": d, "N": 16}
    if kind == "m2_layer":
        dtype = rng.choice(["f32", "f32", "bf16"])
        d, H, N = rng.choice([s for s in M2_SIZES if dtype == "f32" or s[2] >= 64])
        B = rng.randint(1, 4)
        most = 4096 if dtype == "f32" else 16384
        return {"kind": kind, "dtype": dtype, "B": B, "L": _log_int(rng, 16, most // B), "d": d,
                "H": H, "N": N}
    if kind == "ssd":
        dtype = rng.choice(["f32", "bf16"])
        if dtype == "f32" and rng.random() < 0.5:       # the presets' heads
            H, P, N = rng.choice([(4, 64, 16), (8, 64, 16), (8, 128, 16), (12, 128, 16)])
            G = 1
        else:
            H, P, N = rng.choice([8, 24, 32, 64]), 64, rng.choice([64, 128, 128])
            G = rng.choice([1, 1, 1, 2])
        B = rng.randint(1, 4)
        return {"kind": kind, "dtype": dtype, "B": B, "L": _log_int(rng, 64, 8192 // B), "H": H,
                "P": P, "G": G, "N": N, "state": rng.random() < 0.5}
    if kind == "decode":
        layer = rng.choice(["mamba1", "mamba2", "mamba2"])
        if layer == "mamba1" or rng.random() < 0.5:
            d, H, layers = rng.choice(list(PRESETS.values()))
            N = 16
        else:
            d, H, N, layers = 1024, 32, rng.choice([64, 128]), 6
        return {"kind": kind, "layer": layer, "B": _log_int(rng, 1, 64), "d": d, "H": H, "N": N,
                "layers": layers, "V": rng.choice([1000, 32000])}
    n = rng.choice([32000, 128000, 151665, rng.randint(1000, 40000)])
    return {"kind": kind, "rows": _log_int(rng, 1, 64), "n": n, "topK": rng.choice([1, 20, 50, 200]),
            "topP": rng.choice([0.9, 0.95, 1.0]), "temperature": rng.choice([0.7, 0.8, 1.0])}


# ---------------------------------------------------------------- inputs

class _Gen:
    """Seeded tensors on the GPU (float32)."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, device="cuda", generator=self.g) * std + mean

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, device="cuda", generator=self.g) * (hi - lo) + lo

    def ints(self, hi, *shape):
        return torch.randint(0, hi, shape, device="cuda", generator=self.g)


def _conv_scan_inputs(c, seed):
    g = _Gen(seed)
    B, L, D, N = c["B"], c["L"], c["D"], c["N"]
    t = {"x": g.normal(B, L, D), "w": g.uniform(D, K_CONV, lo=-0.5, hi=0.5),
         "bias": g.uniform(D, lo=-0.5, hi=0.5), "z": g.normal(B, L, D),
         "dt": g.normal(B, L, D, std=0.5, mean=-1.0), "Bm": g.normal(B, L, N),
         "Cm": g.normal(B, L, N), "Dk": g.normal(D, std=0.1, mean=1.0),
         "dt_bias": g.normal(D, std=0.5, mean=-1.0),
         "A": -torch.arange(1, N + 1, device="cuda", dtype=torch.float32).repeat(D, 1)
              * g.uniform(D, 1, lo=0.8, hi=1.2)}
    if c["state"]:
        t["conv_state"] = g.normal(B, D, K_CONV - 1)
        t["h0"] = g.normal(B, D, N, std=0.5)
    return t


def _ssd_inputs(c, seed):
    g = _Gen(seed)
    B, L, H, P, G, N = (c[k] for k in ("B", "L", "H", "P", "G", "N"))
    dt = torch.bfloat16 if c["dtype"] == "bf16" else torch.float32
    std = N ** -0.25          # C . B has unit variance
    t = {"x": g.normal(B, L, H, P).to(dt), "Bm": g.normal(B, L, G, N, std=std).to(dt),
         "Cm": g.normal(B, L, G, N, std=std).to(dt), "dt": g.normal(B, L, H, mean=-3.0),
         "A": -g.uniform(H, lo=1.0, hi=16.0), "Dk": g.normal(H, std=0.1, mean=1.0),
         "dt_bias": g.normal(H, std=0.1)}
    if c["state"]:
        t["h0"] = g.normal(B, H, P, N, std=0.5)
    return t


def _dims(c, layer, V, n_layers):
    H = c.get("H") or next(h for d, h, _ in PRESETS.values() if d == c["d"])
    return checkpoint.ModelDims(vocab=V, d_model=c["d"], n_layers=n_layers, d_state=c["N"],
                                d_conv=K_CONV, expand=2, n_heads=H, n_groups=1,
                                layers=[layer] * n_layers)


def _weights(dims, g):
    """Weights of a trained model's scales (device, fp32): projections keep unit variance, dt in
    [1e-3, 1e-1], S4D-real A (Mamba-1) or A in [1, 16] (Mamba-2)."""
    w = {}
    for name, shape in checkpoint.tensor_specs(dims):
        leaf = name.split(".")[-1]
        if leaf in ("norm", "gnorm", "norm_f", "D"):
            t = g.normal(*shape, std=0.1, mean=1.0)
        elif leaf in ("dt_proj_b", "dt_bias"):
            dt = torch.exp(g.uniform(*shape, lo=math.log(1e-3), hi=math.log(1e-1)))
            t = dt + torch.log(-torch.expm1(-dt))
        elif leaf == "A_log" and len(shape) == 2:
            t = torch.log(torch.arange(1, shape[1] + 1, device="cuda", dtype=torch.float32))
            t = t.repeat(shape[0], 1)
        elif leaf == "A_log":
            t = torch.log(g.uniform(*shape, lo=1.0, hi=16.0))
        elif leaf == "conv_w":
            t = g.uniform(*shape, lo=-0.5, hi=0.5)
        elif leaf == "conv_b":
            t = g.uniform(*shape, lo=-0.5, hi=0.5)
        elif leaf == "dt_proj_w":
            t = g.uniform(*shape, lo=-1.0, hi=1.0) * shape[1] ** -0.5
        elif leaf == "embedding":
            t = g.normal(*shape, std=0.02)
        else:
            t = g.normal(*shape, std=0.02)
        w[name] = t
    return w


def _model_inputs(c, seed):
    """(dims, weights, inputs) of a layer or decode case."""
    g = _Gen(seed)
    if c["kind"] == "decode":
        dims = _dims(c, c["layer"], c["V"], c["layers"])
        w = _weights(dims, g)
        t = {"ids": g.ints(c["V"], c["B"]).to(torch.int32), "ssm": [], "conv": []}
        D, B = dims.d_inner, c["B"]
        for _ in range(c["layers"]):
            if c["layer"] == "mamba1":
                t["ssm"].append(g.normal(B, D, c["N"], std=0.1))
                t["conv"].append(g.normal(B, D, K_CONV - 1, std=0.1))
            else:
                t["ssm"].append(g.normal(B, dims.n_heads, dims.head_dim, c["N"], std=0.1))
                t["conv"].append(g.normal(B, D + 2 * c["N"], K_CONV - 1, std=0.1))
        return dims, w, t
    dims = _dims(c, "mamba1" if c["kind"] == "m1_layer" else "mamba2", 16, 1)
    w = _weights(dims, g)
    return dims, w, {"x": g.normal(c["B"], c["L"], c["d"])}


class _View:
    """A library-owned device buffer as torch sees it."""

    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape),
                                         "typestr": "<f4", "version": 3, "strides": None}


def _state_view(owner, ptr, shape):
    """A tensor over a buffer of owner's state; it keeps owner (whose end frees it) alive."""
    v = torch.as_tensor(_View(ptr, shape), device="cuda")
    v.owner = owner
    return v


class _Loaded:
    """A device, a model with its weights and, for decoding, a state: what a session holds."""

    def __init__(self, dims, weights, batch=0):
        self.device = backend.Device(0)
        cfg = {"vocabSize": dims.vocab, "dModel": dims.d_model, "numLayers": dims.n_layers,
               "dState": dims.d_state, "dConv": dims.d_conv, "expand": dims.expand,
               "nHeads": dims.n_heads, "nGroups": dims.n_groups, "dtRank": dims.dt_rank,
               "normEps": dims.norm_eps, "layers": [{"type": t} for t in dims.layers]}
        self.model = backend.Model(self.device, cfg)
        self.model.load_weights(checkpoint.pack(dims, {k: v.cpu().numpy()
                                                       for k, v in weights.items()}))
        self.state = self.model.new_state(batch) if batch else None

    def __del__(self):
        for part in ("state", "model", "device"):
            if getattr(self, part, None) is not None:
                getattr(self, part).destroy()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "conv_scan":
        t = _conv_scan_inputs(case, seed)
        if case["state"]:
            t["conv_out"] = torch.empty_like(t["conv_state"])
            t["hT"] = torch.empty_like(t["h0"])
        return kind, t
    if kind == "ssd":
        t = _ssd_inputs(case, seed)
        t["hT"] = torch.empty(case["B"], case["H"], case["P"], case["N"], device="cuda")
        return kind, t
    if kind == "sample":
        g = _Gen(seed)
        return kind, {"logits": g.normal(case["rows"], case["n"], std=2.0),
                      "u": torch.rand(case["rows"], device="cuda", generator=g.g,
                                      dtype=torch.float64), "case": dict(case)}
    dims, w, t = _model_inputs(case, seed)
    if kind == "decode":
        B = case["B"]
        m = _Loaded(dims, w, B)
        ssm, conv = [], []
        for i in range(dims.n_layers):
            for ptr, src, views in zip(m.state.layer_ptrs(i), (t["ssm"][i], t["conv"][i]),
                                       (ssm, conv)):
                v = _state_view(m, ptr, src.shape)
                v.copy_(src)
                views.append(v)
        out = {"logits": torch.empty(B, dims.vocab, device="cuda"),
               "picks": torch.empty(B, device="cuda", dtype=torch.int32)}
        return kind, {"m": m, "ids": t["ids"], "ssm": ssm, "conv": conv, **out}
    m = _Loaded(dims, w)
    return kind, {"m": m, "x": t["x"], "y": torch.empty_like(t["x"]),
                  "entry": "ssm_mixer_forward_device" +
                           ("_bf16" if case.get("dtype") == "bf16" else "")}


def run(state):
    kind, t = state
    if kind == "conv_scan":
        u = kernels.causal_conv1d(t["x"], t["w"], t["bias"], state_in=t.get("conv_state"),
                                  state_out=t.get("conv_out"))
        y = kernels.selective_scan(u, t["dt"], t["A"], t["Bm"], t["Cm"], t["Dk"], t["z"],
                                   t["dt_bias"], h0=t.get("h0"), hT=t.get("hT"))
        return {"u": u, "y": y, "conv_state": t.get("conv_out"), "hT": t.get("hT")}
    if kind == "ssd":
        y = kernels.ssd_chunk_scan(t["x"], t["dt"], t["A"], t["Bm"], t["Cm"], t["Dk"],
                                   t["dt_bias"], h0=t.get("h0"), hT=t["hT"])
        return {"y": y, "hT": t["hT"]}
    if kind == "sample":
        c = t["case"]
        return kernels.sample(t["logits"], t["u"], c["temperature"], c["topK"], c["topP"])
    m = t["m"]
    if kind == "decode":
        _lib.call("ssm_decode_step_device", m.model.handle, m.state._h, t["ids"].data_ptr(),
                  t["logits"].data_ptr(), t["picks"].data_ptr())
        return {"logits": t["logits"], "ssm": t["ssm"], "conv": t["conv"]}
    B, L, _ = t["x"].shape
    _lib.call(t["entry"], m.model.handle, 0, t["x"].data_ptr(), t["y"].data_ptr(), B, L)
    return t["y"]


# ---------------------------------------------------------------- counts and bounds

def _ssd_flops(T, H, P, G, N):
    """The SSD's contractions in chunks of 64 steps, causal halves only."""
    q = min(T, 64)
    return T * (q * N * G + H * (q * P + 4.0 * P * N))


def _layer_work(kind, c, layer, T, esz_w):
    d, N = c["d"], c["N"]
    D = 2 * d
    if layer == "mamba1":
        R = -(-d // 16)
        nw = 2 * D * d + (R + 2 * N) * D + D * R + d * D + D * (N + K_CONV + 3)
        mm = 2.0 * T * (2 * D * d + (R + 2 * N) * D + D * R + d * D)
        return esz_w * nw, mm + T * D * (2.0 * K_CONV + 7.0 * N)
    H = c["H"]
    nin = 2 * D + 2 * N + H
    nw = nin * d + d * D + (D + 2 * N) * (K_CONV + 1) + D + 3 * H
    mm = 2.0 * T * (nin * d + d * D)
    core = 5.0 * T * D * N if kind == "decode" else _ssd_flops(T, H, D // H, 1, N)
    return esz_w * nw, mm + core + 2.0 * T * (D + 2 * N) * K_CONV


def work(case):
    kind = case["kind"]
    if kind == "conv_scan":
        B, L, D, N = case["B"], case["L"], case["D"], case["N"]
        st = 2 * B * D * (N + K_CONV - 1) if case["state"] else 0
        # x, dt, z in; u, y out; B, C; weights
        return {"bytes": 4.0 * (5 * B * L * D + 2 * B * L * N + D * (N + K_CONV + 3) + st),
                "flops": B * L * D * (2.0 * K_CONV + 7.0 * N)}
    if kind == "ssd":
        B, L, H, P, G, N = (case[k] for k in ("B", "L", "H", "P", "G", "N"))
        e = 2 if case["dtype"] == "bf16" else 4
        st = B * H * P * N * (2 if case["state"] else 1)
        return {"bytes": e * B * L * (H * P + 2.0 * G * N) + 4.0 * (B * L * H * (P + 1) + st),
                "flops": B * _ssd_flops(L, H, P, G, N)}
    if kind == "sample":
        return {"bytes": 4.0 * case["rows"] * case["n"], "flops": 3.0 * case["rows"] * case["n"]}
    if kind == "decode":
        B, d, V, N = case["B"], case["d"], case["V"], case["N"]
        wb, fl = _layer_work(kind, case, case["layer"], B, 4)
        D = 2 * d
        st = B * (D * N + (D + (2 * N if case["layer"] == "mamba2" else 0)) * (K_CONV - 1))
        return {"bytes": case["layers"] * (wb + 8.0 * st) + 4.0 * (V * d + B * V),
                "flops": case["layers"] * fl + 2.0 * B * V * d}
    T = case["B"] * case["L"]
    layer = "mamba1" if kind == "m1_layer" else "mamba2"
    wb, fl = _layer_work(kind, case, layer, T, 2 if case.get("dtype") == "bf16" else 4)
    return {"bytes": wb + 8.0 * T * case["d"], "flops": fl}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if case.get("dtype") == "bf16":
        # measured against 64 bits: 0.0018 for the SSD on bf16 inputs (its weights and states
        # are rounded to bf16 as MFMA operands), 0.0045 for the whole layer
        return {"rel": 7e-3 if kind == "ssd" else 1.5e-2}
    # 32-bit sums in another order: up to 1.2e-6 from 64 bits, measured
    return {"rel": 5e-6}


# ---------------------------------------------------------------- the same in 64 bits

def _softplus(v):
    return torch.clamp(v, min=0) + torch.log1p(torch.exp(-v.abs()))


def _silu(v):
    return v / (1 + torch.exp(-v))


def _conv64(x, w, bias, state=None):
    """(silu(conv), last K - 1 inputs) of x (B, L, C)."""
    B, L, C = x.shape
    k = w.shape[1]
    pre = x.new_zeros(B, k - 1, C) if state is None else state.transpose(1, 2)
    xp = torch.cat([pre, x], 1)
    y = bias + sum(w[:, j] * xp[:, j:j + L] for j in range(k))
    return _silu(y), xp[:, L:].transpose(1, 2).contiguous()


def _scan64(u, dt, A, Bm, Cm, Dk, z, h):
    """dt already softplus'd; h (B, D, N) is the entering state."""
    ys = []
    for t in range(u.shape[1]):
        d = dt[:, t, :, None]
        h = torch.exp(d * A) * h + (d * u[:, t, :, None]) * Bm[:, t, None, :]
        ys.append((h * Cm[:, t, None, :]).sum(-1))
    return (torch.stack(ys, 1) + Dk * u) * _silu(z), h


def _ssd64(x, dt, A, Bm, Cm, Dk, S, q=64):
    """x (B, L, H, P), dt (B, L, H) softplus'd, Bm / Cm (B, L, G, N), S (B, H, P, N)."""
    B, L, H, P = x.shape
    rep = H // Bm.shape[2]
    ys = []
    for t0 in range(0, L, q):
        xc, dc = x[:, t0:t0 + q].double().transpose(1, 2), dt[:, t0:t0 + q].transpose(1, 2)
        bc = Bm[:, t0:t0 + q].double().transpose(1, 2).repeat_interleave(rep, 1)
        cc = Cm[:, t0:t0 + q].double().transpose(1, 2).repeat_interleave(rep, 1)
        a = torch.cumsum(dc * A[:, None], -1)                       # (B, H, q)
        n = a.shape[-1]
        low = torch.ones(n, n, device=x.device, dtype=torch.bool).tril()
        decay = torch.exp((a[..., :, None] - a[..., None, :]).masked_fill(~low, -math.inf))
        dx = (dc[..., None] * xc).contiguous()
        m = torch.matmul(cc, bc.transpose(-1, -2).contiguous()) * decay
        y = torch.matmul(m, dx)
        y += torch.exp(a)[..., None] * torch.matmul(cc, S.transpose(-1, -2).contiguous())
        ys.append((y + Dk[:, None, None] * xc).transpose(1, 2))
        keep = torch.exp(a[..., -1:] - a)[..., None] * dx
        S = torch.exp(a[..., -1])[..., None, None] * S \
            + torch.matmul(keep.transpose(-1, -2).contiguous(), bc)
    return torch.cat(ys, 1), S


def _rms64(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _mixer64(dims, layer, w, x, ssm, conv):
    """One mixer over x (B, L, d) in float64 -> (y, ssm state, conv state)."""
    D, N, H = dims.d_inner, dims.d_state, dims.n_heads
    B, L, _ = x.shape
    zx = x @ w["in_proj"].T
    if layer == "mamba1":
        R = dims.dt_rank
        u, conv = _conv64(zx[..., :D], w["conv_w"], w["conv_b"], conv)
        dbl = u @ w["x_proj"].T
        dt = _softplus(dbl[..., :R] @ w["dt_proj_w"].T + w["dt_proj_b"])
        h = x.new_zeros(B, D, N) if ssm is None else ssm
        y, h = _scan64(u, dt, -torch.exp(w["A_log"]), dbl[..., R:R + N], dbl[..., R + N:], w["D"],
                       zx[..., D:], h)
        return y @ w["out_proj"].T, h, conv
    z, dt = zx[..., :D], _softplus(zx[..., 2 * D + 2 * N:] + w["dt_bias"])
    v, conv = _conv64(zx[..., D:2 * D + 2 * N], w["conv_w"], w["conv_b"], conv)
    P = dims.head_dim
    S = x.new_zeros(B, H, P, N) if ssm is None else ssm
    y, S = _ssd64(v[..., :D].reshape(B, L, H, P), dt, -torch.exp(w["A_log"]),
                  v[..., None, D:D + N], v[..., None, D + N:], w["D"], S)
    y = _rms64(y.reshape(B, L, D) * _silu(z), w["gnorm"], dims.norm_eps)
    return y @ w["out_proj"].T, S, conv


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None
    if kind == "conv_scan":
        t = {k: v.double() for k, v in _conv_scan_inputs(case, seed).items()}
        u, cs = _conv64(t["x"], t["w"], t["bias"], t.get("conv_state"))
        h = t.get("h0")
        if h is None:
            h = u.new_zeros(case["B"], case["D"], case["N"])
        y, hT = _scan64(u, _softplus(t["dt"] + t["dt_bias"]), t["A"], t["Bm"], t["Cm"], t["Dk"],
                        t["z"], h)
        keep = case["state"]
        return {"u": u, "y": y, "conv_state": cs if keep else None, "hT": hT if keep else None}
    if kind == "ssd":
        t = _ssd_inputs(case, seed)
        S = t["h0"].double() if case["state"] else torch.zeros(
            case["B"], case["H"], case["P"], case["N"], device="cuda", dtype=torch.float64)
        y, S = _ssd64(t["x"], _softplus(t["dt"].double() + t["dt_bias"].double()),
                      t["A"].double(), t["Bm"], t["Cm"], t["Dk"].double(), S)
        return {"y": y, "hT": S}
    dims, w, t = _model_inputs(case, seed)
    w = {k: v.double() for k, v in w.items()}

    def of(i):
        p = f"layers.{i}."
        return {k[len(p):]: v for k, v in w.items() if k.startswith(p)}

    if kind == "decode":
        x = w["embedding"][t["ids"].long()][:, None]
        ssm, conv = [], []
        for i, layer in enumerate(dims.layers):
            wi = of(i)
            y, s, c = _mixer64(dims, layer, wi, _rms64(x, wi["norm"], dims.norm_eps),
                               t["ssm"][i].double(), t["conv"][i].double())
            x = x + y
            ssm.append(s)
            conv.append(c)
        logits = _rms64(x[:, 0], w["norm_f"], dims.norm_eps) @ w["embedding"].T
        return {"logits": logits, "ssm": ssm, "conv": conv}
    return _mixer64(dims, dims.layers[0], of(0), t["x"].double(), None, None)[0]
