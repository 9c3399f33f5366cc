"""The work a user of this framework has it do, as measurable cases.

Each case is one call (or one chain, or one whole model pass) through the
public entry points of neuroflow_amd.quant and neuroflow_amd.runtime:

  rows     quant.linear_forward: the static per-tensor layer on one row or a
           few (the published INT8 benchmark's form: one activation row
           against an out x in weight with zero points on both sides)
  static   quant.Layer.forward_per_tensor: the calibrated (per-tensor) layer
           of an IR on a whole activation, asymmetric weights and activations
  token    quant.Int8Linear / Fp8Linear (and the FNO form with a residual):
           the dynamic per-token layer, the path of the local-linear stacks,
           the token mixer projections and the operator networks' layers
  mlp      quant.mlp_forward_per_token: a chain of per-token layers
  codec    quant.fp8_e4m3_*: the E4M3 codec over whole tensors
  fno1d    runtime.InferenceRuntime.run_device over an FNO1d model
  fno2d    the same over an FNO2d model

Inputs are synthetic: seeded random activations of the shape each path sees.
"""
from __future__ import annotations

import math
import os
import tempfile

import numpy as np
import torch

from neuroflow_amd import ir as IR
from neuroflow_amd import quant as Q
from neuroflow_amd import runtime as RT

DEV = "cuda"


# ---- the cases ---------------------------------------------------------------

def listed():
    return [
        # The smallest call: one row through a square static layer, the
        # published benchmark's 1024 x 1024 GEMV. Latency and launches count.
        dict(name="int8_gemv_1024", kind="rows", M=1, K=1024, N=1024),
        # A calibrated layer of an exported model on a whole activation
        # (512 -> 2048, one of the published layer shapes, batched).
        dict(name="int8_static_512x2048", kind="static", M=8192, K=512, N=2048),
        # FNO1d local-linear layer at its serving size: 256 x 1024 points, width 64.
        dict(name="int8_fno1d_layer", kind="token", fmt="int8", M=262144, K=64, N=64, act="gelu", residual=False),
        # FNO2d local-linear layer in FP8: 16 x 256 x 256 points, width 64. The largest activation.
        dict(name="fp8_fno2d_layer", kind="token", fmt="fp8", M=1048576, K=64, N=64, act="gelu", residual=False),
        # Token mixer qkv projection, 8 x 4096 tokens, d = 256, in both formats.
        dict(name="int8_qkv", kind="token", fmt="int8", M=32768, K=256, N=768, act="none", residual=False),
        dict(name="fp8_qkv", kind="token", fmt="fp8", M=32768, K=256, N=768, act="none", residual=False),
        # Operator network branch layer on 4096 samples, FP8 weights.
        dict(name="fp8_branch", kind="token", fmt="fp8", M=4096, K=1024, N=1024, act="relu", residual=False),
        # A ragged layer: 101 sensors into 128 features, an odd row count.
        dict(name="fp8_ragged", kind="token", fmt="fp8", M=20011, K=101, N=128, act="gelu", residual=False),
        # Operator network trunk: 65536 query points through 3 x 1024 hidden layers and a 256-wide head.
        dict(name="int8_trunk_mlp", kind="mlp", M=65536, K=1024, hidden=3, N=256),
        # Encoding a tensor of ragged size to E4M3 bytes and decoding it again.
        dict(name="fp8_codec", kind="codec", op="round_trip", n=16777219),
        # A whole FNO1d model at its serving size with INT8 local-linear layers.
        dict(name="fno1d_model", kind="fno1d", batch=256, n=1024, width=64, modes=16, layers=4, quant="tensor"),
        # A whole FNO2d model of half that width on a 128 x 128 grid, FP8 activations.
        dict(name="fno2d_model", kind="fno2d", batch=16, n=128, width=32, modes=12, layers=4, quant="fp8"),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _feature(rng, lo, hi, steps=(1, 4, 64, 64)):
    """A layer width: mostly a multiple of 64 or 4, sometimes any number."""
    v = _logint(rng, lo, hi)
    step = rng.choice(steps)
    return max(lo, v // step * step)


def draw(rng):
    kind = rng.choice(["rows", "static", "token", "token", "token", "mlp", "codec", "fno1d", "fno2d"])
    if kind == "rows":
        return dict(kind=kind, M=rng.choice([1, 1, 2, rng.randint(3, 32)]), K=_feature(rng, 64, 4096, (64,)),
                    N=_feature(rng, 64, 2048))
    if kind == "static":
        K, N = _feature(rng, 32, 1024), _feature(rng, 32, 2048)
        return dict(kind=kind, M=_logint(rng, 64, min(262144, 2 ** 34 // (K * N), 2 ** 26 // max(K, N))), K=K, N=N)
    if kind == "token":
        # The INT8 row form drops a tail of K % 64 features (the reference's
        # vectorised loop), so INT8 layers in earnest have K a multiple of 64.
        fmt = rng.choice(["int8", "fp8"])
        K = _feature(rng, 64, 1024, (64,)) if fmt == "int8" else _feature(rng, 32, 1024)
        N = _feature(rng, 32, 1024)
        residual = rng.random() < 0.25
        if residual:
            N = K
        ops = 2 ** 35 if fmt == "int8" else 2 ** 33
        M = _logint(rng, 64, min(524288, ops // (K * N), 2 ** 25 // max(K, N)))
        return dict(kind=kind, fmt=fmt, M=M, K=K, N=N, act=rng.choice(["none", "relu", "gelu"]), residual=residual)
    if kind == "mlp":
        return dict(kind=kind, M=_logint(rng, 256, 32768), K=rng.choice([256, 512, 1024]), hidden=rng.randint(1, 3),
                    N=rng.choice([64, 128, 200, 256]))
    if kind == "codec":
        return dict(kind=kind, op=rng.choice(["round_trip", "fake_quant"]), n=_logint(rng, 1000, 16777216))
    if kind == "fno1d":
        n = 2 ** rng.randint(6, 11)
        width = rng.choice([16, 20, 32, 48, 64])
        return dict(kind=kind, batch=_logint(rng, 1, min(256, 2 ** 24 // (n * width))), n=n, width=width,
                    modes=rng.randint(4, min(24, n // 2)), layers=rng.randint(2, 4),
                    quant=rng.choice(["none", "tensor", "tensor", "fp8"]))
    n = 2 ** rng.randint(5, 8)
    width = rng.choice([16, 20, 32, 48, 64])
    return dict(kind=kind, batch=_logint(rng, 1, min(32, 2 ** 24 // (n * n * width))), n=n, width=width,
                modes=rng.randint(4, 14), layers=rng.randint(2, 4), quant=rng.choice(["none", "tensor", "fp8"]))


# ---- inputs ------------------------------------------------------------------

def _rng(case, seed):
    key = [seed] + [v for v in (case.get(k) for k in ("M", "K", "N", "n", "batch", "width", "modes")) if v]
    return np.random.default_rng(key)


def _gen(rng):
    return torch.Generator(device=DEV).manual_seed(int(rng.integers(1 << 62)))


def _linear(rng, n_out, n_in):
    """nn.Linear's default initialisation."""
    b = 1.0 / math.sqrt(n_in)
    return (rng.uniform(-b, b, (n_out, n_in)).astype(np.float32), rng.uniform(-b, b, n_out).astype(np.float32))


def _activations(case, rng):
    """N(0, 1), 1% of the entries 20 times larger in FP8 (the outliers that
    format is chosen for); a ReLU layer's output for an MLP."""
    M, K = case["M"], case["K"]
    g = _gen(rng)
    x = torch.randn(M, K, device=DEV, generator=g)
    if case.get("fmt") == "fp8":
        x = torch.where(torch.rand(M, K, device=DEV, generator=g) < 0.01, x * 20.0, x)
    if case["kind"] == "mlp":
        x = torch.relu(x)
    return x.contiguous()


def _static_layer(case, rng):
    """Asymmetric per-channel weights and a per-tensor activation scale with
    a zero point, as min/max calibration gives them."""
    K, N = case["K"], case["N"]
    W, b = _linear(rng, N, K)
    lo, hi = np.minimum(W.min(1), 0), np.maximum(W.max(1), 0)
    scale = ((hi - lo) / 255.0).astype(np.float32)
    zp = (-128 - np.round(lo / scale)).astype(np.int32)
    Wq = np.clip(np.round(W / scale[:, None]) + zp[:, None], -128, 127).astype(np.int8)
    return Wq, scale, zp, b, np.float32(9.0 / 255.0), 3


def _weights_of(case, rng):
    if case["kind"] == "mlp":
        dims = [case["K"]] + [case["K"]] * case["hidden"] + [case["N"]]
        return [_linear(rng, o, i) for i, o in zip(dims[:-1], dims[1:])]
    return [_linear(rng, case["N"], case["K"])]


# ---- the FNO models ----------------------------------------------------------

def _fno_weights(case, rng):
    w, m, L = case["width"], case["modes"], case["layers"]
    shape = (w, w, m) if case["kind"] == "fno1d" else (w, w, m, m)
    out = {"lift.weight": rng.uniform(-1, 1, (w, 1)), "lift.bias": rng.uniform(-1, 1, w)}
    for i in range(L):
        # Spectral weights large enough that both branches carry the signal.
        out[f"specs.{i}.weights_real"] = rng.standard_normal(shape) / w
        out[f"specs.{i}.weights_imag"] = rng.standard_normal(shape) / w
        out[f"locs.{i}.weight"], out[f"locs.{i}.bias"] = _linear(rng, w, w)
    out["proj_q.weight"], out["proj_q.bias"] = _linear(rng, w, w)
    out["proj_out.weight"], out["proj_out.bias"] = _linear(rng, 1, w)
    return {k: np.asarray(v, np.float32) for k, v in out.items()}


def _fno_input(case, rng):
    """Sums of eight sinusoids on the unit grid, one field per sample."""
    b, n = case["batch"], case["n"]
    t = torch.arange(n, device=DEV, dtype=torch.float64) / n * 2.0 * math.pi

    def col(v):
        return torch.from_numpy(np.asarray(v, np.float64)).to(DEV)

    amp, kx, ky, ph = (col(rng.uniform(0, 1, (8, b, 1))), col(rng.integers(1, 9, (8, b, 1))),
                       col(rng.integers(1, 9, (8, b, 1))), col(rng.uniform(0, 2 * math.pi, (8, b, 1))))
    if case["kind"] == "fno1d":
        x = sum(amp[j] * torch.sin(kx[j] * t + ph[j]) for j in range(8))
    else:
        x = sum(amp[j][..., None] * torch.sin((kx[j] * t)[:, :, None] + (ky[j] * t)[:, None, :] + ph[j][..., None])
                for j in range(8))
    return x.unsqueeze(-1).float().contiguous()


def _gelu64(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _fake_quant64(v, scale, zp=0):
    t = v / scale
    q = torch.sign(t) * torch.floor(t.abs() + 0.5) + zp
    return (q.clamp(-128, 127) - zp) * scale


def _log2_snap64(v, scale):
    """The runtime's FP8 activation snap: powers of two above 2^-6 of the scale."""
    t = v / scale
    a = t.abs()
    r = torch.log2(a.clamp_min(1e-30)) * 8.0
    e = torch.trunc(torch.sign(r) * torch.floor(r.abs() + 0.5) / 8.0)
    return torch.where(t < 0, -1.0, 1.0) * torch.where(a < 2.0 ** -6, a, torch.exp2(e).clamp_max(448.0)) * scale


def _fno_forward64(case, weights, x, qparams=None, record=None):
    """The model in float64. qparams: name -> scale of the activation
    quantisation (none while calibrating); record collects each absmax."""
    two_d = case["kind"] == "fno2d"
    m, n, w = case["modes"], case["n"], case["width"]
    dims = (1, 2) if two_d else (1,)
    W = {k: torch.from_numpy(v).to(DEV, torch.float64) for k, v in weights.items()}
    quant = case["quant"] if qparams else "none"
    if quant == "tensor" and not two_d:
        for k, v in W.items():
            if v.ndim >= 2:
                W[k] = _fake_quant64(v, _channel_scale(weights[k]).to(DEV, torch.float64))

    def fq(v, key):
        if record is not None:
            record[key] = float(v.abs().max())
        if quant == "none" or key not in qparams:
            return v
        return _fake_quant64(v, qparams[key]) if quant == "tensor" else _log2_snap64(v, qparams[key])

    h = x.double() @ W["lift.weight"].T + W["lift.bias"]
    # FNO1d quantises each layer's input per tensor (the FP8 record applies to
    # the local branch alone); FNO2d quantises where the value is produced.
    h_q = fq(h, "lift.output") if two_d or quant != "fp8" else h
    h = h_q
    for i in range(case["layers"]):
        wc = torch.complex(W[f"specs.{i}.weights_real"], W[f"specs.{i}.weights_imag"])
        if two_d:
            mh, mw = min(m, n), min(m, n // 2 + 1)
            spec = torch.fft.rfft2(h, dim=dims)
            full = torch.zeros_like(spec)
            full[:, :mh, :mw] = torch.einsum("bxyi,ioxy->bxyo", spec[:, :mh, :mw], wc[:, :, :mh, :mw])
            x1 = torch.fft.irfft2(full, s=(n, n), dim=dims)
        else:
            mm = min(m, n // 2 + 1)
            spec = torch.fft.rfft(h, dim=1)
            full = torch.zeros_like(spec)
            full[:, :mm] = torch.einsum("bmi,iom->bmo", spec[:, :mm], wc[:, :, :mm])
            x1 = torch.fft.irfft(full, n=n, dim=1)
        x2 = fq(h @ W[f"locs.{i}.weight"].T + W[f"locs.{i}.bias"], f"locs.{i}.output")
        h = _gelu64(x1 + x2)
        if not two_d and quant == "tensor" and i + 1 < case["layers"]:
            h = _fake_quant64(h, qparams[f"locs.{i}.output"])
    q = h @ W["proj_q.weight"].T + W["proj_q.bias"]
    if two_d:
        q = fq(q, "proj_q.output")
    return (_gelu64(q) @ W["proj_out.weight"].T + W["proj_out.bias"])


def _channel_scale(t):
    """Symmetric per-channel scale: axis 0 of a matrix, axis 1 of a spectral weight."""
    ax = (1,) if t.ndim == 2 else (0,) + tuple(range(2, t.ndim))
    s = np.abs(t).max(axis=ax, keepdims=True).astype(np.float32) / np.float32(127.0)
    return torch.from_numpy(s)


def _fno_model(case, seed):
    rng = _rng(case, seed)
    weights, x = _fno_weights(case, rng), _fno_input(case, rng)
    records, qparams = None, None
    if case["quant"] != "none":
        amax = {}
        _fno_forward64(case, weights, x[:2], record=amax)
        qmax = 127.0 if case["quant"] == "tensor" else 448.0
        qparams = {k: float(np.float32(a) / np.float32(qmax)) for k, a in amax.items()}
        records = []
        if case["quant"] == "tensor" and case["kind"] == "fno1d":
            for k, t in weights.items():
                if t.ndim >= 2:
                    s = _channel_scale(t).numpy().reshape(-1)
                    records.append((1, k, s, np.zeros(s.size, np.int32), 0 if t.ndim == 2 else 1))
        for k, s in qparams.items():
            records.append((0, k, s, 0) if case["quant"] == "tensor" else (3, k, s))
    return weights, x, records, qparams


def _fno_runtime(case, weights, records):
    w, m, L = case["width"], case["modes"], case["layers"]
    one_d = case["kind"] == "fno1d"
    data = IR.write_binary(1 if one_d else 2, [1, 1, w, m, L, 1, 0] if one_d else [1, 1, w, m, m, L, 1], "gelu",
                           weights, records)
    fd, path = tempfile.mkstemp(suffix=".nneuroir")
    try:
        with os.fdopen(fd, "wb") as f:
            f.write(data)
        rt = RT.load().InferenceRuntime(path)
    finally:
        os.unlink(path)
    if one_d and case["quant"] == "tensor":
        rt.enable_int8_gemm()
    return rt


# ---- prepare, run ------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("fno1d", "fno2d"):
        weights, x, records, _ = _fno_model(case, seed)
        return dict(kind=kind, rt=_fno_runtime(case, weights, records), x=x, y=torch.empty_like(x),
                    shape=list(x.shape))
    rng = _rng(case, seed)
    if kind == "codec":
        x = torch.randn(case["n"], device=DEV, generator=_gen(rng)) * 3.0
        return dict(kind=kind, op=case["op"], x=x, scale=float(np.float32(4.5 * 3.0 / 448.0)))
    if kind in ("rows", "static"):
        Wq, scale, zp, b, scale_A, zp_A = _static_layer(case, rng)
        x = _activations(case, rng)
        if kind == "static":
            sum_w = Wq.sum(1, dtype=np.int32) - case["K"] * zp
            return dict(kind=kind, layer=Q.Layer.from_int8_blob(Wq, scale, zp, b, sum_w), x=x,
                        scale_A=float(scale_A), zp_A=zp_A)
        to = lambda a: torch.from_numpy(a).to(DEV)
        p = Q.Int8LinearParams(to(Wq), to(scale), to(zp), to(b), float(scale_A), zp_A)
        return dict(kind=kind, params=p, x=x[0].contiguous() if case["M"] == 1 else x)
    weights = _weights_of(case, rng)
    x = _activations(case, rng)
    if kind == "mlp":
        return dict(kind=kind, x=x, layers=[Q.Int8Linear(W, b, device=DEV).token_params for W, b in weights],
                    acts=["relu"] * case["hidden"] + ["none"])
    cls = Q.Fp8Linear if case["fmt"] == "fp8" else Q.Int8Linear
    state = dict(kind=kind, fmt=case["fmt"], layer=cls(*weights[0], device=DEV), x=x, act=case["act"], x1=None)
    if case["residual"]:
        state["x1"] = torch.randn(case["M"], case["N"], device=DEV, generator=_gen(rng))
    return state


def run(state):
    kind = state["kind"]
    if kind == "rows":
        return Q.linear_forward(state["params"], state["x"])
    if kind == "static":
        return state["layer"].forward_per_tensor(state["x"], state["scale_A"], state["zp_A"])
    if kind == "token":
        if state["x1"] is None:
            return state["layer"](state["x"], state["act"])
        if state["fmt"] == "fp8":
            return Q.fp8_fno_layer_per_token(state["layer"].params, state["x"], state["x1"], state["act"])
        return Q.fno_layer_per_token(state["layer"].token_params, state["x"], state["x1"], state["act"])
    if kind == "mlp":
        return Q.mlp_forward_per_token(state["layers"], state["x"], state["acts"])
    if kind == "codec":
        if state["op"] == "fake_quant":
            return Q.fp8_e4m3_fake_quant(state["x"], state["scale"])
        bits = Q.fp8_e4m3_to_bits(state["x"])
        return bits, Q.fp8_e4m3_from_bits(bits)
    state["rt"].run_device(state["x"].data_ptr(), state["shape"], state["y"].data_ptr(), state["shape"],
                           torch.cuda.current_stream().cuda_stream)
    return state["y"]


# ---- what a pass cannot do without ----------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "codec":
        n = case["n"]
        return dict(bytes=8 * n if case["op"] == "fake_quant" else 10 * n, flops=n)
    if kind in ("fno1d", "fno2d"):
        w, m, L, n, b = case["width"], case["modes"], case["layers"], case["n"], case["batch"]
        two_d = kind == "fno2d"
        pts = n * n if two_d else n
        bins = m * m if two_d else m
        fft = 2.5 * pts * math.log2(pts)
        flops = b * (2 * pts * w + L * (w * 2 * fft + 8 * bins * w * w + 2 * pts * w * w) + 2 * pts * w * w + 2 * pts * w)
        return dict(bytes=8 * b * pts + 4 * L * (2 * bins + 1) * w * w + 4 * w * w, flops=flops)
    M, K, N = case["M"], case["K"], case["N"]
    if kind == "mlp":
        L = case["hidden"]
        return dict(bytes=4 * M * K + L * K * K + N * K + 4 * M * N, flops=2 * M * (L * K * K + N * K))
    bytes_ = 4 * M * K + N * K + 12 * N + 4 * M * N * (2 if case.get("residual") else 1)
    return dict(bytes=bytes_, flops=2 * M * N * K)


# ---- what the outputs should be ---------------------------------------------------

def tolerance(case):
    kind = case["kind"]
    if kind == "codec" or kind in ("rows", "static"):
        return "exact"
    if kind == "mlp" or (kind == "token" and case["fmt"] == "int8" and case["act"] != "gelu"):
        return "exact"
    # About four times what the path measured against exact().
    if kind == "token":
        return {"rel": 3e-7}
    # A rounding difference moves a quantised activation by a whole step (a
    # factor of two in the FP8 snap) and travels through the later layers.
    return {"rel": {"none": 1.2e-6, "tensor": 5e-3, "fp8": 1.2e-2}[case["quant"]]}


def _codes64(x, scale, zp=0):
    """clamp(round_half_away(fl32(x / scale)) + zp): the float32 quotient
    rounded from the float64 one (exact: 53 bits hold it)."""
    t = (x.double() / scale).float().double()
    return (torch.sign(t) * torch.floor(t.abs() + 0.5) + zp).clamp(-128, 127)


def _e4m3_value64(v):
    """The E4M3 value of a float32 in [-448, 448]: three mantissa bits, ties
    to even; multiples of 2^-9 up to 7 below 2^-6."""
    v = v.double()
    a = v.abs()
    step = torch.exp2(torch.floor(torch.log2(a.clamp_min(2.0 ** -20))) - 3.0)
    r = torch.where(a < 2.0 ** -6, torch.round(a * 512.0).clamp_max(7.0) / 512.0, torch.round(a / step) * step)
    return torch.sign(v) * r.clamp_max(448.0)


def _fp8_values64(x, scale):
    inv = (1.0 / scale.double()).float().double()
    return _e4m3_value64((x.double() * inv).float().clamp(-448.0, 448.0))


def _scales(x, qmax):
    s = (x.abs().amax(1, keepdim=True).double() / qmax).float()
    return torch.where(s > 0, s, torch.ones_like(s))


def _token_layer64(fmt, x, W, b):
    Wt, bt = torch.from_numpy(W).to(DEV), torch.from_numpy(b).to(DEV, torch.float64)
    qmax, q = (448.0, _fp8_values64) if fmt == "fp8" else (127.0, lambda v, s: _codes64(v, s.double()))
    sw, sx = _scales(Wt, qmax), _scales(x, qmax)
    return (q(x, sx) @ q(Wt, sw).T) * sx.double() * sw.double().T + bt


def exact(case, seed):
    kind = case["kind"]
    if kind in ("fno1d", "fno2d"):
        weights, x, _, qparams = _fno_model(case, seed)
        return _fno_forward64(case, weights, x, qparams=qparams)
    rng = _rng(case, seed)
    if kind == "codec":
        x = torch.randn(case["n"], device=DEV, generator=_gen(rng)) * 3.0
        if case["op"] == "fake_quant":
            scale = torch.tensor(np.float32(4.5 * 3.0 / 448.0), device=DEV)
            return _fp8_values64(x, scale) * scale.double()
        return None, _e4m3_value64(x)
    if kind in ("rows", "static"):
        Wq, scale, zp, b, scale_A, zp_A = _static_layer(case, rng)
        x = _activations(case, rng)
        q = _codes64(x, float(scale_A), zp_A)
        W64, zpw = torch.from_numpy(Wq).to(DEV, torch.float64), torch.from_numpy(zp).to(DEV, torch.float64)
        K = case["K"]
        sum_q, sum_w = q.sum(1, keepdim=True), W64.sum(1)
        # The two forms' integer terms, as the reference writes them.
        zp_terms = -zp_A * (sum_w - K * zpw) if kind == "static" else -2 * zp_A * sum_w + 3 * K * zp_A * zpw
        t = q @ W64.T + zp_terms - 2 * zpw * sum_q + K * zpw * zp_A
        y = t * float(scale_A) * torch.from_numpy(scale).to(DEV, torch.float64) + torch.from_numpy(b).to(DEV).double()
        return y[0] if kind == "rows" and case["M"] == 1 else y
    weights = _weights_of(case, rng)
    x = _activations(case, rng)
    if kind == "mlp":
        for W, b in weights[:-1]:
            x = torch.relu(_token_layer64("int8", x, W, b)).float()
        return _token_layer64("int8", x, *weights[-1])
    y = _token_layer64(case["fmt"], x, *weights[0])
    if case["residual"]:
        y = y + torch.randn(case["M"], case["N"], device=DEV, generator=_gen(rng)).double()
    return torch.relu(y) if case["act"] == "relu" else _gelu64(y) if case["act"] == "gelu" else y
