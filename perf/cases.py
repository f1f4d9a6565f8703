"""The work that the framework's speed is measured on.

The framework serves one path: the fp16 inference forward of a stacked `nn.LSTM` with a `Linear`
head, through `convert_regressor_module` (a forecaster: all rows of equal length, or ragged rows),
`PersistentLSTM` (the `nn.LSTM` drop-in that returns the output sequence and the states) and
`input_projection` (the GEMM over all time steps that a caller may run by itself).  There is no
backward pass and one compute type (fp16 with fp32 accumulation).

A model's weights are prepared once (a user's program keeps the converted module); every pass takes its
batch from a loader, so the batch is a tensor object the model has not been called with before.
"""
from __future__ import annotations

import math

import torch
import torch.nn as nn

from persistent_lstm_hip_amd import convert_regressor_module
from persistent_lstm_hip_amd.extension import require_extension
from persistent_lstm_hip_amd.model import PersistentLSTM

DEVICE = "cuda"


def _case(kind, **kw):
    return dict(kind=kind, **kw)


def listed():
    return [
        # One series of a live forecaster: the smallest call, all latency (the README's model, batch 1).
        _case("regressor", name="online_one_series", I=5, H=128, L=4, O=24, B=1, T=64),
        # The benchmark's smallest configuration: one layer, a handful of series.
        _case("regressor", name="one_layer_b8", I=5, H=128, L=1, O=24, B=8, T=64),
        # A small model over a year of daily values, nothing a multiple of a tile.
        _case("regressor", name="daily_h60", I=7, H=60, L=3, O=7, B=200, T=365),
        # The headline configuration: 4 layers, hidden 128, batch 512, 1000 steps.
        _case("regressor", name="headline_h128", I=5, H=128, L=4, O=24, B=512, T=1000),
        # The same with rows of unequal lengths (packed-sequence semantics).
        _case("ragged", name="ragged_h128", I=5, H=128, L=4, O=24, B=512, T=1000, lo=200),
        # Batch scoring of more series than one launch holds.
        _case("regressor", name="batch_1500_h128", I=5, H=128, L=4, O=24, B=1500, T=250),
        # The wider configurations of the benchmark's sweep.
        _case("regressor", name="sweep_h256", I=5, H=256, L=4, O=24, B=512, T=1000),
        _case("regressor", name="sweep_h512", I=5, H=512, L=4, O=24, B=512, T=1000),
        # The largest hidden size served, at the sweep's batch and length: the largest call.
        _case("regressor", name="largest_h1024", I=5, H=1024, L=4, O=24, B=512, T=1000),
        # nn.LSTM drop-in inside a larger model: initial states in, output sequence and states out.
        _case("lstm", name="features_h400", I=40, H=400, L=2, B=40, T=128),
        # The drop-in over wide embeddings (input wider than the hidden size).
        _case("lstm", name="embeddings_i300", I=300, H=128, L=2, B=64, T=200),
        # The input projection of all steps at once, at the headline's sizes.
        _case("projection", name="projection_k128", rows=512000, K=128, N=512),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case: hidden 16..1024, batch 1..1500 (up to 512 above hidden 512), 8..1000 steps, 1..4
    layers, mostly narrow inputs; a few projections."""
    pick = rng.random()
    if pick < 0.07:
        return _case("projection", rows=16 * _log_int(rng, 64, 32000), K=128 * rng.randint(1, 8), N=512 * rng.randint(1, 4))
    H = _log_int(rng, 16, 1024)
    B = _log_int(rng, 1, 1500 if H <= 512 else 512)
    T = _log_int(rng, 8, 1000)
    L = rng.randint(1, 4)
    I = _log_int(rng, 1, 64) if rng.random() < 0.85 else rng.randint(65, 400)
    if pick < 0.25:
        return _case("lstm", I=I, H=H, L=L, B=B, T=T)
    if pick < 0.42:
        return _case("ragged", I=I, H=H, L=L, O=rng.randint(1, 48), B=B, T=T, lo=max(1, T // 5))
    return _case("regressor", I=I, H=H, L=L, O=rng.randint(1, 48), B=B, T=T)


class _Regressor(nn.Module):
    """A user's native model: `.lstm` and `.linear`."""

    def __init__(self, I, H, L, O):
        super().__init__()
        self.lstm = nn.LSTM(I, H, L, batch_first=True)
        self.linear = nn.Linear(H, O)


def _native(case, seed):
    """PyTorch's default initialisation from the seed."""
    with torch.random.fork_rng(devices=[]):
        torch.manual_seed(seed)
        return _Regressor(case["I"], case["H"], case["L"], case.get("O", 1)).eval()


def _inputs(case, seed):
    """The tensors of one pass, on the GPU (lengths: on the host, as a data loader gives them)."""
    g = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    if case["kind"] == "projection":
        x = torch.randn(case["rows"], case["K"], device=DEVICE, generator=g).half()
        w = (torch.randn(case["N"], case["K"], device=DEVICE, generator=g) / math.sqrt(case["K"])).half()
        return {"x": x, "w": w}
    B, T, I, L, H = (case[k] for k in ("B", "T", "I", "L", "H"))
    d = {"x": torch.randn(B, T, I, device=DEVICE, generator=g).half()}
    if case["kind"] == "ragged":
        gl = torch.Generator().manual_seed(seed + 2)
        d["lengths"] = torch.sort(torch.randint(case["lo"], T + 1, (B,), generator=gl), descending=True).values
    if case["kind"] == "lstm":
        d["h0"] = torch.tanh(torch.randn(L, B, H, device=DEVICE, generator=g)).half()
        d["c0"] = torch.randn(L, B, H, device=DEVICE, generator=g).half()
    return d


def prepare(case, seed):
    d = _inputs(case, seed)
    if case["kind"] == "projection":
        ext = require_extension()
        out = torch.empty(case["rows"], case["N"], device=DEVICE, dtype=torch.float16)
        return dict(case=case, x=ext.to_blocked(d["x"]), w=d["w"], out=out)
    native = _native(case, seed)
    if case["kind"] == "lstm":
        model = PersistentLSTM.from_native_module(native.lstm)
    else:
        model = convert_regressor_module(native)
    model = model.to(DEVICE).half().eval()
    return dict(case=case, model=model, loader=[d["x"]], lengths=d.get("lengths"),
                hx=(d["h0"], d["c0"]) if case["kind"] == "lstm" else None)


def run(state):
    kind = state["case"]["kind"]
    if kind == "projection":
        return require_extension().input_projection(state["x"], state["w"], state["out"], blocked=True)
    x = state["loader"][0].detach()  # the loader's next batch: another tensor object each time
    with torch.no_grad():
        if kind == "ragged":
            return state["model"].forward_ragged(x, state["lengths"])
        if kind == "lstm":
            out, (h_n, c_n) = state["model"](x, state["hx"])
            return [out, h_n, c_n]
        return state["model"](x)


def work(case):
    if case["kind"] == "projection":
        M, K, N = case["rows"], case["K"], case["N"]
        return {"bytes": 2.0 * (M * K + N * K + M * N), "flops": 2.0 * M * N * K}
    I, H, L, B, T = (case[k] for k in ("I", "H", "L", "B", "T"))
    O = case.get("O", 0)
    steps = B * T if case["kind"] != "ragged" else B * (case["lo"] + T) / 2
    params = 4 * H * (I + H) + (L - 1) * 8 * H * H + 8 * L * H + O * (H + 1)
    nbytes = 2.0 * (steps * I + params)
    if case["kind"] == "lstm":
        nbytes += 2.0 * (steps * H + 4 * L * B * H)
    else:
        nbytes += 2.0 * B * O
    return {"bytes": nbytes, "flops": 2.0 * steps * 4 * H * ((I + H) + (L - 1) * 2 * H) + 2.0 * B * H * O}


def tolerance(case):
    # Each side's distance from the float64 result is 2.0e-4 to 2.8e-4 in every case: the final rounding to
    # fp16 (a projection), or fp16 h at every step and, in wide models, fp16 projections (the states carry
    # the roundings on but do not let them grow).  About four times that.
    return {"rel": 1e-3}


def exact(case, seed):
    """The forward in float64 on the same fp16 weights and inputs."""
    d = _inputs(case, seed)
    if case["kind"] == "projection":
        # out in the blocked layout of `prepare`: [rows / 16][N / 32][4 groups of 8 columns][16 rows][8]
        M, N = case["rows"], case["N"]
        w64 = d["w"].double().t().contiguous()
        parts = [p.double() @ w64 for p in d["x"].split(65536)]
        y = torch.cat(parts)
        return y.reshape(M // 16, 16, N // 32, 4, 8).permute(0, 2, 3, 1, 4).reshape(M, N)
    B, T, I, L, H = (case[k] for k in ("B", "T", "I", "L", "H"))
    native = _native(case, seed).half().to(DEVICE)
    p = {k: v.detach().double() for k, v in native.named_parameters()}
    lengths = d["lengths"].to(DEVICE) if "lengths" in d else None
    h = [torch.zeros(B, H, dtype=torch.float64, device=DEVICE) for _ in range(L)]
    c = [torch.zeros(B, H, dtype=torch.float64, device=DEVICE) for _ in range(L)]
    if "h0" in d:
        h, c = [t.double() for t in d["h0"]], [t.double() for t in d["c0"]]
    wih = [p[f"lstm.weight_ih_l{l}"].t().contiguous() for l in range(L)]
    whh = [p[f"lstm.weight_hh_l{l}"].t().contiguous() for l in range(L)]
    bias = [p[f"lstm.bias_ih_l{l}"] + p[f"lstm.bias_hh_l{l}"] for l in range(L)]
    seq = torch.empty(B, T, H, dtype=torch.float64, device=DEVICE) if case["kind"] == "lstm" else None
    x = d["x"].transpose(0, 1).contiguous()
    for t in range(T):
        inp = x[t].double()
        live = (lengths > t).unsqueeze(1) if lengths is not None else None
        for l in range(L):
            z = torch.addmm(bias[l], inp, wih[l]).addmm_(h[l], whh[l])
            i, f, g, o = z.chunk(4, dim=1)
            cn = torch.sigmoid(f) * c[l] + torch.sigmoid(i) * torch.tanh(g)
            hn = torch.sigmoid(o) * torch.tanh(cn)
            if live is not None:
                cn, hn = torch.where(live, cn, c[l]), torch.where(live, hn, h[l])
            c[l], h[l] = cn, hn
            inp = hn
        if seq is not None:
            seq[:, t] = inp
    if seq is not None:
        return [seq, torch.stack(h), torch.stack(c)]
    return torch.addmm(p["linear.bias"], h[-1], p["linear.weight"].t().contiguous())
