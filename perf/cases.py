"""The work whose speed counts: selective scans, whole layers and whole models, prefill and
decode, over the sizes, types and layouts that programs on this library use.

Kinds of case:

  scan    ``selective_scan`` on row-major (batch, dim, seqlen) tensors: the op a program
          calls by itself.
  layer   ``MambaBlock.prefill`` on (batch, seqlen, d_model), called eagerly.
  step    ``MambaBlock.step`` on one token per sequence, called eagerly and functionally
          (states in, new states out), as a program that drives the layers itself does.
  prompt  ``GraphPrefill`` of a whole model on a (batch, seqlen) prompt: last position's logits and
          the states that decoding goes on from.
  decode  ``MambaModel.step`` of a whole model, its states updated in place, replayed from a HIP
          graph that the program captured once, as serving loops do (and as ``GraphDecoder``
          does, which hands out only ids): logits and states.
"""

from __future__ import annotations

import math

import torch

from mamba_metal_amd import GraphPrefill, MambaBlock, MambaConfig, MambaModel, selective_scan

DEVICE = "cuda:0"
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
VOCAB = 50280


def listed():
    return [
        # A short single sequence on few channels in fp32: one call's latency.
        dict(name="scan_f32_small", kind="scan", dtype="f32", batch=1, dim=16, dstate=16, seqlen=4096,
             flags=True),
        # The scan benchmark of the reference implementation: few channels, long, fp32, y only.
        dict(name="scan_f32_long", kind="scan", dtype="f32", batch=1, dim=16, dstate=16, seqlen=32768,
             flags=False),
        # A batch of sequences at the width of a small model's inner dimension.
        dict(name="scan_f16_batch", kind="scan", dtype="f16", batch=8, dim=1536, dstate=16, seqlen=8192,
             flags=True),
        # The largest: long sequences at the width of a large model.
        dict(name="scan_f16_large", kind="scan", dtype="f16", batch=4, dim=5120, dstate=16, seqlen=32768,
             flags=True),
        # Sizes that no tile divides: an odd length (so odd row strides) and an odd batch.
        dict(name="scan_bf16_odd", kind="scan", dtype="bf16", batch=3, dim=1000, dstate=16, seqlen=3001,
             flags=True),
        # A layer in full precision on an odd length.
        dict(name="layer_f32_odd", kind="layer", dtype="f32", batch=2, d_model=512, seqlen=1021),
        # A large layer prefilling a full serving batch.
        dict(name="layer_f16_batch", kind="layer", dtype="f16", batch=64, d_model=2560, seqlen=512),
        # One layer's decode step called eagerly at a small batch: launches and host time.
        dict(name="step_bf16_small", kind="step", dtype="bf16", batch=5, d_model=768),
        # A whole small model on one long prompt: the latency of the first token.
        dict(name="prompt_f16_single", kind="prompt", dtype="f16", batch=1, d_model=768, n_layer=24,
             seqlen=2048),
        # A few prompts of an odd length through a middle-sized model's layers.
        dict(name="prompt_bf16_odd", kind="prompt", dtype="bf16", batch=3, d_model=1024, n_layer=4,
             seqlen=777),
        # A whole small model decoding one sequence: the latency of a token.
        dict(name="decode_f16_single", kind="decode", dtype="f16", batch=1, d_model=768, n_layer=24),
        # A large model's layers decoding a full serving batch: throughput.
        dict(name="decode_f16_batch", kind="decode", dtype="f16", batch=64, d_model=2560, n_layer=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    dtype = rng.choice(["f32", "f16", "f16", "bf16"])
    kind = rng.choice(["scan", "scan", "scan", "layer", "step", "prompt", "decode", "decode"])
    if kind == "scan":
        while True:
            case = dict(kind=kind, dtype=dtype, batch=_log_int(rng, 1, 16), dim=_log_int(rng, 16, 5120),
                        dstate=rng.choice([16, 16, 16, 16, 8, 32]), seqlen=_log_int(rng, 300, 32768),
                        flags=rng.random() < 0.75)
            # lengths and widths are multiples of something as often as they are odd
            if rng.random() < 0.5:
                case["dim"] = max(16, case["dim"] // 16 * 16)
                case["seqlen"] = max(256, case["seqlen"] // 64 * 64)
            if case["batch"] * case["dim"] * case["dstate"] * case["seqlen"] <= (3 << 30) // (2 if dtype == "f32" else 1):
                return case
    d_model = rng.choice([256, 512, 768, 1024, 1536, 2048, 2560])
    if kind == "step":
        return dict(kind=kind, dtype=dtype, batch=_log_int(rng, 1, 96), d_model=d_model)
    if kind == "decode":
        return dict(kind=kind, dtype=rng.choice(["f16", "bf16"]), batch=_log_int(rng, 1, 96), d_model=d_model,
                    n_layer=rng.choice([2, 4, 8]))
    while True:
        case = dict(kind=kind, dtype=dtype, batch=_log_int(rng, 1, 32), d_model=d_model,
                    seqlen=_log_int(rng, 33, 4096))
        if kind == "prompt":
            case["n_layer"] = rng.choice([2, 4, 8])
        tokens = case["batch"] * case["seqlen"] * case.get("n_layer", 1)
        if tokens * d_model * d_model <= (1 << 37) // (4 if dtype == "f32" else 1):
            return case


# ------------------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype, std=1.0, mean=0.0):
    return (torch.randn(shape, generator=g, device=DEVICE) * std + mean).to(dtype)


def _scan_inputs(case, seed):
    """u, B, C, z ~ N(0, 1).  With flags: delta before its softplus ~ N(-1, 1/2), A = -(1..dstate)
    and D, as a model's scan has them; without: the final step sizes and decay rates of the
    reference's benchmark, delta ~ U(0.01, 0.1), A ~ -U(0.1, 2)."""
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    b, d, n, L = case["batch"], case["dim"], case["dstate"], case["seqlen"]
    s = {"u": _normal(g, (b, d, L), dt)}
    if case["flags"]:
        s["delta"] = _normal(g, (b, d, L), dt, 0.5, -1.0)
        s["A"] = -torch.arange(1, n + 1, device=DEVICE, dtype=torch.float32).expand(d, n).contiguous()
        s["D"] = _normal(g, (d,), torch.float32, 0.1, 1.0)
        s["z"] = _normal(g, (b, d, L), dt)
    else:
        s["delta"] = (torch.rand((b, d, L), generator=g, device=DEVICE) * 0.09 + 0.01).to(dt)
        s["A"] = -(torch.rand((d, n), generator=g, device=DEVICE) * 1.9 + 0.1)
    s["B"] = _normal(g, (b, n, L), dt)
    s["C"] = _normal(g, (b, n, L), dt)
    return s


def _block_weights(g, d_model, dt, prefix=""):
    """A layer's parameters: projections scaled by their fan-in, step sizes from 1e-3 to 1e-1."""
    di, r, n, k = 2 * d_model, math.ceil(d_model / 16), 16, 4
    bias = torch.exp(torch.rand((di,), generator=g, device=DEVICE) * math.log(100.0) + math.log(1e-3))
    A_log = torch.log(torch.arange(1, n + 1, device=DEVICE, dtype=torch.float32)).expand(di, n)
    w = {
        "in_proj.weight": _normal(g, (2 * di, d_model), dt, d_model ** -0.5),
        "conv1d.weight": _normal(g, (di, 1, k), dt, k ** -0.5),
        "conv1d.bias": _normal(g, (di,), dt, 0.1),
        "x_proj.weight": _normal(g, (r + 2 * n, di), dt, di ** -0.5),
        "dt_proj.weight": _normal(g, (di, r), dt, r ** -0.5),
        "dt_proj.bias": torch.log(torch.expm1(bias)).to(dt),
        "A_log": A_log + 0.1 * torch.randn((di, n), generator=g, device=DEVICE),
        "D": _normal(g, (di,), torch.float32, 0.1, 1.0),
        "out_proj.weight": _normal(g, (d_model, di), dt, di ** -0.5),
    }
    return {prefix + key: v for key, v in w.items()}


def _model_weights(g, d_model, n_layer, dt):
    w = {"embeddings.weight": _normal(g, (VOCAB, d_model), dt, 0.05)}
    for i in range(n_layer):
        w[f"layers.{i}.norm.weight"] = _normal(g, (d_model,), dt, 0.1, 1.0)
        w.update(_block_weights(g, d_model, dt, f"layers.{i}.mixer."))
    w["norm_f.weight"] = _normal(g, (d_model,), dt, 0.1, 1.0)
    return w


def _load(make, weights):
    with torch.device("meta"):
        module = make()
    module = module.to_empty(device=DEVICE).requires_grad_(False).eval()
    module.load_state_dict(weights)
    return module


def _states(g, batch, d_model, dt, layers):
    di = 2 * d_model
    convs = [_normal(g, (batch, di, 4), dt) for _ in range(layers)]
    ssms = [_normal(g, (batch, di, 16), torch.float32, 0.5) for _ in range(layers)]
    return convs, ssms


def _inputs(case, seed):
    """Everything that the seed decides, weights included, as plain tensors."""
    if case["kind"] == "scan":
        return _scan_inputs(case, seed)
    g, dt, b, dm = _gen(seed), DTYPES[case["dtype"]], case["batch"], case["d_model"]
    if case["kind"] in ("layer", "step"):
        s = {"weights": _block_weights(g, dm, dt)}
        s["x"] = _normal(g, (b, case.get("seqlen", 1), dm), dt)
        if case["kind"] == "step":
            s["convs"], s["ssms"] = _states(g, b, dm, dt, 1)
        return s
    s = {"weights": _model_weights(g, dm, case["n_layer"], dt)}
    s["ids"] = torch.randint(0, VOCAB, (b, case.get("seqlen", 1)), generator=g, device=DEVICE)
    if case["kind"] == "decode":
        s["convs"], s["ssms"] = _states(g, b, dm, dt, case["n_layer"])
    return s


# ------------------------------------------------------------------------------ one pass
@torch.no_grad()
def prepare(case, seed):
    s = _inputs(case, seed)
    s["kind"] = case["kind"]
    if case["kind"] == "scan":
        s["options"] = dict(D=s["D"], z=s["z"], delta_softplus=True, return_state=True) if case["flags"] else {}
        return s
    dt = DTYPES[case["dtype"]]
    if case["kind"] in ("layer", "step"):
        s["block"] = _load(lambda: MambaBlock(case["d_model"], dtype=dt), s.pop("weights"))
        if case["kind"] == "step":  # the packed copies of the weights are made on first use
            s["block"].step(s["x"], s["convs"][0], s["ssms"][0])
        return s
    cfg = MambaConfig(d_model=case["d_model"], n_layer=case["n_layer"], vocab_size=VOCAB)
    model = s["model"] = _load(lambda: MambaModel(cfg, dtype=dt), s.pop("weights"))
    if case["kind"] == "prompt":
        s["prefill"] = GraphPrefill(model)
        s["prefill"](s["ids"])  # captures the graph of this prompt shape
        return s
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.inference_mode():
        with torch.cuda.stream(side):
            model.step(s["ids"], s["convs"], s["ssms"])
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["out"] = model.step(s["ids"], s["convs"], s["ssms"], inplace=True)
    return s


@torch.inference_mode()
def run(state):
    kind = state["kind"]
    if kind == "scan":
        return selective_scan(state["u"], state["delta"], state["A"], state["B"], state["C"],
                              **state["options"])
    if kind == "layer":
        return state["block"].prefill(state["x"])
    if kind == "step":
        return state["block"].step(state["x"], state["convs"][0], state["ssms"][0])
    if kind == "prompt":
        return state["prefill"](state["ids"])
    state["graph"].replay()
    return state["out"]


# ------------------------------------------------------------------------------ what it takes
def _size(dtype):
    return 4 if dtype == "f32" else 2


def work(case):
    es, b = _size(case["dtype"]), case["batch"]
    if case["kind"] == "scan":
        d, n, L = case["dim"], case["dstate"], case["seqlen"]
        tensors = 4 if case["flags"] else 3  # u, delta, y (z)
        byt = b * d * L * es * tensors + 2 * b * n * L * es + d * n * 4
        if case["flags"]:
            byt += d * 4 + b * d * n * 4
        # a state's step: the decay's product and exponential, the input's product, two fused
        # multiply-adds
        return {"bytes": byt, "flops": 7 * b * d * n * L}
    dm, layers, L = case["d_model"], case.get("n_layer", 1), case.get("seqlen", 1)
    di, r, n = 2 * dm, math.ceil(dm / 16), 16
    params = 2 * di * dm + di * 4 + (r + 2 * n) * di + di * r + di * dm
    rows = b * L
    flops = layers * rows * (2 * params + 7 * di * n)
    byt = layers * (params * es + di * (n + 1) * 4)
    state = b * di * (4 * es + n * 4) * layers  # conv and SSM states
    byt += state * (2 if case["kind"] in ("step", "decode") else 1)
    if case["kind"] in ("layer", "step"):
        return {"bytes": byt + 2 * rows * dm * es, "flops": flops}
    byt += VOCAB * dm * es + b * VOCAB * es + rows * dm * es
    return {"bytes": byt, "flops": flops + 2 * b * VOCAB * dm}


def tolerance(case):
    """About four times the distance from 64 bits (2-norm) that the cases have: the outputs' own
    rounding, fp32 sums, and in a model 16-bit roundings carried from layer to layer."""
    whole = case["kind"] in ("prompt", "decode")
    if case["dtype"] == "f32":  # 1e-7 to 2e-7 (scan), 9e-7 (layer), 1.3e-6 (two layers)
        return {"rel": 1e-5 if whole else 5e-6}
    if case["kind"] == "scan":  # 2.1e-4 and 1.7e-3: y's rounding
        return {"rel": 1e-3} if case["dtype"] == "f16" else {"rel": 7e-3}
    if case["dtype"] == "f16":  # 7e-4 (layer), 4e-3 (24 layers)
        return {"rel": 1.5e-2 if whole else 3e-3}
    return {"rel": 3e-2 if whole else 2e-2}  # 5.4e-3 (layer), 1.2e-2 (4 layers)


# ------------------------------------------------------------------------------ in 64 bits
def _exact_scan(u, delta, A, B, C, D=None, z=None):
    """u, delta (b, d, L) already final (softplus applied); everything float64 or cast per step."""
    b, d, L = u.shape
    h = torch.zeros((b, d, A.shape[1]), dtype=torch.float64, device=u.device)
    y = torch.empty((b, d, L), dtype=torch.float64, device=u.device)
    Bt, Ct = B.transpose(1, 2).double(), C.transpose(1, 2).double()  # (b, L, n)
    step = 512  # convert some steps at a time, time first
    for t0 in range(0, L, step):
        dts = delta[..., t0:t0 + step].double().permute(2, 0, 1).contiguous()
        us = u[..., t0:t0 + step].double().permute(2, 0, 1).contiguous()
        dus = dts * us
        for t in range(dts.shape[0]):
            Bv, Cv = Bt[:, t0 + t, None, :], Ct[:, t0 + t, None, :]
            h = torch.exp(dts[t][..., None] * A).mul_(h).add_(dus[t][..., None] * Bv)
            y[..., t0 + t] = (h * Cv).sum(-1)
    if D is not None:
        y += D[:, None] * u.double()
    if z is not None:
        y *= torch.nn.functional.silu(z.double())
    return y, h


def _exact_block(w, x, p="", conv=None, ssm=None):
    """A layer on (b, L, d_model) float64 from the given states (zeros where None)."""
    F, W = torch.nn.functional, lambda key: w[p + key].double()
    b, L, dm = x.shape
    di, r, n = 2 * dm, math.ceil(dm / 16), 16
    xz = x @ W("in_proj.weight").T
    xm, z = xz[..., :di].transpose(1, 2), xz[..., di:]
    hist = torch.zeros((b, di, 4), dtype=torch.float64, device=x.device) if conv is None else conv.double()
    full = torch.cat([hist, xm], dim=2)  # (b, di, 4 + L)
    new_conv = full[..., -4:]
    taps = W("conv1d.weight")[:, 0, :]
    xc = sum(full[..., 1 + k:1 + k + L] * taps[:, k, None] for k in range(4)) + W("conv1d.bias")[:, None]
    xc = F.silu(xc)
    dbl = xc.transpose(1, 2) @ W("x_proj.weight").T
    dt = F.softplus(dbl[..., :r] @ W("dt_proj.weight").T + W("dt_proj.bias"), threshold=60.0)
    A, Bm, Cm = -torch.exp(W("A_log")), dbl[..., r:r + n], dbl[..., r + n:]
    if ssm is None:
        y, h = _exact_scan(xc, dt.transpose(1, 2), A, Bm.transpose(1, 2), Cm.transpose(1, 2), W("D"))
    else:  # one token
        d1 = dt[:, 0, :, None]
        h = torch.exp(d1 * A) * ssm.double() + d1 * xc * Bm[:, 0, None, :]
        y = (h * Cm[:, 0, None, :]).sum(-1, keepdim=True) + W("D")[:, None] * xc
    y = y.transpose(1, 2) * F.silu(z)
    return y @ W("out_proj.weight").T, new_conv, h


@torch.inference_mode()
def exact(case, seed):
    s = _inputs(case, seed)
    if case["kind"] == "scan":
        A = s["A"].double()
        if not case["flags"]:
            return _exact_scan(s["u"], s["delta"], A, s["B"], s["C"])[0]
        delta = torch.nn.functional.softplus(s["delta"].double())
        return _exact_scan(s["u"], delta, A, s["B"], s["C"], s["D"].double(), s["z"])
    w = s["weights"]
    if case["kind"] == "layer":
        return _exact_block(w, s["x"].double())
    if case["kind"] == "step":
        return _exact_block(w, s["x"].double(), "", s["convs"][0], s["ssms"][0])

    def norm(x, key):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w[key].double()

    E = w["embeddings.weight"].double()
    x, convs, ssms = E[s["ids"]], [], []
    for i in range(case["n_layer"]):
        start = (s["convs"][i], s["ssms"][i]) if case["kind"] == "decode" else (None, None)
        y, conv, ssm = _exact_block(w, norm(x, f"layers.{i}.norm.weight"), f"layers.{i}.mixer.", *start)
        x = x + y
        convs.append(conv)
        ssms.append(ssm)
    return norm(x[:, -1:], "norm_f.weight") @ E.T, convs, ssms
