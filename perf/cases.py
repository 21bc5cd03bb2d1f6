"""The work that users of this framework have it do, as measurable cases: the
selective scan, the causal convolution, Mamba-2's SSD scan, the fused mixer and
the decode step, each through its public entry point.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs, weights and plans on the GPU
    run(state)          one pass and its outputs
    work(case)          bytes and operations that the pass cannot do without
    tolerance(case)     how far another correct implementation may be off
    exact(case, seed)   run()'s outputs in 64 bits from plain torch

Sizes come from the models this repository runs (Mamba-130M: d_model 768,
d_inner 1536, dstate 16, dt_rank 48, 24 layers; Mamba-2.8B and Mamba-2 2.7B
layers: d_inner 5120, 80 heads x 64, dstate 128) and from generic odd ones.
Layouts: "time" is a contiguous (batch, dim, seqlen) tensor, "channel" the
transposed view of a (batch, seqlen, dim) one, as transformers passes it.
"""

import math
import os
import sys
import types

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "mamba-cpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import mamba_cpu  # noqa: E402
import mamba_cpu.decode  # noqa: E402

DEV = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def listed():
    return [
        # One convolution step of a serving batch, the smallest call there is:
        # 64 sequences, the Mamba-130M fused (x, z) width, width 4.
        {"name": "conv_update_f32_b64", "op": "conv_update", "dtype": "f32", "b": 64, "d": 3072, "w": 4, "ring": 0},
        # One state step of a Mamba-2 2.7B layer for the same serving batch:
        # bf16 activations, the state kept in float32.
        {"name": "state_update_bf16_b64_h80", "op": "state_update", "dtype": "bf16", "b": 64, "h": 80, "p": 64,
         "n": 128, "g": 1, "z": False},
        # A training step's scan at Mamba-130M width: the headline workload.
        {"name": "scan_train_f32_b8_l1024", "op": "scan", "dtype": "f32", "b": 8, "d": 1536, "l": 1024, "n": 16,
         "z": True, "layout": "time", "train": True},
        # Prefill of one ragged prompt at the same width, as transformers'
        # mixer calls it: channel-contiguous views, the last state returned.
        {"name": "scan_prefill_f32_b1_l1999", "op": "scan", "dtype": "f32", "b": 1, "d": 1536, "l": 1999, "n": 16,
         "z": True, "layout": "channel", "train": False},
        # Training on one long sequence at Mamba-2.8B width in bf16.
        {"name": "scan_train_bf16_b1_l16384", "op": "scan", "dtype": "bf16", "b": 1, "d": 5120, "l": 16384, "n": 16,
         "z": False, "layout": "time", "train": True},
        # The complex-A scan (S4-style parametrisation) in training.
        {"name": "scan_complex_train_f32_b8_l1024", "op": "scan_complex", "dtype": "f32", "b": 8, "d": 1536,
         "l": 1024, "n": 16, "z": True, "train": True},
        # Training through the convolution in bf16.
        {"name": "conv_train_bf16_b8_l2048", "op": "conv", "dtype": "bf16", "b": 8, "d": 3072, "l": 2048, "w": 4,
         "layout": "time", "packed": 0, "train": True},
        # The same in float32 on a batch padded to its longest, odd, length.
        {"name": "conv_train_f32_b4_l1021", "op": "conv", "dtype": "f32", "b": 4, "d": 1536, "l": 1021, "w": 4,
         "layout": "time", "packed": 0, "train": True},
        # A training step's SSD scan at the Mamba-2 2.7B layer in bf16.
        {"name": "ssd_train_bf16_b4_l2048_h80", "op": "ssd", "dtype": "bf16", "b": 4, "l": 2048, "h": 80, "p": 64,
         "n": 128, "g": 1, "z": True, "train": True},
        # Prefill of a ragged batch at the Mamba-2 130M layer in float32, as
        # transformers' mixer calls it: no gate, the final states returned.
        {"name": "ssd_prefill_f32_b4_l1000_h24", "op": "ssd", "dtype": "f32", "b": 4, "l": 1000, "h": 24, "p": 64,
         "n": 128, "g": 1, "z": False, "train": False},
        # A training step's fused Mamba-130M mixer at 4 x 256 tokens.
        {"name": "mixer_train_f32_b4_l256", "op": "mixer", "b": 4, "l": 256, "dm": 768, "n": 16},
        # One token of Mamba-130M for four sequences, from embedding to
        # logits, replayed from its captured graph.
        {"name": "decode_mamba_f32_b4", "op": "decode", "dtype": "f32", "kind": "mamba", "b": 4, "layers": 24,
         "dm": 768, "n": 16, "vocab": 50280},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _fit(rng, limit, fixed, lo, hi):
    """A length from lo to hi, log-uniform, with fixed * length <= limit."""
    return max(lo, min(_log(rng, lo, hi), limit // fixed))


def draw(rng):
    op = rng.choice(["scan", "scan", "scan", "conv", "conv", "ssd", "ssd", "scan_complex", "conv_update",
                     "state_update", "mixer", "decode"])
    if op in ("scan", "scan_complex"):
        most = 8 * 1536 * 1024 if op == "scan_complex" else 5120 * 16384
        b = rng.choice([1, 1, 2, 3, 4, 8])
        d = rng.choice([_log(rng, 60, 5120), 1536, 2048, 2560, 5120])
        c = {"op": op, "dtype": "f32" if op == "scan_complex" else rng.choice(["f32", "bf16"]), "b": b, "d": d,
             "l": _fit(rng, most // 2, b * d, 17, 16384), "n": rng.choice([16, 16, 16, 8, 32]),
             "z": rng.random() < 0.6, "train": rng.random() < 0.6}
        if op == "scan_complex":
            c["n"] = rng.choice([16, 8])
        else:
            c["layout"] = rng.choice(["time", "channel"])
        return c
    if op == "conv":
        b = rng.choice([1, 2, 3, 4, 8])
        d = rng.choice([_log(rng, 60, 5376), 1536, 3072, 5120])
        layout = rng.choice(["time", "time", "channel"])
        return {"op": op, "dtype": rng.choice(["f32", "bf16", "f16"]), "b": b, "d": d,
                "l": _fit(rng, 8 * 3072 * 2048, b * d, 17, 16384), "w": rng.choice([4, 4, 4, 3, 2]),
                "layout": layout, "packed": rng.choice([0, 0, 5]), "train": rng.random() < 0.6}
    if op == "ssd":
        b, h = rng.choice([1, 2, 3, 4, 8]), rng.choice([8, 16, 24, 32, 48, 80])
        train = rng.random() < 0.6
        return {"op": op, "dtype": rng.choice(["f32", "bf16"]), "b": b,
                "l": _fit(rng, 4 * 2048 * 80 // 2, b * h, 33, 8192), "h": h, "p": rng.choice([64, 64, 32]),
                "n": rng.choice([128, 128, 64]), "g": rng.choice([1, 1, 2, 8]), "z": rng.random() < 0.5,
                "train": train}
    if op == "conv_update":
        return {"op": op, "dtype": rng.choice(["f32", "bf16"]), "b": _log(rng, 1, 128),
                "d": rng.choice([1536, 3072, 5376, _log(rng, 60, 5376)]), "w": rng.choice([4, 4, 3]),
                "ring": rng.choice([0, 0, 8])}
    if op == "state_update":
        if rng.random() < 0.5:  # Mamba-1: one head row per channel
            return {"op": op, "dtype": rng.choice(["f32", "bf16"]), "b": _log(rng, 1, 128), "h": 0,
                    "p": rng.choice([1536, 5120, _log(rng, 60, 5120)]), "n": 16, "g": 1, "z": rng.random() < 0.5}
        return {"op": op, "dtype": rng.choice(["f32", "bf16"]), "b": _log(rng, 1, 64),
                "h": rng.choice([24, 48, 80]), "p": 64, "n": rng.choice([128, 128, 64]), "g": rng.choice([1, 8]),
                "z": rng.random() < 0.3}
    if op == "mixer":
        return {"op": op, "b": rng.choice([1, 2, 4]), "l": _log(rng, 33, 512), "dm": 64 * rng.randint(4, 16),
                "n": 16}
    kind = rng.choice(["mamba", "mamba2"])
    return {"op": op, "dtype": rng.choice(["f32", "bf16"]), "kind": kind, "b": rng.randint(1, 8),
            "layers": rng.randint(2, 24), "dm": rng.choice([256, 512, 768, 1024]),
            "n": 16 if kind == "mamba" else 128, "vocab": rng.choice([1000, 50280])}


# ---- inputs ----

class _Rng:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def n(self, *shape):
        return torch.randn(*shape, generator=self.g, device=DEV)

    def u(self, *shape):
        return torch.rand(*shape, generator=self.g, device=DEV)


def _laid(r, case, b, d, l):
    """(b, d, l) normal values in the case's dtype and layout."""
    dt = DTYPES[case["dtype"]]
    if case.get("layout") == "channel":
        return r.n(b, l, d).to(dt).transpose(1, 2)
    return r.n(b, d, l).to(dt)


def _log_a(r, *shape):
    return -torch.exp(r.u(*shape) * math.log(16))


def _packed_ids(r, b, l, count):
    """Ids of `count` sequences of random lengths packed in each row."""
    cuts = torch.sort((r.u(b, count - 1) * l).long(), dim=1).values
    return (torch.arange(l, device=DEV)[None, :, None] >= cuts[:, None, :]).sum(-1).to(torch.int32)


def _scan_inputs(case, r):
    b, d, l, n = (case[k] for k in "bdln")
    t = {"u": _laid(r, case, b, d, l), "delta": _laid(r, case, b, d, l)}
    dt = DTYPES[case["dtype"]]
    if case["op"] == "scan_complex":
        t["A"] = torch.complex(_log_a(r, d, n), r.n(d, n) * math.pi)
        t["B"], t["C"] = r.n(b, n, 2 * l), r.n(b, n, 2 * l)
    else:
        t["A"] = _log_a(r, d, n)
        t["B"], t["C"] = r.n(b, n, l).to(dt), r.n(b, n, l).to(dt)
    t["D"] = r.n(d)
    if case["z"]:
        t["z"] = _laid(r, case, b, d, l)
    t["delta_bias"] = r.u(d) * 2 - 4
    return t


def _ssd_inputs(case, r):
    b, l, h, p, n, g = (case[k] for k in "blhpng")
    dt = DTYPES[case["dtype"]]
    t = {"x": r.n(b, l, h, p).to(dt), "dt": r.n(b, l, h) * 0.5 - 1.0, "A": _log_a(r, h),
         "B": r.n(b, l, g, n).to(dt), "C": r.n(b, l, g, n).to(dt), "D": r.n(h), "dt_bias": r.u(h) * 0.5}
    if case["z"]:
        t["z"] = r.n(b, l, h, p).to(dt)
    return t


def _mixer_inputs(case, r):
    b, l, dm, n = case["b"], case["l"], case["dm"], case["n"]
    d, rank = 2 * dm, math.ceil(dm / 16)
    lin = lambda o, i: (r.u(o, i) * 2 - 1) / math.sqrt(i)  # noqa: E731
    return {"xz": r.n(b, l, 2 * d).transpose(1, 2), "conv1d_weight": (r.u(d, 1, 4) * 2 - 1) * 0.5,
            "conv1d_bias": (r.u(d) * 2 - 1) * 0.5, "x_proj_weight": lin(rank + 2 * n, d),
            "delta_proj_weight": lin(d, rank), "out_proj_weight": lin(dm, d),
            "A": -torch.arange(1, n + 1, device=DEV, dtype=torch.float32).repeat(d, 1), "D": torch.ones(d, device=DEV),
            "delta_bias": r.u(d) * 4 - 6}


class _Model(torch.nn.Module):
    """The parts of a Mamba or Mamba-2 language model that
    mamba_cpu.decode.GraphedDecodeStep reads, with random weights."""

    def __init__(self, case, r):
        super().__init__()
        dm, n, dt = case["dm"], case["n"], DTYPES[case["dtype"]]
        d, m2 = 2 * dm, case["kind"] == "mamba2"
        heads, rank = d // 64, math.ceil(dm / 16)
        conv_dim = d + 2 * n if m2 else d

        def mod(**parts):
            m = torch.nn.Module()
            for k, v in parts.items():
                setattr(m, k, torch.nn.Parameter(v, requires_grad=False) if torch.is_tensor(v) else v)
            return m

        def lin(o, i, bias=None):
            return mod(weight=((r.u(o, i) * 2 - 1) / math.sqrt(i)).to(dt), bias=bias)

        def norm(width):
            m = mod(weight=(1 + 0.1 * r.n(width)).to(dt))
            m.variance_epsilon = 1e-5
            return m

        layers = []
        for i in range(case["layers"]):
            mx = mod(in_proj=lin(d + conv_dim + heads if m2 else 2 * d, dm),
                     conv1d=mod(weight=((r.u(conv_dim, 1, 4) * 2 - 1) * 0.5).to(dt),
                                bias=((r.u(conv_dim) * 2 - 1) * 0.5).to(dt)),
                     out_proj=lin(dm, d))
            mx.activation, mx.intermediate_size, mx.ssm_state_size, mx.conv_kernel_size = "silu", d, n, 4
            if m2:
                mx.norm = norm(d)
                mx.dt_bias = torch.nn.Parameter((r.u(heads) * 4 - 6).to(dt), requires_grad=False)
                mx.A_log = torch.nn.Parameter((r.u(heads) * math.log(16)).to(dt), requires_grad=False)
                mx.D = torch.nn.Parameter(torch.ones(heads, device=DEV, dtype=dt), requires_grad=False)
            else:
                mx.x_proj = lin(rank + 2 * n, d)
                mx.dt_proj = lin(d, rank, (r.u(d) * 4 - 6).to(dt))
                mx.A_log = torch.nn.Parameter(
                    torch.arange(1, n + 1, device=DEV).float().log().repeat(d, 1).to(dt), requires_grad=False)
                mx.D = torch.nn.Parameter(torch.ones(d, device=DEV, dtype=dt), requires_grad=False)
            blk = mod(norm=norm(dm), mixer=mx)
            blk.layer_idx, blk.residual_in_fp32 = i, True
            layers.append(blk)
        self.config = types.SimpleNamespace(model_type=case["kind"])
        self.backbone = mod(norm_f=norm(dm))
        self.backbone.layers = torch.nn.ModuleList(layers)
        self.backbone.embeddings = torch.nn.Embedding(case["vocab"], dm, device=DEV, dtype=dt,
                                                      _weight=(r.n(case["vocab"], dm)).to(dt))
        self.lm_head = lin(case["vocab"], dm)


def _decode_parts(case, seed):
    r = _Rng(seed)
    model = _Model(case, r)
    b, dm, n, dt = case["b"], case["dm"], case["n"], DTYPES[case["dtype"]]
    d, m2 = 2 * dm, case["kind"] == "mamba2"
    conv = r.n(case["layers"], b, d + 2 * n if m2 else d, 4).to(dt)
    ssm = r.n(*((case["layers"], b, d // 64, 64, n) if m2 else (case["layers"], b, d, n))) * 0.1
    layers = [types.SimpleNamespace(conv_states={0: conv[i]}, recurrent_states={0: ssm[i]}, record_past=False)
              for i in range(case["layers"])]
    token = (r.u(b, 1) * case["vocab"]).long().clamp_(max=case["vocab"] - 1)
    return model, types.SimpleNamespace(layers=layers), conv, ssm, token


def prepare(case, seed):
    op = case["op"]
    r = _Rng(seed)
    if op in ("scan", "scan_complex", "ssd", "mixer"):
        make = {"ssd": _ssd_inputs, "mixer": _mixer_inputs}.get(op, _scan_inputs)
        t = make(case, r)
        s = {"case": case, "t": t}
        if case.get("train", True):
            for v in t.values():
                v.requires_grad_()
            if op == "mixer":
                s["gout"] = r.n(case["b"], case["l"], case["dm"])
            elif op == "ssd":
                s["gout"] = r.n(*t["x"].shape).to(t["x"].dtype)
            else:
                s["gout"] = _laid(r, case, case["b"], case["d"], case["l"])
        return s
    if op == "conv":
        b, d, l, w = (case[k] for k in "bdlw")
        t = {"x": _laid(r, case, b, d, l), "weight": r.n(d, w) * 0.5, "bias": r.n(d) * 0.1 ** 0.5}
        s = {"case": case, "t": t, "seq_idx": _packed_ids(r, b, l, case["packed"]) if case["packed"] else None}
        if case["train"]:
            for v in t.values():
                v.requires_grad_()
            s["gout"] = _laid(r, case, b, d, l)
        return s
    if op == "conv_update":
        b, d, w = (case[k] for k in "bdw")
        dt = DTYPES[case["dtype"]]
        s = {"case": case, "x": r.n(b, d).to(dt), "weight": r.n(d, w) * 0.5, "bias": r.n(d) * 0.1 ** 0.5}
        if case["ring"]:  # a pool of ring buffers, of which the batch uses every other one
            s["state"] = r.n(2 * b, d, case["ring"]).to(dt)
            s["pos"] = (r.u(b) * 1000).to(torch.int32)
            s["rows"] = torch.arange(0, 2 * b, 2, device=DEV, dtype=torch.int32)
        else:
            s["state"] = r.n(b, d, w - 1).to(dt)
        return s
    if op == "state_update":
        b, h, p, n, g = (case[k] for k in "bhpng")
        dt = DTYPES[case["dtype"]]
        if h:  # Mamba-2's per-head values, expanded as transformers passes them
            s = {"state": r.n(b, h, p, n), "x": r.n(b, h, p).to(dt),
                 "dt": (r.n(b, h) * 0.5).to(dt)[:, :, None].expand(b, h, p),
                 "A": _log_a(r, h)[:, None, None].expand(h, p, n), "B": r.n(b, g, n).to(dt),
                 "C": r.n(b, g, n).to(dt), "D": r.n(h)[:, None].expand(h, p),
                 "z": r.n(b, h, p).to(dt) if case["z"] else None, "dt_bias": (r.u(h) * 2 - 4)[:, None].expand(h, p)}
        else:
            s = {"state": r.n(b, p, n), "x": r.n(b, p).to(dt), "dt": (r.n(b, p) * 0.5).to(dt), "A": _log_a(r, p, n),
                 "B": r.n(b, n).to(dt), "C": r.n(b, n).to(dt), "D": r.n(p),
                 "z": r.n(b, p).to(dt) if case["z"] else None, "dt_bias": r.u(p) * 2 - 4}
        return {"case": case, **s}
    model, cache, conv, ssm, token = _decode_parts(case, seed)
    step = mamba_cpu.decode.GraphedDecodeStep(model, cache, case["b"])
    step.token.copy_(token)
    return {"case": case, "step": step, "conv": conv, "ssm": ssm}


# ---- one pass ----

def run(s):
    case = s["case"]
    op = case["op"]
    if op in ("scan", "scan_complex"):
        t = s["t"]
        if not case["train"]:
            out, last = mamba_cpu.selective_scan_fn(**t, delta_softplus=True, return_last_state=True)
            return {"out": out, "last": last}
        out = mamba_cpu.selective_scan_fn(**t, delta_softplus=True)
    elif op == "ssd":
        t = s["t"]
        main = [t[k] for k in ("x", "dt", "A", "B", "C")]
        rest = {k: t[k] for k in ("D", "z", "dt_bias") if k in t}
        if not case["train"]:
            out, final = mamba_cpu.mamba_chunk_scan_combined(*main, 256, **rest, dt_softplus=True,
                                                             return_final_states=True)
            return {"out": out, "final": final}
        out = mamba_cpu.mamba_chunk_scan_combined(*main, 256, **rest, dt_softplus=True)
    elif op == "conv":
        t = s["t"]
        out = mamba_cpu.causal_conv1d_fn(t["x"], t["weight"], t["bias"], seq_idx=s["seq_idx"], activation="silu")
        if not case["train"]:
            return {"out": out}
    elif op == "mixer":
        t = s["t"]
        out = mamba_cpu.mamba_inner_fn(**t, out_proj_bias=None, delta_softplus=True)
    elif op == "conv_update":
        kw = {"cache_seqlens": s["pos"], "conv_state_indices": s["rows"]} if case["ring"] else {}
        out = mamba_cpu.causal_conv1d_update(s["x"], s["state"], s["weight"], s["bias"], activation="silu", **kw)
        return {"out": out, "state": s["state"]}
    elif op == "state_update":
        out = mamba_cpu.selective_state_update(s["state"], s["x"], s["dt"], s["A"], s["B"], s["C"], s["D"], s["z"],
                                               s["dt_bias"], dt_softplus=True)
        return {"out": out, "state": s["state"]}
    else:
        return {"logits": s["step"].replay(), "conv": s["conv"], "ssm": s["ssm"]}
    grads = torch.autograd.grad(out, list(t.values()), s["gout"])
    return {"out": out, **{"d" + k: v for k, v in zip(t, grads)}}


# ---- what a pass cannot do without ----

def work(case):
    op = case["op"]
    e = 4 if case.get("dtype", "f32") == "f32" else 2
    if op in ("scan", "scan_complex"):
        b, d, l, n = (case[k] for k in "bdln")
        cx = 2 if op == "scan_complex" else 1
        x, bc, prm = b * d * l * e, 2 * b * n * l * e * cx, 4 * (d * n * cx + 2 * d)
        z = int(case["z"])
        fwd = (3 + z) * x + bc + prm
        # decay, exponential, input, state and output terms of a state-step
        ops = 8 * cx * cx
        if not case["train"]:
            return {"bytes": fwd + 4 * b * d * n * cx, "flops": ops * b * d * l * n}
        return {"bytes": fwd + (5 + 2 * z) * x + 2 * bc + 2 * prm, "flops": 3 * ops * b * d * l * n}
    if op == "ssd":
        b, l, h, p, n, g = (case[k] for k in "blhpng")
        x, bc, z = b * l * h * p * e, 2 * b * l * g * n * e, int(case["z"])
        fwd = (2 + z) * x + bc + 4 * b * l * h
        # state update and output, each 2 p n per head and step
        ops = 4 * p * n * b * l * h
        if not case["train"]:
            return {"bytes": fwd + 4 * b * h * p * n, "flops": ops}
        return {"bytes": fwd + (3 + 2 * z) * x + 2 * bc + 8 * b * l * h, "flops": 3 * ops}
    if op == "conv":
        b, d, l, w = (case[k] for k in "bdlw")
        x = b * d * l * e
        ids = 4 * b * l if case["packed"] else 0
        if not case["train"]:
            return {"bytes": 2 * x + ids, "flops": 2 * w * b * d * l}
        return {"bytes": 5 * x + 2 * ids, "flops": 6 * w * b * d * l}
    if op == "conv_update":
        b, d, w = (case[k] for k in "bdw")
        moved = (w if case["ring"] else 2 * (w - 1)) + 2
        return {"bytes": moved * b * d * e + 4 * d * (w + 1), "flops": 2 * w * b * d}
    if op == "state_update":
        b, h, p, n, g = (case[k] for k in "bhpng")
        rows = max(h, 1) * p
        per = 4 * (2 * rows + rows * n) if not h else 12 * h
        dt = b * (h if h else rows) * e
        return {"bytes": 8 * b * rows * n + (2 + int(case["z"])) * b * rows * e + dt + per + 2 * b * g * n * e,
                "flops": 6 * b * rows * n}
    if op == "mixer":
        b, l, dm, n = case["b"], case["l"], case["dm"], case["n"]
        d, rank = 2 * dm, math.ceil(dm / 16)
        weights = d * (rank + 2 * n) + d * rank + dm * d + d * (n + 7)
        gemm = 2 * b * l * (d * (rank + 2 * n) + d * rank + dm * d)
        return {"bytes": 4 * (4 * d + 2 * dm) * b * l + 12 * weights, "flops": 3 * gemm + 24 * b * l * d * n}
    b, dm, n, layers, vocab = (case[k] for k in ("b", "dm", "n", "layers", "vocab"))
    d, rank = 2 * dm, math.ceil(dm / 16)
    conv_dim = d + 2 * n if case["kind"] == "mamba2" else d
    if case["kind"] == "mamba2":
        per = dm * (d + conv_dim + d // 64) + dm * d + 5 * conv_dim
    else:
        per = dm * 2 * d + d * (rank + 2 * n) + d * rank + dm * d + d * (n + 7)
    weights = layers * per + vocab * dm
    states = layers * b * (2 * conv_dim * 4 * e + 8 * d * n)
    return {"bytes": weights * e + states + 4 * b * vocab, "flops": 2 * b * weights}


def tolerance(case):
    """About four times the largest error of any output against exact(), over
    the listed and some sixty drawn cases: 16-bit values carry a rounding or
    two (up to 2^-9 of a bf16 value, 2^-12 of an f16 one); the sums over a
    whole row of steps behind dA and the bias gradients lead among the 32-bit
    ones."""
    op, dt = case["op"], case.get("dtype", "f32")
    if op == "decode":  # rounding travels through all layers
        return {"rel": 2e-6 if dt == "f32" else 3e-2}
    if dt != "f32":
        return {"rel": 1e-2 if dt == "bf16" else 1e-3}
    if op == "ssd":
        return {"rel": 4e-5 if case["train"] else 1e-6}
    return {"rel": {"scan": 4e-6, "scan_complex": 5e-6, "mixer": 6e-6}.get(op, 1e-6)}


# ---- the same in 64 bits, from plain torch ----

def _d(t):
    return None if t is None else t.detach().to(torch.complex128 if t.is_complex() else torch.float64)


def _grads64(leaves, fn, gout, rows):
    """Outputs and gradients of fn over batch rows taken one at a time (its
    per-row tensors, in `rows`, sliced), so that the graph of one row at a time
    is held. fn(leaves) -> (out, *others); gradients of out only."""
    leaf = {k: _d(v).requires_grad_(gout is not None) for k, v in leaves.items()}
    b = next(iter(leaf[k] for k in rows)).shape[0]
    outs = []
    for i in range(b):
        part = {k: v[i:i + 1] if k in rows else v for k, v in leaf.items()}
        res = fn(part)
        if gout is not None:
            res[0].backward(_d(gout[i:i + 1]))
        outs.append([v.detach() for v in res])
    outs = [torch.cat(v) for v in zip(*outs)]
    return outs, {"d" + k: v.grad for k, v in leaf.items()}


def _scan64(t, seqlen):
    """out and last state of the selective scan, one step after the other."""
    cx = t["A"].is_complex()
    dt = F.softplus(t["delta"] + t["delta_bias"][None, :, None])
    if cx:
        pair = lambda X: torch.view_as_complex(  # noqa: E731
            X.unflatten(-1, (seqlen, 2)).contiguous()).unbind(-1)
        B, C = pair(t["B"]), pair(t["C"])
    else:
        B, C = t["B"].unbind(-1), t["C"].unbind(-1)
    dts, us, ys = dt.unbind(-1), (dt * t["u"]).unbind(-1), []
    h = torch.zeros(*dts[0].shape, t["A"].shape[1], dtype=t["A"].dtype, device=DEV)
    for i in range(seqlen):
        h = torch.exp(dts[i][..., None] * t["A"]) * h + us[i][..., None] * B[i][:, None]
        y = (h * C[i][:, None]).sum(-1)
        ys.append(2 * y.real if cx else y)
    y = torch.stack(ys, -1) + t["D"][None, :, None] * t["u"]
    return (y * F.silu(t["z"]) if "z" in t else y), h


def _ssd64(t, heads):
    rep = heads // t["B"].shape[2]
    dt = F.softplus(t["dt"] + t["dt_bias"])
    dec, dx = torch.exp(dt * t["A"]).unbind(1), (dt[..., None] * t["x"]).unbind(1)
    B, C = (t[k].repeat_interleave(rep, 2).unbind(1) for k in "BC")
    h, ys = 0, []
    for i in range(len(dec)):
        h = dec[i][..., None, None] * h + dx[i][..., None] * B[i][:, :, None]
        ys.append((h * C[i][:, :, None]).sum(-1))
    y = torch.stack(ys, 1) + t["D"][:, None] * t["x"]
    return (y * F.silu(t["z"]) if "z" in t else y), h


def _conv64(x, weight, bias, ids=None):
    w, l = weight.shape[1], x.shape[-1]
    out = bias[None, :, None].expand_as(x)
    for k in range(w):
        lag = w - 1 - k
        tap = F.pad(x, (lag, 0))[..., :l]
        if ids is not None and lag:
            tap = tap * (F.pad(ids, (lag, 0), value=-1)[..., :l] == ids)[:, None]
        out = out + weight[None, :, k, None] * tap
    return F.silu(out)


def _mixer64(t):
    d, rank, n = t["A"].shape[0], t["delta_proj_weight"].shape[1], t["A"].shape[1]
    x, z = t["xz"][:, :d], t["xz"][:, d:]
    u = _conv64(x, t["conv1d_weight"][:, 0], t["conv1d_bias"])
    dt, B, C = (u.transpose(1, 2) @ t["x_proj_weight"].t()).split([rank, n, n], -1)
    delta = (dt @ t["delta_proj_weight"].t()).transpose(1, 2)
    y, _ = _scan64({"u": u, "delta": delta, "A": t["A"], "B": B.transpose(1, 2), "C": C.transpose(1, 2),
                    "D": t["D"], "z": z, "delta_bias": t["delta_bias"]}, x.shape[-1])
    return y.transpose(1, 2) @ t["out_proj_weight"].t()


def _rms64(x, w, eps=1e-5):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * _d(w)


def _decode64(case, seed):
    model, _, conv, ssm, token = _decode_parts(case, seed)
    dm, n, m2 = case["dm"], case["n"], case["kind"] == "mamba2"
    d, conv, ssm = 2 * dm, _d(conv), _d(ssm)
    hid = _d(model.backbone.embeddings.weight)[token[:, 0]]
    for i, blk in enumerate(model.backbone.layers):
        mx = blk.mixer
        proj = _rms64(hid, blk.norm.weight) @ _d(mx.in_proj.weight).t()
        if m2:
            gate, x, dt = proj.split([d, d + 2 * n, d // 64], -1)
        else:
            x, gate = proj.split([d, d], -1)
        conv[i] = torch.cat([conv[i][..., 1:], x[..., None]], -1)
        x = F.silu((conv[i] * _d(mx.conv1d.weight)[:, 0]).sum(-1) + _d(mx.conv1d.bias))
        A, D = -torch.exp(_d(mx.A_log)), _d(mx.D)
        if m2:
            x, B, C = x.split([d, n, n], -1)
            x = x.unflatten(-1, (-1, 64))
            dt = F.softplus(dt + _d(mx.dt_bias))
            ssm[i] = torch.exp(dt * A)[..., None, None] * ssm[i] + (dt[..., None] * x)[..., None] * B[:, None, None]
            y = ((ssm[i] * C[:, None, None]).sum(-1) + D[:, None] * x).flatten(1)
            y = _rms64(y * F.silu(gate), mx.norm.weight)
        else:
            rank = mx.dt_proj.weight.shape[1]
            dt, B, C = (x @ _d(mx.x_proj.weight).t()).split([rank, n, n], -1)
            dt = F.softplus(dt @ _d(mx.dt_proj.weight).t() + _d(mx.dt_proj.bias))
            ssm[i] = torch.exp(dt[..., None] * A) * ssm[i] + (dt * x)[..., None] * B[:, None]
            y = ((ssm[i] * C[:, None]).sum(-1) + D * x) * F.silu(gate)
        hid = hid + y @ _d(mx.out_proj.weight).t()
    logits = _rms64(hid, model.backbone.norm_f.weight) @ _d(model.lm_head.weight).t()
    return {"logits": logits, "conv": conv, "ssm": ssm}


def exact(case, seed):
    op = case["op"]
    if op == "decode":
        return _decode64(case, seed)
    s = prepare(case, seed)
    if op in ("scan", "scan_complex", "ssd"):
        t, rows = s["t"], [k for k in ("u", "delta", "B", "C", "z", "x", "dt") if k in s["t"]]
        fn = (lambda p: _ssd64(p, case["h"])) if op == "ssd" else (lambda p: _scan64(p, case["l"]))  # noqa: E731
        (out, last), grads = _grads64(t, fn, s.get("gout"), rows)
        if case["train"]:
            return {"out": out, **grads}
        return {"out": out, "final" if op == "ssd" else "last": last}
    if op in ("conv", "mixer"):
        t = {k: _d(v).requires_grad_() for k, v in s["t"].items()}
        ids = s.get("seq_idx")
        out = _mixer64(t) if op == "mixer" else _conv64(t["x"], t["weight"], t["bias"], ids)
        if "gout" not in s:
            return {"out": out.detach()}
        grads = torch.autograd.grad(out, list(t.values()), _d(s["gout"]))
        return {"out": out.detach(), **{"d" + k: v for k, v in zip(t, grads)}}
    if op == "conv_update":
        x, st, w = _d(s["x"]), _d(s["state"]), _d(s["weight"])
        k = w.shape[1]
        if case["ring"]:
            ring, rows, pos = st.shape[-1], s["rows"].long(), s["pos"].long()
            at = lambda j: (pos + j) % ring  # noqa: E731
            taps = [st[rows, :, at(j - (k - 1))] for j in range(k - 1)] + [x]
            st[rows, :, at(0)] = x
        else:
            taps = list(st.unbind(-1)) + [x]
            st = torch.stack(taps[1:], -1)
        out = _d(s["bias"]) + sum(taps[j] * w[:, j] for j in range(k))
        return {"out": F.silu(out), "state": st}
    v = {k: _d(s[k]) for k in ("state", "x", "dt", "A", "B", "C", "D", "z", "dt_bias")}
    dt = F.softplus(v["dt"] + v["dt_bias"])
    if case["h"]:
        rep = case["h"] // case["g"]
        B, C = (v[k].repeat_interleave(rep, 1)[:, :, None] for k in "BC")
    else:
        B, C = v["B"][:, None], v["C"][:, None]
    st = torch.exp(dt[..., None] * v["A"]) * v["state"] + (dt * v["x"])[..., None] * B
    y = (st * C).sum(-1) + v["D"] * v["x"]
    return {"out": y if v["z"] is None else y * F.silu(v["z"]), "state": st}
