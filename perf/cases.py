"""The work this package is measured on: its public entry points at the sizes a program uses.

``listed()`` names the cases; ``draw(rng)`` gives further ones of the same ranges.  ``prepare``
makes what a program holds before the call (inputs, parameters, the module), ``run`` is one pass
through the public entry points, ``exact`` the same pass in plain torch in 64 bits.

Kinds of case (the key ``kind``):
  wkv         chunk_rwkv6, forward and backward (a training step's WKV6, head-first)
  wkv_infer   fused_recurrent_rwkv6 without gradients, state in and out (decode: T = 1; prefill)
  shift_mix   timemix.token_shift_mix, forward and backward
  decay       timemix.decay_lora, forward and backward
  gn_gate     timemix.group_norm_gate on the head-first WKV output, forward and backward
  channel_mix modules.RWKV6ChannelMix, forward and backward
  time_mix    modules.RWKV6TimeMix, forward and backward
  layer       modules.RWKV6Layer with fp32 parameters, forward and backward
  lm          modules.RWKV6Model with fp32 parameters, a prompt's logits without gradients
"""
import importlib

import torch
import torch.nn.functional as F

pkg = importlib.import_module("rwkv-megatron_amd")

HEAD = 64
VOCAB = 65536
DEV = "cuda"
BF16 = torch.bfloat16


# ---------------------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------------------

def listed():
    return [
        # one layer's WKV6 of a training step whose B*H fills the device
        dict(name="wkv_train_8x32x4096", kind="wkv", B=8, H=32, T=4096, state=False),
        # long context, one sequence, state carried in and out with its gradients
        dict(name="wkv_long_1x32x32768", kind="wkv", B=1, H=32, T=32768, state=True),
        # the tiny language model's WKV6: few, short sequences
        dict(name="wkv_short_2x8x512", kind="wkv", B=2, H=8, T=512, state=False),
        # one generated token for eight conversations: the smallest call
        dict(name="wkv_decode_8x32x1", kind="wkv_infer", B=8, H=32, T=1),
        # a prompt of odd length before decoding
        dict(name="wkv_prefill_2x32x1001", kind="wkv_infer", B=2, H=32, T=1001),
        # the token mixing of one 1.6B-shape layer in training
        dict(name="shift_mix_4096x4x2048", kind="shift_mix", T=4096, B=4, C=2048),
        # its decay bottleneck
        dict(name="decay_4096x4x2048", kind="decay", T=4096, B=4, C=2048),
        # its GroupNorm and gate
        dict(name="gn_gate_4096x4x2048", kind="gn_gate", T=4096, B=4, C=2048),
        # a whole channel mix in training at a shorter context
        dict(name="channel_mix_2048x2x2048", kind="channel_mix", T=2048, B=2, C=2048, F=7168),
        # a whole time mix in training, 1.6B shape
        dict(name="time_mix_4096x4x2048", kind="time_mix", T=4096, B=4, C=2048),
        # one layer of the tiny language model's training step: bound by launches
        dict(name="layer_512x2x512", kind="layer", T=512, B=2, C=512, F=1792),
        # the tiny language model over a prompt of odd length
        dict(name="lm_prompt_1x777", kind="lm", B=1, T=777, C=512, F=1792, L=2),
    ]


def _log_int(rng, lo, hi):
    """A whole number from lo to hi, spread over the logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """One more case.  No drawn case has more tokens x heads (or tokens x channels) than the
    listed case of its kind that has the most."""
    kind = rng.choice(["wkv", "wkv", "wkv_decode", "wkv_prefill", "shift_mix", "decay", "gn_gate",
                       "channel_mix", "time_mix", "layer", "lm"])
    if kind == "wkv":
        B, H = rng.choice([1, 2, 3, 4, 8]), rng.choice([8, 16, 32, 64])
        T = _log_int(rng, 48, min(32768, (8 * 32 * 4096) // (B * H)))
        return dict(kind="wkv", B=B, H=H, T=T, state=rng.random() < 0.4)
    if kind == "wkv_decode":
        return dict(kind="wkv_infer", B=_log_int(rng, 1, 64), H=rng.choice([8, 32, 64]),
                    T=rng.choice([1, 1, 1, 2, 4]))
    if kind == "wkv_prefill":
        B, H = rng.choice([1, 2, 4, 8]), rng.choice([8, 32, 64])
        return dict(kind="wkv_infer", B=B, H=H, T=_log_int(rng, 8, (8 * 32 * 4096) // (B * H)))
    if kind in ("shift_mix", "decay", "gn_gate"):
        B, C = rng.choice([1, 2, 3, 4]), rng.choice([512, 1024, 2048, 4096])
        T = _log_int(rng, 64, (4096 * 4 * 2048) // (B * C))
        return dict(kind=kind, T=T, B=B, C=C)
    if kind == "channel_mix":
        B, (C, Fh) = rng.choice([1, 2, 3]), rng.choice([(512, 1792), (2048, 7168)])
        return dict(kind="channel_mix", T=_log_int(rng, 64, 4096 // B), B=B, C=C, F=Fh)
    if kind == "time_mix":
        B, C = rng.choice([1, 2, 4]), rng.choice([512, 1024, 2048])
        return dict(kind="time_mix", T=_log_int(rng, 64, 16384 // B), B=B, C=C)
    if kind == "layer":
        B = rng.choice([1, 2, 4])
        return dict(kind="layer", T=_log_int(rng, 64, 4096 // B), B=B, C=512, F=1792)
    return dict(kind="lm", B=rng.choice([1, 2]), T=_log_int(rng, 128, 1024), C=512, F=1792, L=2)


# ---------------------------------------------------------------------------------------
# inputs and parameters
# ---------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape, std=1.0, dtype=BF16):
    return torch.randn(*shape, generator=g, device=DEV).mul_(std).to(dtype)


def _rand(g, *shape, lo=0.0, hi=1.0, dtype=BF16):
    return torch.rand(*shape, generator=g, device=DEV).mul_(hi - lo).add_(lo).to(dtype)


def _wkv_inputs(case, seed):
    """r, k, v ~ N(0,1), log-decay -exp(U(-6, -0.5)), u ~ N(0, 0.1^2), states ~ N(0, 0.5^2)."""
    g = _gen(seed)
    B, H, T = case["B"], case["H"], case["T"]
    s = {n: _randn(g, B, H, T, HEAD) for n in ("r", "k", "v")}
    s["w"] = -torch.exp(_rand(g, B, H, T, HEAD, lo=-6.0, hi=-0.5, dtype=torch.float32))
    s["w"] = s["w"].to(BF16)
    s["u"] = _randn(g, H, HEAD, std=0.1, dtype=torch.float32)
    if case["kind"] == "wkv_infer" or case["state"]:
        s["h0"] = _randn(g, B, H, HEAD, HEAD, std=0.5, dtype=torch.float32)
    if case["kind"] == "wkv":
        s["do"] = _randn(g, B, H, T, HEAD)
        if case["state"]:
            s["dhT"] = _randn(g, B, H, HEAD, HEAD, dtype=torch.float32)
    return s


def _ramp(C, lo, hi):
    return torch.linspace(lo, hi, C, device=DEV)


def _time_mix_params(g, C, dtype, prefix=""):
    """A time mix's parameters at trained magnitudes: LoRA outputs of a few tenths, mixing
    coefficients in (0, 1), the decay ramp from -6 to -1."""
    p = {
        "bottleneck_token_shift.weight_down": _randn(g, C, 5, 32, std=0.5 * C ** -0.5, dtype=dtype),
        "bottleneck_token_shift.weight_up": _randn(g, 5, 32, C, std=0.04, dtype=dtype),
        "bottleneck_token_shift.bias": _rand(g, 5, C, dtype=dtype),
        "bottleneck_decay.weight_down": _randn(g, C, 1, 64, std=0.5 * C ** -0.5, dtype=dtype),
        "bottleneck_decay.weight_up": _randn(g, 1, 64, C, std=0.04, dtype=dtype),
        "bottleneck_decay.bias": (_ramp(C, -6.0, -1.0)[None] + _randn(g, 1, C, std=0.1, dtype=torch.float32)).to(dtype),
        "mix_coeff_input": _rand(g, C, dtype=dtype),
        "core_attention.time_first": (1 + _randn(g, C, std=0.3, dtype=torch.float32)).to(dtype),
        "group_norm.weight": _rand(g, C, lo=0.5, hi=1.5, dtype=dtype),
        "group_norm.bias": _randn(g, C, std=0.1, dtype=dtype),
    }
    for n in ("receptance", "key", "value", "gate", "proj"):
        p[f"linear_{n}.weight"] = _randn(g, C, C, std=C ** -0.5, dtype=dtype)
    return {prefix + n: t for n, t in p.items()}


def _channel_mix_params(g, C, Fh, dtype, prefix=""):
    p = {"mix_coeffs": _rand(g, 2, C, dtype=dtype),
         "linear_up.weight": _randn(g, Fh, C, std=C ** -0.5, dtype=dtype),
         "linear_gate.weight": _randn(g, C, C, std=C ** -0.5, dtype=dtype),
         "linear_down.weight": _randn(g, C, Fh, std=Fh ** -0.5, dtype=dtype)}
    return {prefix + n: t for n, t in p.items()}


def _norm_params(g, C, dtype, prefix):
    return {prefix + "weight": _rand(g, C, lo=0.5, hi=1.5, dtype=dtype),
            prefix + "bias": _randn(g, C, std=0.1, dtype=dtype)}


def _layer_params(g, C, Fh, dtype, prefix=""):
    p = _norm_params(g, C, dtype, prefix + "input_layernorm.")
    p.update(_norm_params(g, C, dtype, prefix + "pre_mlp_layernorm."))
    p.update(_time_mix_params(g, C, dtype, prefix + "self_attention."))
    p.update(_channel_mix_params(g, C, Fh, dtype, prefix + "mlp."))
    return p


def _inputs(case, seed):
    """Inputs and parameters by name, made from the seed alone."""
    kind = case["kind"]
    if kind in ("wkv", "wkv_infer"):
        return _wkv_inputs(case, seed)
    g = _gen(seed)
    if kind == "lm":
        C, dt = case["C"], torch.float32
        p = {"embedding.weight": _randn(g, VOCAB, C, std=0.5, dtype=dt),
             "output_layer.weight": _randn(g, VOCAB, C, std=C ** -0.5, dtype=dt)}
        p.update(_norm_params(g, C, dt, "pre_norm."))
        p.update(_norm_params(g, C, dt, "final_layernorm."))
        for i in range(case["L"]):
            p.update(_layer_params(g, C, case["F"], dt, f"layers.{i}."))
        tokens = torch.randint(0, VOCAB, (case["B"], case["T"]), generator=g, device=DEV)
        return {"p": p, "tokens": tokens}
    T, B, C = case["T"], case["B"], case["C"]
    s = {"x": _randn(g, T, B, C), "dy": _randn(g, T, B, C)}
    if kind == "shift_mix":
        s["dy"] = [s["dy"]] + [_randn(g, T, B, C) for _ in range(4)]
    if kind in ("shift_mix", "decay", "gn_gate"):
        tm = _time_mix_params(g, C, BF16)
        if kind == "shift_mix":
            t = "bottleneck_token_shift."
            s["p"] = [tm["mix_coeff_input"], tm[t + "weight_down"], tm[t + "weight_up"], tm[t + "bias"]]
        elif kind == "decay":
            t = "bottleneck_decay."
            s["p"] = [tm[t + "weight_down"], tm[t + "weight_up"], tm[t + "bias"]]
        else:
            s["o"] = _randn(g, B, C // HEAD, T, HEAD, std=4.0)
            s["p"] = [tm["group_norm.weight"], tm["group_norm.bias"]]
    elif kind in ("time_mix", "layer"):
        # The first token's WKV output is (r . u k) v: its GroupNorm forgets the factor, and the
        # gradient through it is a difference of nearly equal numbers over |r . u k|, on which no
        # two 16-bit evaluations agree.  The next tokens' are sums of a few such terms.  The first
        # eight outputs carry no loss here.
        s["dy"][:8] = 0
        s["p"] = (_time_mix_params(g, C, BF16) if kind == "time_mix"
                  else _layer_params(g, C, case["F"], torch.float32))
    else:
        s["p"] = _channel_mix_params(g, C, case["F"], BF16)
    return s


# ---------------------------------------------------------------------------------------
# the package's passes
# ---------------------------------------------------------------------------------------

def _config(case, dtype):
    C = case["C"]
    return pkg.modules.TransformerConfig(
        hidden_size=C, num_attention_heads=C // HEAD, ffn_hidden_size=case.get("F", 7168),
        num_layers=case.get("L", 24), params_dtype=dtype, perform_initialization=False)


def _module(case, device):
    M, kind = pkg.modules, case["kind"]
    if kind == "lm":
        return M.RWKV6Model(_config(case, torch.float32), VOCAB, device=device)
    if kind == "layer":
        return M.RWKV6Layer(_config(case, torch.float32), 2, device=device)
    make = M.RWKV6TimeMix if kind == "time_mix" else M.RWKV6ChannelMix
    return make(_config(case, BF16), 2, device=device)


def prepare(case, seed):
    kind, s = case["kind"], _inputs(case, seed)
    s["case"] = case
    if kind == "wkv":
        for n in ("r", "k", "v", "w", "u") + (("h0",) if case["state"] else ()):
            s[n].requires_grad_(True)
    elif kind in ("shift_mix", "decay", "gn_gate"):
        s["x"].requires_grad_(True)
        if kind == "gn_gate":
            s["o"].requires_grad_(True)
        for t in s["p"]:
            t.requires_grad_(True)
    elif kind != "wkv_infer":
        M = pkg.modules
        s["m"] = _module(case, DEV)
        if kind != "lm":
            s["x"].requires_grad_(True)
        s["m"].load_state_dict(s.pop("p"))
        s["params"] = list(s["m"].parameters())
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "wkv_infer":
        with torch.no_grad():
            o, hT = pkg.wkv.fused_recurrent_rwkv6(s["r"], s["k"], s["v"], s["w"], s["u"], scale=1.0,
                                                  initial_state=s["h0"], output_final_state=True)
        return {"o": o, "state": hT}
    if kind == "wkv":
        o, hT = pkg.wkv.chunk_rwkv6(s["r"], s["k"], s["v"], s["w"], s["u"], scale=1.0,
                                    initial_state=s.get("h0"), output_final_state=case["state"])
        wrt = [s[n] for n in ("r", "k", "v", "w", "u")]
        if case["state"]:
            return {"o": o.detach(), "state": hT.detach(),
                    "grads": torch.autograd.grad([o, hT], wrt + [s["h0"]], [s["do"], s["dhT"]])}
        return {"o": o.detach(), "grads": torch.autograd.grad(o, wrt, s["do"])}
    if kind == "shift_mix":
        out = pkg.timemix.token_shift_mix(s["x"], *s["p"])
        return {"out": [t.detach() for t in out],
                "grads": torch.autograd.grad(out, [s["x"]] + s["p"], s["dy"])}
    if kind == "decay":
        out = pkg.timemix.decay_lora(s["x"], *s["p"])
        return {"out": out.detach(), "grads": torch.autograd.grad(out, [s["x"]] + s["p"], s["dy"])}
    if kind == "gn_gate":
        out = pkg.timemix.group_norm_gate(s["o"], s["x"], *s["p"], 1e-5)
        return {"out": out.detach(),
                "grads": torch.autograd.grad(out, [s["o"], s["x"]] + s["p"], s["dy"])}
    if kind == "lm":
        with torch.no_grad():
            return {"logits": s["m"](s["tokens"])}
    out = s["m"](s["x"])
    out = out if kind == "layer" else out[0]
    return {"out": out.detach(), "grads": torch.autograd.grad(out, [s["x"]] + s["params"], s["dy"])}


# ---------------------------------------------------------------------------------------
# the work a pass cannot do without, and what its results may be off by
# ---------------------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("wkv", "wkv_infer"):
        bh, T = case["B"] * case["H"], case["T"]
        state = 4 * HEAD * HEAD * bh                                  # one fp32 state per sequence
        step = 2 * HEAD * HEAD * bh * T                               # one 64 x 64 product per token
        if kind == "wkv_infer":                                       # r k v w in, o out, states
            return dict(bytes=5 * 2 * HEAD * bh * T + 2 * state, flops=2 * step)
        # r k v w do in, o dr dk dv dw out; h0 dhT in, hT dh0 out
        return dict(bytes=10 * 2 * HEAD * bh * T + (4 * state if case["state"] else 0), flops=7 * step)
    T, B, C = case["T"], case["B"], case["C"]
    N, act = T * B, 2 * T * B * C
    if kind == "shift_mix":      # x, 5 dy in; 5 mixes, dx out; down and up, forward and backward
        return dict(bytes=12 * act + 2 * 2 * 2 * 5 * 32 * C, flops=3 * 2 * 2 * N * C * 5 * 32)
    if kind == "decay":          # x, dy in; out, dx out
        return dict(bytes=4 * act + 2 * 2 * 2 * 64 * C, flops=3 * 2 * 2 * N * C * 64)
    if kind == "gn_gate":        # o, gate, dy in; y, d_o, d_gate out
        return dict(bytes=6 * act, flops=40 * N * C)
    step = 2 * HEAD * C * N
    if kind == "channel_mix":
        w = C * (2 * case["F"] + C)
        return dict(bytes=4 * act + 2 * 2 * w, flops=6 * N * w)
    tm = 5 * C * C + 2 * C * (5 * 32 + 64)
    if kind == "time_mix":
        return dict(bytes=4 * act + 2 * 2 * tm, flops=6 * N * tm + 7 * step)
    w = tm + C * (2 * case["F"] + C)
    if kind == "layer":
        return dict(bytes=4 * act + 2 * 4 * w, flops=6 * N * w + 7 * step)
    w = case["L"] * w + VOCAB * C
    return dict(bytes=4 * w + 4 * N * C + 2 * N * VOCAB, flops=2 * N * w + 2 * step * case["L"])


def tolerance(case):
    """bf16 outputs of bf16 operands: about four times the error against the 64-bit result.  The
    blocks and the model hand bf16 activations from product to product; their parameter
    gradients carry those roundings."""
    kind = case["kind"]
    if kind in ("wkv", "wkv_infer", "gn_gate"):
        return {"rel": 0.012}
    if kind in ("shift_mix", "decay"):
        return {"rel": 0.016}
    return {"rel": 0.03}


# ---------------------------------------------------------------------------------------
# the same passes in plain torch, 64 bits
# ---------------------------------------------------------------------------------------

def _wkv64(r, k, v, w, u, h0):
    """o, final state of the RWKV-6 recurrence for [B,H,T,64] tensors, in blocks of 16 tokens:
    pairwise decays inside a block, the state carried from block to block."""
    B, H, T, K = r.shape
    bl = 16
    n = -(-T // bl)
    pad = lambda t: F.pad(t, (0, 0, 0, n * bl - T)).reshape(B, H, n, bl, K)
    r, k, v, w = pad(r), pad(k), pad(v), pad(w)
    G = w.cumsum(3)
    Gp = G - w
    mask = torch.ones(bl, bl, device=r.device, dtype=torch.bool).tril(-1)[..., None]
    D = (Gp.unsqueeze(4) - G.unsqueeze(3)).masked_fill(~mask, float("-inf")).exp()
    A = ((r.unsqueeze(4) * D) * k.unsqueeze(3)).sum(-1)
    o = A @ v + (r * u[None, :, None, None, :] * k).sum(-1, keepdim=True) * v
    end = G[:, :, :, -1]
    add = (k * (end.unsqueeze(3) - G).exp()).transpose(3, 4) @ v
    S, starts = h0, []
    for c in range(n):
        starts.append(S)
        S = end[:, :, c].exp().unsqueeze(-1) * S + add[:, :, c]
    o = o + (r * Gp.exp()) @ torch.stack(starts, 2)
    return o.reshape(B, H, n * bl, K)[:, :, :T], S


def _shift(x):
    return torch.cat([torch.zeros_like(x[:1]), x[:-1]], 0)


def _lora64(x, down, up, bias):
    C, E, R = down.shape
    neck = torch.tanh(x @ down.reshape(C, E * R)).reshape(*x.shape[:-1], E, R)
    return torch.stack([neck[..., e, :] @ up[e] + bias[e] for e in range(E)], -2)


def _token_shift_mix64(x, maa, down, up, bias):
    delta = _shift(x) - x
    m = _lora64(x + delta * maa, down, up, bias)
    return [x + delta * m[..., e, :] for e in range(5)]


def _gn_gate64(o, g, gamma, beta):
    B, H, T, K = o.shape
    o = o - o.mean(-1, keepdim=True)
    o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-5)
    return (o.permute(2, 0, 1, 3).reshape(T, B, H * K) * gamma + beta) * F.silu(g)


def _time_mix64(x, p, pre=""):
    q = lambda n: p[pre + n]
    bt, bd = "bottleneck_token_shift.", "bottleneck_decay."
    mw, mk, mv, mr, mg = _token_shift_mix64(x, q("mix_coeff_input"), q(bt + "weight_down"),
                                            q(bt + "weight_up"), q(bt + "bias"))
    decay = _lora64(mw, q(bd + "weight_down"), q(bd + "weight_up"), q(bd + "bias"))[..., 0, :]
    T, B, C = x.shape
    hf = lambda t: t.view(T, B, C // HEAD, HEAD).permute(1, 2, 0, 3)
    lin = lambda t, n: t @ q(f"linear_{n}.weight").t()
    o, _ = _wkv64(hf(lin(mr, "receptance")), hf(lin(mk, "key")), hf(lin(mv, "value")),
                  hf(-torch.exp(decay)), q("core_attention.time_first").view(C // HEAD, HEAD),
                  x.new_zeros(B, C // HEAD, HEAD, HEAD))
    y = _gn_gate64(o, lin(mg, "gate"), q("group_norm.weight"), q("group_norm.bias"))
    return lin(y, "proj")


def _channel_mix64(x, p, pre=""):
    q = lambda n: p[pre + n]
    delta = _shift(x) - x
    up, gate = (x + delta * q("mix_coeffs")[e] for e in range(2))
    h = torch.relu(up @ q("linear_up.weight").t()) ** 2
    return (h @ q("linear_down.weight").t()) * torch.sigmoid(gate @ q("linear_gate.weight").t())


def _ln64(x, p, pre):
    x = x - x.mean(-1, keepdim=True)
    x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5)
    return x * p[pre + "weight"] + p[pre + "bias"]


def _layer64(x, p, pre=""):
    x = x + _time_mix64(_ln64(x, p, pre + "input_layernorm."), p, pre + "self_attention.")
    return x + _channel_mix64(_ln64(x, p, pre + "pre_mlp_layernorm."), p, pre + "mlp.")


def _lm64(tokens, p, L):
    x = _ln64(p["embedding.weight"][tokens.t()], p, "pre_norm.")
    for i in range(L):
        x = _layer64(x, p, f"layers.{i}.")
    return _ln64(x, p, "final_layernorm.") @ p["output_layer.weight"].t()


def exact(case, seed):
    kind, s = case["kind"], _inputs(case, seed)
    d = lambda t: t.double().requires_grad_(True)
    if kind in ("wkv", "wkv_infer"):
        x = [d(s[n]) for n in ("r", "k", "v", "w", "u")]
        shape = (case["B"], case["H"], HEAD, HEAD)
        h0 = d(s["h0"]) if "h0" in s else torch.zeros(shape, device=DEV, dtype=torch.float64)
        if kind == "wkv_infer":
            with torch.no_grad():
                o, hT = _wkv64(*x, h0)
            return {"o": o, "state": hT}
        o, hT = _wkv64(*x, h0)
        if case["state"]:
            return {"o": o.detach(), "state": hT.detach(),
                    "grads": torch.autograd.grad([o, hT], x + [h0], [s["do"].double(), s["dhT"].double()])}
        return {"o": o.detach(), "grads": torch.autograd.grad(o, x, s["do"].double())}
    if kind == "shift_mix":
        x, p = d(s["x"]), [d(t) for t in s["p"]]
        out = _token_shift_mix64(x, *p)
        return {"out": [t.detach() for t in out],
                "grads": torch.autograd.grad(out, [x] + p, [t.double() for t in s["dy"]])}
    if kind == "decay":
        x, p = d(s["x"]), [d(t) for t in s["p"]]
        out = _lora64(x, *p)[..., 0, :]
        return {"out": out.detach(), "grads": torch.autograd.grad(out, [x] + p, s["dy"].double())}
    if kind == "gn_gate":
        o, x, p = d(s["o"]), d(s["x"]), [d(t) for t in s["p"]]
        out = _gn_gate64(o, x, *p)
        return {"out": out.detach(), "grads": torch.autograd.grad(out, [o, x] + p, s["dy"].double())}
    # the module's parameters in the order in which it lists them
    p = {n: d(s["p"][n]) for n, _ in _module(case, "meta").named_parameters()}
    if kind == "lm":
        with torch.no_grad():
            return {"logits": _lm64(s["tokens"], p, case["L"])}
    x = d(s["x"])
    block = {"time_mix": _time_mix64, "channel_mix": _channel_mix64, "layer": _layer64}[kind]
    out = block(x, p)
    return {"out": out.detach(), "grads": torch.autograd.grad(out, [x] + list(p.values()), s["dy"].double())}
