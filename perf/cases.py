"""The work that a user of this library has it do, as cases that can be timed and compared.

A decoder calls the feed-forward block once per layer and step: one token (decode), a speculative
verify block (16 or 32 tokens), a wider verify window (64), a short or a full prompt chunk (up to
2048 tokens), as ``Qwen36MLP.forward`` with the residual stream or as ``forward_rmsnorm`` with the
decoder's norm in front.  Weights are bfp8, the bf4 / bfp8 mix or bf16.  Before any of that, each
layer's checkpoint tensors are quantised and packed once by ``load_mlp_weights``.

Fields of a case: ``kind`` "forward" (``norm`` false), "norm" (``forward_rmsnorm``) or "load";
``hidden`` / ``intermediate`` (multiples of 256); ``tokens``; ``fmt``; ``residual`` (forward only);
``f32`` (an fp32 output instead of bf16).
"""
import math

import torch

import __graft_entry__

pkg = __graft_entry__.load_package()

H27, I27 = 5120, 17408  # the 27B layer
EPS = 1e-6
VALUE_BYTES = {"bf16": 2.0, "bfp8": 17 / 16, "bf4": 9 / 16}


def _case(kind, hidden, intermediate, tokens, fmt, residual=False, f32=False, name=None):
    c = {"kind": kind, "hidden": hidden, "intermediate": intermediate, "tokens": tokens, "fmt": fmt,
         "residual": residual, "f32": f32}
    return c if name is None else {"name": name, **c}


def listed():
    return [
        # the smallest model the library's tests run, one token: launches and host time count
        _case("forward", 1024, 3072, 1, "bf16", residual=True, name="decode1-small-bf16"),
        # plain decode, the whole feed-forward half of a decoder layer in one call
        _case("norm", H27, I27, 1, "bfp8", name="decode1-bfp8"),
        # a 16-token speculative verify block in each weight format
        _case("forward", H27, I27, 16, "bfp8", residual=True, name="verify16-bfp8"),
        _case("norm", H27, I27, 16, "bf4", name="verify16-bf4"),
        _case("forward", H27, I27, 16, "bf16", residual=True, name="verify16-bf16"),
        # one GPU's share of a layer split two ways: the fp32 partial that the all-reduce takes
        _case("forward", H27, I27 // 2, 16, "bfp8", f32=True, name="tp2-share16-bfp8"),
        # a 32-token verify block
        _case("norm", H27, I27, 32, "bfp8", name="verify32-bfp8"),
        # a 64-token verify window
        _case("forward", H27, I27, 64, "bfp8", residual=True, name="window64-bfp8"),
        # a short prompt of an odd length
        _case("norm", H27, I27, 201, "bf4", f32=True, name="prompt201-bf4"),
        # the ragged last chunk of a longer prompt, with the checkpoint's own weights
        _case("forward", H27, I27, 777, "bf16", residual=True, name="prompt777-bf16"),
        # a full prefill chunk
        _case("forward", H27, I27, 2048, "bfp8", residual=True, name="prefill2048-bfp8"),
        # one layer's checkpoint tensors to packed weights, as at model load
        _case("load", H27, I27, 0, "bfp8", name="load-bfp8"),
    ]


def draw(rng):
    """Shapes: the 27B layer, its two-way share, or any pair of multiples of 256 below them; tokens
    spread over their logarithm from 1 to 2000 (bf16 weights: to 1200)."""
    fmt = rng.choice(["bfp8", "bfp8", "bf4", "bf16"])
    pick = rng.random()
    if pick < 0.45:
        hidden, intermediate = H27, I27
    elif pick < 0.6:
        hidden, intermediate = H27, I27 // 2
    else:
        hidden = 256 * rng.randint(4, 20)
        intermediate = 256 * rng.randint(8, 68)
    if rng.random() < 0.1:
        hidden, intermediate = 256 * rng.randint(4, 20), 256 * rng.randint(8, 67)
        return _case("load", hidden, intermediate, 0, fmt)
    tokens = int(math.exp(rng.uniform(0.0, math.log(1200 if fmt == "bf16" else 2000))))
    if rng.random() < 0.4:
        return _case("norm", hidden, intermediate, tokens, fmt, f32=rng.random() < 0.3)
    return _case("forward", hidden, intermediate, tokens, fmt, residual=rng.random() < 0.7, f32=rng.random() < 0.3)


def _inputs(case, seed):
    """Checkpoint tensors ~ N(0, 0.02), activations ~ N(0, 1) with an RMSNorm-like channel gain,
    norm weights around zero (the gain is 1 + w)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(7919 * seed + 17)
    H, I, M = case["hidden"], case["intermediate"], case["tokens"]

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)

    sd = {"gate_proj.weight": (normal(I, H) * 0.02).bfloat16(), "up_proj.weight": (normal(I, H) * 0.02).bfloat16(),
          "down_proj.weight": (normal(H, I) * 0.02).bfloat16()}
    if case["kind"] == "load":
        return sd, None, None, None
    gain = 0.5 + torch.rand((H,), generator=g, device="cuda", dtype=torch.float32)
    x = (normal(M, H) * gain).bfloat16()
    r = normal(M, H).bfloat16() if case["residual"] else None
    w = (normal(H) * 0.1).bfloat16() if case["kind"] == "norm" else None
    return sd, x, r, w


def prepare(case, seed):
    sd, x, r, w = _inputs(case, seed)
    if case["kind"] == "load":
        return {"case": case, "sd": sd}
    mlp = pkg.Qwen36MLP("cuda", sd, weight_format=case["fmt"], max_tokens=case["tokens"])
    return {"case": case, "mlp": mlp, "x": x, "r": r, "w": w}


def run(state):
    case = state["case"]
    if case["kind"] == "load":
        lw = pkg.load_mlp_weights(torch.device("cuda"), state["sd"], weight_format=case["fmt"])
        return [lw.w1.buf, lw.w2.buf, lw.w3.buf]
    dtype = torch.float32 if case["f32"] else torch.bfloat16
    if case["kind"] == "norm":
        return state["mlp"].forward_rmsnorm(state["x"], state["w"], eps=EPS, out_dtype=dtype)
    return state["mlp"].forward(state["x"], residual=state["r"], out_dtype=dtype)


def work(case):
    H, I, M, fmt = case["hidden"], case["intermediate"], case["tokens"], case["fmt"]
    gate_up, down = VALUE_BYTES[fmt], VALUE_BYTES["bfp8" if fmt == "bf4" else fmt]
    weights = H * I * (2 * gate_up + down)
    if case["kind"] == "load":
        return {"bytes": 3 * H * I * 2 + weights, "flops": 0}
    rows = M * H * (2 + (4 if case["f32"] else 2) + (2 if case["residual"] else 0))
    return {"bytes": weights + rows + (2 * H if case["kind"] == "norm" else 0), "flops": 6 * M * H * I}


def tolerance(case):
    if case["kind"] == "load":
        return "exact"
    if case["fmt"] == "bf16":  # h is rounded to bf16 between the projections
        return {"rel": 8e-3, "max": 0.05}
    # h is rounded to fp16 between the projections; a bf16 output is rounded once more
    return {"rel": 1.2e-3, "max": 0.01} if case["f32"] else {"rel": 6e-3, "max": 0.03}


# ---------------------------------------------------------------- plain torch, 64 bits


def _block_float(w, magnitude_bits):
    """A bf16 matrix as its block-float weights mean it, in float64: 16 values along K share the
    largest exponent, each keeps `magnitude_bits` bits, rounded half to even."""
    v = w.double().reshape(w.shape[0], -1, 16)
    largest = v.abs().amax(dim=2, keepdim=True)
    binade = largest / torch.frexp(largest)[0]  # the power of two above it, exactly (a zero group: 0 / 0)
    step = torch.where(largest > 0, binade, 1.0) * 2.0 ** -magnitude_bits
    step = step.clamp(min=2.0 ** -126)
    top = 2 ** magnitude_bits - 1
    return (torch.round(v / step).clamp(-top, top) * step).reshape(w.shape)


def exact(case, seed):
    if case["kind"] == "load":
        return None
    sd, x, r, w = _inputs(case, seed)
    xd = x.double()
    if case["kind"] == "norm":
        r = x
        n = xd * torch.rsqrt(xd.square().mean(dim=1, keepdim=True) + EPS) * (1 + w.double())
        xd = n.bfloat16().double()  # the norm hands the block a bf16 tensor
    bits = {"gate_proj": {"bfp8": 7, "bf4": 3}, "up_proj": {"bfp8": 7, "bf4": 3}, "down_proj": {"bfp8": 7, "bf4": 7}}

    def weight(name):
        t = sd[name + ".weight"]
        return t.double() if case["fmt"] == "bf16" else _block_float(t, bits[name][case["fmt"]])

    g = xd @ weight("gate_proj").T
    u = xd @ weight("up_proj").T
    y = (g / (1 + torch.exp(-g)) * u) @ weight("down_proj").T
    return y if r is None else y + r.double()
