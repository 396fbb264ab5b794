"""GPU tests of the kernels and dispatch branches at the sizes where they can go wrong: the edges of
their tiles and of their sizes' ranges, remainders, and inputs that are not finite.  The bar is
``parity_helpers.check``'s (1e-2 of the oracle's RMS, the fp32 output)."""
import pytest

from oracle import mlp as omlp
from parity_helpers import check, host_weights

pytestmark = pytest.mark.gpu


def _mlp(pkg, cuda, H, I, fmt, M, layer=40):
    from qwen_mlp_amd import workloads

    sd = workloads.state_dict(H, I, layer=layer, device=cuda)
    return pkg.Qwen36MLP(cuda, sd, weight_format=fmt, max_tokens=M), sd


@pytest.mark.parametrize("fmt", ["bf16", "bfp8"])
@pytest.mark.parametrize("H,M", [(256, 5), (8192, 5), (8448, 5), (8448, 40), (2304, 33)])
def test_row_pass_lengths(pkg, cuda, fmt, H, M):
    """The norm / conversion pass: a row of 32 chunks for 256 threads, the longest row held in
    registers, the shortest re-read from memory, a row that is not a whole number of chunks per
    thread."""
    import torch
    from qwen_mlp_amd import workloads

    mlp, sd = _mlp(pkg, cuda, H, 512, fmt, M)
    nw = (torch.randn(H, generator=torch.Generator(cuda).manual_seed(3), device=cuda) * 0.3).to(torch.bfloat16)
    h = (workloads.activations(M, H, seed=60 + M, device=cuda).float() * 5.0).to(torch.bfloat16)
    y = mlp.forward_rmsnorm(h, nw, eps=1e-6, out_dtype=torch.float32)
    p = mlp.forward(h, out_dtype=torch.float32)
    torch.cuda.synchronize()
    hw = host_weights(pkg, sd, fmt)
    hf = h.float().cpu().numpy()
    ref = omlp.norm_swiglu(hf, nw.float().cpu().numpy(), hw["gate_proj"], hw["up_proj"], hw["down_proj"], 1e-6)
    check(y.cpu().numpy(), ref, f"row pass, norm {fmt} H={H} M={M}")
    ref = omlp.swiglu(hf, hw["gate_proj"], hw["up_proj"], hw["down_proj"], h_bf16=fmt == "bf16")
    check(p.cpu().numpy(), ref, f"row pass {fmt} H={H} M={M}")


@pytest.mark.parametrize("fmt", ["bf16", "bfp8", "bf4"])
@pytest.mark.parametrize("M", [5, 24, 40])
def test_non_finite_rows_stay_in_their_rows(pkg, cuda, fmt, M):
    """A NaN or an infinity makes every output of its own token row not finite, plain and behind the
    norm, and changes no bit of the other rows."""
    import torch
    from qwen_mlp_amd import workloads

    H = 1024
    mlp, _ = _mlp(pkg, cuda, H, 3072, fmt, M)
    nw = torch.zeros(H, dtype=torch.bfloat16, device=cuda)
    x = workloads.activations(M, H, seed=70 + M, device=cuda)
    bad = x.clone()
    bad[2, 700] = float("nan")
    bad[4, 3] = float("-inf")
    keep = [m for m in range(M) if m not in (2, 4)]
    for fn in (lambda t: mlp.forward(t, out_dtype=torch.float32),
               lambda t: mlp.forward_rmsnorm(t, nw, out_dtype=torch.float32)):
        good, got = fn(x), fn(bad)
        torch.cuda.synchronize()
        assert torch.isfinite(good).all()
        assert torch.equal(got[keep], good[keep])
        assert not torch.isfinite(got[[2, 4]]).any()


@pytest.mark.parametrize("fmt", ["bfp8", "bf4"])
@pytest.mark.parametrize("H", [2048, 8448])
@pytest.mark.parametrize("M", [1, 16, 24])
@pytest.mark.parametrize("depth", [29, 31, 34])
def test_normalised_rows_keep_small_values(pkg, cuda, fmt, H, M, depth):
    """Behind the norm, values far below their K range's maximum still count: one channel of each
    256 is 2^depth times larger than the others, gate reads only those channels and up only the
    others.  As fp16 with the maximum in [2^14, 2^15) the others are subnormal (6 bits of them left
    at depth 34; each is rounded on its own, and up sums thousands); the product stays near
    2^(depth - 27) times below the h bound, 11 bits or a few less."""
    import numpy as np
    import torch
    from oracle import bf16 as obf16

    I = 512
    g = torch.Generator(cuda).manual_seed(H + M + depth)

    def mantissas(*shape):
        return 1.0 + torch.rand(shape, generator=g, device=cuda)

    big = torch.arange(0, H, 256, device=cuda)
    group = torch.zeros(H, dtype=torch.bool, device=cuda)
    group[(big[:, None] + torch.arange(16, device=cuda)).flatten()] = True
    gate = torch.zeros(I, H, device=cuda)
    gate[:, big] = 0.125
    up = mantissas(I, H) * 0.25
    up[:, group] = 0.0
    sd = {"gate_proj.weight": gate.bfloat16(), "up_proj.weight": up.bfloat16(),
          "down_proj.weight": torch.randn(H, I, generator=g, device=cuda).bfloat16()}
    x = mantissas(M, H) * 2.0 ** -depth
    x[:, big] = mantissas(M, 1).expand(M, big.numel())
    x = x.bfloat16()
    mlp = pkg.Qwen36MLP(cuda, sd, weight_format=fmt, max_tokens=M)
    y = mlp.forward_rmsnorm(x, torch.zeros(H, dtype=torch.bfloat16, device=cuda), eps=1e-6, out_dtype=torch.float32)
    torch.cuda.synchronize()
    hw = host_weights(pkg, sd, fmt)
    xf = x.float().cpu().numpy()
    n = obf16.round_f32(omlp.rmsnorm(xf, np.zeros(H, np.float32), 1e-6))
    ref = omlp.swiglu(n, hw["gate_proj"], hw["up_proj"], hw["down_proj"], dtype=np.float64)
    small = ~group.cpu().numpy()  # where the residual is too small to round the sum
    check(y.cpu().numpy()[:, small] - xf[:, small], ref[:, small], f"small values {fmt} H={H} M={M} 2^-{depth}")


@pytest.mark.parametrize("fmt", ["bf16", "bfp8", "bf4"])
@pytest.mark.parametrize("rows,cols", [(16, 256), (48, 2048), (16, 2304), (32, 4352), (16, 45056), (16, 45312)])
def test_quantize_pack_matches_the_separate_passes(pkg, cuda, fmt, rows, cols):
    """The one-pass conversion writes the bytes of quantise + pack: fewer superblocks than waves, a
    remainder, the longest row whose exponents wait in LDS and the shortest whose do not; any finite
    bit pattern, denormals, ranges wide enough to flush groups, zero groups."""
    import torch
    from qwen_mlp_amd import _lib, mlp

    g = torch.Generator(cuda).manual_seed(rows + cols)
    normal = torch.randn(rows, cols, generator=g, device=cuda) * 0.02
    anyv = torch.randint(-32768, 32768, (rows, cols), generator=g, device=cuda).to(torch.int16).view(torch.bfloat16)
    binades = torch.randint(-30, 1, (rows, cols // 16), generator=g, device=cuda).float()
    inputs = {
        "any": torch.where(torch.isfinite(anyv.float()), anyv, torch.zeros_like(anyv)),
        "normal": normal.bfloat16(),
        "wide": (normal * torch.exp2(binades).repeat_interleave(16, dim=1)).bfloat16(),
        "denormal": (normal.double() * 2.0 ** -126).bfloat16(),
        "sparse": (normal * (torch.rand(rows, cols, generator=g, device=cuda) < 0.05)).bfloat16(),
        "zero": torch.zeros_like(anyv),
    }
    for name, w in inputs.items():
        got = mlp.pack_weight(w, fmt, strict=False)
        if fmt == "bf16":
            buf = torch.empty_like(got.buf)
            _lib.check(_lib.lib().qmlp_pack(_lib.ptr(w), None, rows, cols, _lib.FMT_BF16, _lib.ptr(buf), buf.numel(),
                                            _lib.stream_handle()), "qmlp_pack")
        else:
            want = mlp.pack_canonical(*mlp._quantize(w, fmt, None), fmt, strict=False)
            buf = want.buf
            assert (got.max_row_norm, got.flushed_groups) == (want.max_row_norm, want.flushed_groups), name
        assert torch.equal(got.buf, buf), name
    if fmt != "bf16":
        w = inputs["normal"].clone()
        w[rows - 1, 5], w[rows - 2, cols - 1] = float("nan"), float("-inf")
        with pytest.raises(ValueError, match="non-finite values in 2 groups"):
            mlp.pack_weight(w, fmt)


# (H, I, M) whose plans, over the three formats, take every built tile: each height in each mode, with
# one token block and with several, and each mode's sums (tests/test_abi.py checks that they do).
TILE_SHAPES = ([(2048, 6144, M) for M in (33, 65, 97, 129, 161, 193, 225, 321, 385, 449, 577, 777, 1153)]
               + [(5120, 17408, M) for M in (68, 97, 201, 321, 449, 705, 777, 1281)]
               + [(5376, 12288, 300), (256, 2560, 100), (2560, 256, 640), (768, 2048, 1800), (256, 10240, 1800),
                  (5120, 8192, 68), (768, 256, 33), (512, 3072, 33), (256, 17408, 68), (256, 5120, 2048),
                  (5120, 256, 2048), (3072, 4096, 1400), (1536, 17408, 500), (5120, 8192, 1600)])


@pytest.mark.parametrize("fmt", ["bf16", "bfp8", "bf4"])
@pytest.mark.parametrize("H,I,M", TILE_SHAPES)
def test_tile_heights_and_splits(pkg, cuda, fmt, H, I, M):
    """Many-token tiles of every height with one live token row in the last block or a ragged one,
    whole, split from the first tile on, and split behind whole rounds (the printed line is the
    plan); plain and behind the norm, twice."""
    import ctypes

    import numpy as np
    import torch
    from qwen_mlp_amd import _lib, workloads

    out = (ctypes.c_int * 8)()
    for down in (0, 1):
        assert pkg.lib().qmlp_plan_tiles(M, H, I, {"bf16": 0, "bfp8": 1, "bf4": 2}[fmt], down, 256, out) == 0
        print(fmt, H, I, M, "down" if down else "gate/up", list(out)[:6], flush=True)
    mlp, sd = _mlp(pkg, cuda, H, I, fmt, M)
    x = workloads.activations(M, H, seed=80 + M, device=cuda)
    nw = (torch.randn(H, generator=torch.Generator(cuda).manual_seed(5), device=cuda) * 0.1).to(torch.bfloat16)
    y = mlp.forward(x, residual=x, out_dtype=torch.float32)
    n = mlp.forward_rmsnorm(x, nw, out_dtype=torch.float32)
    assert torch.equal(mlp.forward(x, residual=x, out_dtype=torch.float32), y)
    assert torch.equal(mlp.forward(x, residual=x), y.to(torch.bfloat16))
    assert torch.equal(mlp.forward_rmsnorm(x, nw, out_dtype=torch.float32), n)
    torch.cuda.synchronize()
    rows = np.unique(np.r_[np.arange(0, M, 61), np.arange(0, M, 32)[-3:], M - 1])
    hw = host_weights(pkg, sd, fmt)
    xf = x.float().cpu().numpy()[rows]
    check(y.cpu().numpy()[rows],
          omlp.swiglu(xf, hw["gate_proj"], hw["up_proj"], hw["down_proj"], residual=xf, h_bf16=fmt == "bf16"),
          f"tiles {fmt} H={H} I={I} M={M}")
    check(n.cpu().numpy()[rows],
          omlp.norm_swiglu(xf, nw.float().cpu().numpy(), hw["gate_proj"], hw["up_proj"], hw["down_proj"], 1e-6),
          f"tiles, norm {fmt} H={H} I={I} M={M}")
