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
