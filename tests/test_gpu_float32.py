"""The float32 kernels on the matrix cores against float64: every workgroup shape of the product at the edges of its
tiles and of K."""

import pytest
import torch

import plain_qwen3 as plain
from test_gpu_kernels import close, rnd

pytestmark = pytest.mark.gpu
F64 = torch.float64
SHAPES = 8                     # workgroup shapes of the float32 product


# A sum of K float32 products in any order lies within about sqrt(K) * 6e-8 of the exact one, relative to the root of
# the summed squares, which is what the largest result of a random product is a few times of: 6e-6 covers K = 4096.
@pytest.mark.parametrize("shape", range(SHAPES + 1))
@pytest.mark.parametrize("M,N,K", [(1, 16, 16), (1, 33, 4), (5, 70, 100), (16, 130, 1000), (17, 64, 2048), (33, 127, 36),
                                   (65, 200, 516), (130, 96, 4096)])
def test_gemm_f32(shape, M, N, K):
    from tie_amd import kernels

    x, w = rnd(M, K, seed=M), rnd(N, K, seed=N, scale=0.1)
    want = plain.linear(x, w)
    x, w = x.cuda(), w.cuda()
    out = torch.full((M, N), float("nan"), device="cuda")
    kernels.gemm_f32(x, w, out, shape=shape)
    close(out, want, 6e-6, f"product {M}x{N}x{K}, shape {shape}")
    base = rnd(M, N, seed=7).cuda()
    acc = base.clone()
    kernels.gemm_f32(x, w, acc, accumulate=True, shape=shape)
    close(acc, want + base.cpu().to(F64), 6e-6, "added to what was there")
    for splits in (2, 3, 16):
        planes = torch.full((splits, M, N), float("nan"), device="cuda")
        kernels.gemm_f32(x, w, planes, splits=splits, shape=shape)
        close(planes.sum(0), want, 6e-6, f"{splits} planes")


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("M,I,K", [(1, 8, 64), (5, 24, 200), (17, 136, 1000), (70, 72, 516)])
def test_gemm_f32_gated(M, I, K, activation):
    from tie_amd import kernels

    x, gate, up = rnd(M, K, seed=M), rnd(I, K, seed=2, scale=0.1), rnd(I, K, seed=3, scale=0.1)
    g, u = plain.linear(x, gate), plain.linear(x, up)
    act = g / (1 + torch.exp(-g)) if activation == "silu" else torch.nn.functional.gelu(g, approximate="tanh")
    w = kernels.interleave_gate_up(gate, up).cuda()
    for shape in range(SHAPES + 1):
        out = torch.full((M, I), float("nan"), device="cuda")
        kernels.gemm_f32(x.cuda(), w, out, shape=shape, gated=1 + kernels.GATE_ACTIVATIONS[activation])
        close(out, act * u, 6e-6, f"gated product, shape {shape}")
    kernels.linear_swiglu(x.cuda(), w, out, activation=activation)
    close(out, act * u, 6e-6, "gated product")


def test_gemm_f32_keeps_a_bad_row_to_itself():
    """An infinity in one row of x, or behind the last k of a row, reaches that row's results and no other's."""
    from tie_amd import kernels

    for shape in range(1, SHAPES + 1):
        x, w = rnd(40, 52, seed=1).cuda(), rnd(48, 52, seed=2).cuda()
        good = torch.empty(40, 48, device="cuda")
        kernels.gemm_f32(x, w, good, shape=shape)
        x[7, 51] = float("inf")
        w[9, 0] = float("nan")
        out = torch.empty(40, 48, device="cuda")
        kernels.gemm_f32(x, w, out, shape=shape)
        bad = ~torch.isfinite(out)
        assert bool(bad[7].all()) and bool(bad[:, 9].all())
        bad[7], bad[:, 9] = False, False
        assert not bool(bad.any())
        keep = [i for i in range(40) if i != 7], [j for j in range(48) if j != 9]
        assert torch.equal(out[keep[0]][:, keep[1]], good[keep[0]][:, keep[1]])


def test_the_32_bit_path_takes_these_kernels():
    """The dispatcher: operands the kernel takes go there (other results only by rounding), the others as before."""
    from tie_amd import kernels

    x, w = rnd(5, 64, seed=1).cuda(), rnd(24, 64, seed=2).cuda()
    out, same = torch.empty(5, 24, device="cuda"), torch.empty(5, 24, device="cuda")
    kernels.linear(x, w, out)
    kernels.gemm_f32(x, w, same)
    assert torch.equal(out, same)
    odd = torch.empty(5 * 64 + 1, device="cuda")[1:].view(5, 64).copy_(x)      # rows that begin off a 16-byte address
    assert not kernels.gemm_f32_takes(odd, w, out)
    kernels.linear(odd, w, same)
    close(same, out.cpu().to(F64), 2e-6, "an input off a 16-byte address")
    kernels.linear(x[:, :62].contiguous(), w[:, :62].contiguous(), out)
    close(out, plain.linear(x[:, :62].cpu(), w[:, :62].cpu()), 2e-6, "K % 4 != 0")
