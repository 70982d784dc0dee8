"""The float32 kernels on the matrix cores against float64: every workgroup shape of the product at the edges of its
tiles and of K, and the attention over all head sizes, groups, masks, caps, sinks, page types and shares."""

import pytest
import torch

import plain_qwen3 as plain
from test_gpu_kernels import attention_case, close, rnd

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


# The same bound; a tile is 64 rows of x and 64 of w a wave, k in slices of 32 that two groups of waves may share.
@pytest.mark.parametrize("shape", [9, 10, 11, 12])
@pytest.mark.parametrize("M,N,K", [(1, 1, 4), (63, 64, 32), (64, 65, 36), (65, 127, 64), (130, 513, 100), (70, 300, 2052)])
def test_gemm_f32_on_pieces(shape, M, N, K):
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
    # numbers whose pieces or sums leave bfloat16's range, and numbers that are none, come out as float32 makes them
    x[0] = torch.finfo(torch.float32).max
    w[0] = 1e-30
    out2 = torch.full((M, N), float("nan"), device="cuda")
    kernels.gemm_f32(x, w, out2, shape=shape)
    close(out2[0, 0], (x[0].double() * w[0].double()).sum().cpu(), 6e-6, "beyond bfloat16's largest")
    assert torch.equal(out2[1:, 1:], out[1:, 1:])
    x[0, K - 1], w[0, 0] = float("inf"), float("nan")
    kernels.gemm_f32(x, w, out2, shape=shape)
    assert not bool(torch.isfinite(out2[0]).any()) and bool(torch.isnan(out2[:, 0]).all())
    assert torch.equal(out2[1:, 1:], out[1:, 1:])


def test_gemm_f32_cut_in_three_by_its_plan():
    """301 rows over 4096 x 2048: 22, 22 and 20 slices of 32 k. The planes' sum, and what the norm that adds them makes of it;
    the same bound as above."""
    from tie_amd import kernels

    M, N, K = 301, 4096, 2048
    assert kernels.gemm_f32_splits(M, N, K) == 3
    x, w, base = rnd(M, K, seed=M), rnd(N, K, seed=N, scale=0.1), rnd(M, N, seed=7)
    want = plain.linear(x, w)
    planes = torch.full((3, M, N), float("nan"), device="cuda")
    kernels.gemm_f32(x.cuda(), w.cuda(), planes, splits=3)
    close(planes.sum(0), want, 6e-6, "three planes")
    weight, stream, normed = (1 + 0.1 * rnd(N, seed=3)).cuda(), base.cuda(), torch.full((M, N), float("nan"), device="cuda")
    kernels.add_partials(stream, planes, weight, 1e-6, normed)
    total = want.double() + base.double()
    close(stream, total, 6e-6, "the stream with three planes")
    close(normed, plain.rms_norm(total.float(), weight.cpu(), 1e-6), 6e-6, "its norm")


@pytest.mark.parametrize("shape", [9, 10, 11, 12])
def test_gemm_f32_on_pieces_takes_every_piece(shape):
    """x = 1 + 2^-11 + 2^-21 and w = 1 + 2^-10 + 2^-20, whose pieces are these powers, at one k of a row each, every k of two
    slices in turn. The six products of pieces that are taken sum to a float32 number; the others are below 2^-29. Without any
    one of the three smallest it would be off by 2^-21 or more, without the others by more than that."""
    from tie_amd import kernels

    M, N, K = 96, 130, 64
    x, w = torch.zeros(M, K), torch.zeros(N, K)
    x[torch.arange(M), torch.arange(M) % K] = 1 + 2.0 ** -11 + 2.0 ** -21
    w[torch.arange(N), torch.arange(N) % K] = 1 + 2.0 ** -10 + 2.0 ** -20
    out = torch.full((M, N), float("nan"), device="cuda")
    kernels.gemm_f32(x.cuda(), w.cuda(), out, shape=shape)
    assert float((out.cpu().to(F64) - x.to(F64) @ w.to(F64).T).abs().max()) <= 2.0 ** -23


@pytest.mark.parametrize("shape", [9, 10, 11, 12])
@pytest.mark.parametrize("down,up", [(100, 100), (112, 110), (115, 110), (126, 110), (140, 120), (148, 124), (70, -60)])
def test_gemm_f32_on_pieces_of_small_numbers(shape, down, up):
    """Numbers far below 1, subnormal ones among them, against numbers far above it, either way round: nothing of either is
    lost. A sum of 64 products is within 16 roundings, 2^-24 of the summed sizes each; results that are subnormal themselves
    are within one of their last bits."""
    from tie_amd import kernels

    M, N, K = 70, 130, 64
    small = rnd(N, K, seed=5) * 2.0 ** -min(down, 126) * 2.0 ** -max(0, down - 126)
    large = rnd(N, K, seed=6) * 2.0 ** up
    for x, w in ((small[:M], large), (large[:M], small)):
        want, size = [a @ b.T for a, b in ((x.to(F64), w.to(F64)), (x.to(F64).abs(), w.to(F64).abs()))]
        out = torch.full((M, N), float("nan"), device="cuda")
        kernels.gemm_f32(x.cuda(), w.cuda(), out, shape=shape)
        off = (out.cpu().to(F64) - want).abs()
        assert bool((off <= 16 * 2.0 ** -24 * size + 2.0 ** -149).all()), (down, up, float((off / size).max()))


@pytest.mark.parametrize("shape", [9, 10, 11, 12])
@pytest.mark.parametrize("K", [4, 32, 516, 2048])
def test_gemm_f32_on_pieces_is_no_further_off_than_float32_instructions(shape, K):
    """Root of the summed squares of the error against 64 bits, random signs: 0.4 to 0.7 of the other kernel's, which is 4e-8
    to 4e-7 of the result. Without any of the second-order products of pieces it would be 2.4e-6 and more."""
    from tie_amd import kernels

    x, w = rnd(130, K, seed=K).cuda(), rnd(256, K, seed=K + 1, scale=0.02).cuda()
    want = x.double() @ w.double().T

    def error(shape):
        out = torch.full((130, 256), float("nan"), device="cuda")
        kernels.gemm_f32(x, w, out, shape=shape)
        return float((out.double() - want).norm())

    assert error(shape) <= error(8)


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("M,I,K", [(5, 24, 200), (70, 136, 516)])
def test_gemm_f32_gated_on_pieces(M, I, K, activation):
    from tie_amd import kernels

    x, gate, up = rnd(M, K, seed=M), rnd(I, K, seed=2, scale=0.1), rnd(I, K, seed=3, scale=0.1)
    g, u = plain.linear(x, gate), plain.linear(x, up)
    act = g / (1 + torch.exp(-g)) if activation == "silu" else torch.nn.functional.gelu(g, approximate="tanh")
    w = kernels.interleave_gate_up(gate, up).cuda()
    for shape in (9, 10, 11, 12):
        out = torch.full((M, I), float("nan"), device="cuda")
        kernels.gemm_f32(x.cuda(), w, out, shape=shape, gated=1 + kernels.GATE_ACTIVATIONS[activation])
        close(out, act * u, 6e-6, f"gated product, shape {shape}")


def run(case, H, S, Dh, nsplit=1, **more):
    from tie_amd import kernels

    KVH = case["kc"].shape[1]
    new = (case["query_start"][1:] - case["query_start"][:-1]).tolist()
    q = case["q"]
    out = torch.full_like(q, float("nan"))
    part_o = torch.full((q.shape[0] * H * nsplit * Dh,), float("nan"), device="cuda")
    part_ml = torch.full((q.shape[0] * H * nsplit * 2,), float("nan"), device="cuda")
    kernels.attention_f32(q, case["kc"], case["vc"], out, case["query_start"], case["context_lens"], case["tables"],
                          kernels.attention_f32_tiles(new, H // KVH), H, Dh ** -0.5, nsplit=nsplit,
                          part_o=part_o if nsplit > 1 else None, part_ml=part_ml if nsplit > 1 else None, **more)
    return out


@pytest.mark.parametrize("nsplit", [1, 2, 16])
@pytest.mark.parametrize("H,KVH,Dh,bs", [(4, 2, 16, 16), (6, 2, 32, 16), (3, 1, 48, 32), (4, 4, 64, 16), (5, 5, 80, 16),
                                         (14, 2, 96, 64), (16, 1, 112, 16), (16, 8, 128, 16), (20, 1, 144, 16),
                                         (40, 2, 192, 16), (2, 1, 256, 16)])
def test_attention_f32_mixed_batch(H, KVH, Dh, bs, nsplit):
    # a whole prompt, a portion that continues a cached prefix, single decoded tokens, a one-token prompt
    case, S = attention_case(H, KVH, Dh, bs, lens_new=[13, 37, 1, 1, 1], lens_ctx=[13, 61, 40, 300, 1], seed=3)
    close(run(case, H, S, Dh, nsplit), case["want"], 1e-5, f"attention H={H} KVH={KVH} Dh={Dh}, {nsplit} shares")


@pytest.mark.parametrize("nsplit", [1, 3])
def test_attention_f32_many_sequences(nsplit):
    """More sequences than a wave has lanes, single tokens and portions mixed; then single tokens alone."""
    new = [1 + (i * 7) % 5 for i in range(70)]
    case, S = attention_case(4, 2, 32, 16, lens_new=new, lens_ctx=[n + (i * 13) % 90 for i, n in enumerate(new)], seed=4)
    close(run(case, 4, S, 32, nsplit), case["want"], 1e-5, "seventy sequences")
    case, S = attention_case(4, 2, 32, 16, lens_new=[1] * 70, lens_ctx=[1 + i for i in range(70)], seed=5)
    close(run(case, 4, S, 32, nsplit), case["want"], 1e-5, "seventy single tokens")


@pytest.mark.parametrize("nsplit", [1, 4])
@pytest.mark.parametrize("window", [1, 5, 16, 17, 100])
def test_attention_f32_window_edges(window, nsplit):
    case, S = attention_case(4, 2, 16, 16, lens_new=[9, 1, 20], lens_ctx=[30, 141, 20], seed=7, window=window)
    close(run(case, 4, S, 16, nsplit, window=window), case["want"], 1e-5, f"window {window}")


@pytest.mark.parametrize("more", [{"chunk": 1}, {"chunk": 24}, {"softcap": 5.0}, {"sinks": True}, {"chunk": 24, "sinks": True},
                                  {"window": 20, "softcap": 2.0, "sinks": True}])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("nsplit", [1, 5])
def test_attention_f32_against_the_generic_kernel(more, dtype, nsplit):
    """Chunks, caps, sinks and narrow pages: the same as the kernel that walks key by key, whose tests hold these."""
    from tie_amd import kernels

    H, KVH, Dh = 8, 2, 64
    case, S = attention_case(H, KVH, Dh, 16, lens_new=[33, 1, 1, 50], lens_ctx=[33, 200, 7, 90], seed=9)
    for name in ("kc", "vc"):
        case[name] = torch.nan_to_num(case[name].clamp(-6e4, 6e4).to(dtype))
    more = dict(more)
    if more.get("sinks"):
        more["sinks"] = rnd(H, seed=11).cuda()
    want = torch.empty_like(case["q"])
    kernels.paged_attention_generic(case["q"], case["kc"], case["vc"], want, case["query_start"], case["context_lens"],
                                    case["tables"], case["seq_of_row"], H, Dh ** -0.5, **more)
    # two float32 orders of the same sums of up to 200 terms
    close(run(case, H, S, Dh, nsplit, **more), want.cpu().to(F64), 4e-6, f"{more} over {dtype}")


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_attention_f32_values_that_are_no_numbers(bad):
    """A value that is no number reaches the rows that see its key, at every place of a tile, and no other row."""
    from tie_amd import kernels

    H, KVH, Dh, n = 4, 2, 32, 37
    for key in (0, 3, 16, 21, 36):
        case, S = attention_case(H, KVH, Dh, 16, lens_new=[n], lens_ctx=[n], seed=12)
        clean = run(case, H, S, Dh)
        page = int(case["tables"][0, key // 16])
        case["vc"][page, 1, 5, key % 16] = bad
        out = run(case, H, S, Dh).view(n, H, Dh)
        want = clean.view(n, H, Dh).clone()
        seen = ~torch.isfinite(out)
        expect = torch.zeros_like(seen)
        expect[key:, 2:, 5] = True                      # the heads of KV head 1, its sixth dimension, rows from the key on
        assert torch.equal(seen, expect), f"key {key}"
        close(out[~expect], want[~expect].cpu().to(F64), 2e-6, f"the other results, key {key}")


@pytest.mark.parametrize("nsplit", [1, 3])
def test_attention_f32_scores_of_minus_infinity(nsplit):
    """A key whose score is -inf weighs nothing beside any other, also where it is all a tile shows a row, or all that one
    wave of a workgroup or one share holds: the same as the kernel that walks key by key."""
    from tie_amd import kernels

    H, KVH, Dh, n = 4, 2, 32, 140
    for keys in ((0,), (16,), (31, 32), (48, 49, 50), tuple(range(64, 80)), tuple(range(1, 140))):
        case, S = attention_case(H, KVH, Dh, 16, lens_new=[n], lens_ctx=[n], seed=13)
        case["q"].view(n, H, Dh)[:, :, 2].abs_().add_(0.1)
        for key in keys:
            case["kc"][int(case["tables"][0, key // 16]), :, key % 16, 2] = -float("inf")
        want = torch.empty_like(case["q"])
        kernels.paged_attention_generic(case["q"], case["kc"], case["vc"], want, case["query_start"], case["context_lens"],
                                        case["tables"], case["seq_of_row"], H, Dh ** -0.5)
        out = run(case, H, S, Dh, nsplit)
        there = torch.isfinite(want)
        assert bool(there[1:].all()) and bool(there[0].all()) == (0 not in keys)     # row 0 sees key 0 alone
        assert torch.equal(torch.isfinite(out), there), f"keys {keys}"
        close(out[there], want[there].cpu().to(F64), 4e-6, f"keys {keys}")


def test_the_32_bit_path_takes_these_kernels():
    """The dispatchers: operands the kernels take go there (other results only by rounding), the others as before."""
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


# Few rows: lanes along K, 256 of it a load, so a sum is of 64 chains and the bound above holds as it is.
@pytest.mark.parametrize("shape", range(-3, 0))
@pytest.mark.parametrize("M,N,K", [(1, 16, 4), (1, 33, 256), (2, 7, 260), (3, 64, 1000), (4, 130, 2048), (4, 9, 2816),
                                   (3, 70, 516), (4, 48, 6148)])
def test_gemm_f32_few_rows(shape, M, N, K):
    from tie_amd import kernels

    x, w = rnd(M, K, seed=M), rnd(N, K, seed=N, scale=0.1)
    want = plain.linear(x, w)
    x, w = x.cuda(), w.cuda()
    out = torch.full((M + 1, N), float("nan"), device="cuda")
    kernels.gemm_f32(x, w, out[:M], shape=shape)
    close(out[:M], want, 6e-6, f"product {M}x{N}x{K}, shape {shape}")
    assert bool(out[M].isnan().all())                         # a shape's spare rows are not stored
    base = rnd(M, N, seed=7).cuda()
    acc = base.clone()
    kernels.gemm_f32(x, w, acc, accumulate=True, shape=shape)
    close(acc, want + base.cpu().to(F64), 6e-6, "added to what was there")
    good = out[:M].clone()
    x[M - 1, K - 1], w[N - 1, 0] = float("inf"), float("nan")
    kernels.gemm_f32(x, w, out[:M], shape=shape)
    bad = ~torch.isfinite(out[:M])
    assert bool(bad[M - 1].all()) and bool(bad[:, N - 1].all()) and int(bad.sum()) == M + N - 1
    assert torch.equal(out[:M - 1, :N - 1], good[:M - 1, :N - 1])
    with pytest.raises(kernels.InvalidArgument):
        kernels.gemm_f32(torch.zeros(5, K, device="cuda"), w, torch.empty(5, N, device="cuda"), shape=shape)


@pytest.mark.parametrize("shape", range(-3, 0))
@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
def test_gemm_f32_few_rows_gated(shape, activation):
    from tie_amd import kernels

    for M, I, K in ((1, 8, 64), (3, 24, 1028), (4, 40, 516)):
        x, gate, up = rnd(M, K, seed=M), rnd(I, K, seed=2, scale=0.1), rnd(I, K, seed=3, scale=0.1)
        g, u = plain.linear(x, gate), plain.linear(x, up)
        act = g / (1 + torch.exp(-g)) if activation == "silu" else torch.nn.functional.gelu(g, approximate="tanh")
        out = torch.full((M, I), float("nan"), device="cuda")
        kernels.gemm_f32(x.cuda(), kernels.interleave_gate_up(gate, up).cuda(), out, shape=shape,
                         gated=1 + kernels.GATE_ACTIVATIONS[activation])
        close(out, act * u, 6e-6, f"gated product {M}x{I}x{K}, shape {shape}")
