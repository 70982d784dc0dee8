"""Vosurax on the GPU against the plain implementation: each mechanism's kernel alone, then whole models under
every way of cutting the work, in float32 (tight) and bfloat16, and greedy generation through the engine."""

import copy
import json
import subprocess
import sys

import numpy as np
import pytest
import torch

import plain_vosurax as plain
import trace_helpers as th
from vosurax_fixtures import BLOCK_SIZE, CONFIGS, load_plain, write_model

pytestmark = pytest.mark.gpu
F64 = torch.float64


def rnd(*shape, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g, dtype=torch.float32) * scale


def close(got, want, rel, what=""):
    got, want = got.detach().cpu().to(F64), want.detach().cpu().to(F64)
    assert torch.isfinite(got).all(), f"{what}: non-finite values"
    err = float((got - want).abs().max() / want.abs().max().clamp_min(1e-30))
    assert err <= rel, f"{what}: relative error {err:.3e} > {rel:.0e}"


def i32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def scratch_memory(fill=float("nan")):
    """Scratch as the kernels are handed it: what nobody wrote is not zero."""
    held = {}

    def get(name, shape, dtype=torch.float32):
        key = (name, tuple(shape), dtype)
        if key not in held:
            t = torch.empty(tuple(shape), dtype=dtype, device="cuda")
            if dtype.is_floating_point:
                t.fill_(fill)
            held[key] = t
        return held[key]

    return get


def chunks_of(lengths, rows=64):
    from tie_amd import kernels

    class Batch:
        host_new_tokens, memo = list(lengths), {}

    return kernels.scan_chunks(Batch, "cuda", rows=rows, force=True)


def starts_of(lengths):
    starts = [0]
    for n in lengths:
        starts.append(starts[-1] + n)
    return starts


# ------------------------------------------------------------------------------------------- kernels alone
def memory_inputs(H, d, e, T, seed, gates):
    """Projection rows [q | k | v | g | i | f] and the gates' biases. ``gates``: "mixed", "forgetful" (states are lost at
    once), "keeping" (hardly anything is) or "far apart" (input gates between both ends of the cap)."""
    proj = rnd(T, H * (2 * d + 2 * e) + 2 * H, seed=seed)
    at = H * (2 * d + 2 * e)
    spread, f_bias = {"mixed": (2.0, 1.5), "forgetful": (3.0, -8.0), "keeping": (1.0, 9.0), "far apart": (25.0, 3.0)}[gates]
    proj[:, at:at + H] *= spread
    proj[:, at + H:] *= 2.0
    return proj, 0.5 * rnd(H, seed=seed + 1), f_bias + 0.3 * rnd(H, seed=seed + 2)


def plain_memory(proj, i_bias, f_bias, cap, H, d, e, states):
    """Outputs [T, H e] of one sequence's rows and the states they leave."""
    proj, T = proj.to(F64), proj.shape[0]
    q, k = (proj[:, i * H * d:(i + 1) * H * d].view(T, H, d) for i in (0, 1))
    v = proj[:, 2 * H * d:2 * H * d + H * e].view(T, H, e)
    at = H * (2 * d + 2 * e)
    li = plain.capped(proj[:, at:at + H] + i_bias.to(F64), cap)
    lf = torch.nn.functional.logsigmoid(plain.capped(proj[:, at + H:at + 2 * H] + f_bias.to(F64), cap))
    outs, left = [], []
    for h in range(H):
        o, s = plain.matrix_memory_scan(q[:, h] * d ** -0.5, k[:, h], v[:, h], li[:, h], lf[:, h], states[h])
        outs.append(o)
        left.append(s)
    return torch.cat(outs, 1), left


@pytest.mark.parametrize("gates", ["mixed", "forgetful", "keeping", "far apart"])
@pytest.mark.parametrize("way", ["walk", "chunks", "ragged chunks"])
@pytest.mark.parametrize("H,d,e", [(2, 8, 12), (3, 32, 64), (1, 9, 5), (2, 100, 130), (1, 200, 33), (1, 300, 40), (2, 64, 31)])
def test_the_matrix_memory(H, d, e, way, gates):
    """Three steps of sequences of unequal lengths through their slots, walked or in chunks; a neighbour's slot stays."""
    from tie_amd import kernels

    cap = 6.0
    tolerance = 4e-4 if gates == "far apart" else 5e-5      # denominators as small as exp(-cap) divide sums of order one
    slots, steps = [4, 0, 2], ([70, 1, 3], [1, 131, 64], [65, 33, 1])
    state = torch.zeros(5, H, d, e, device="cuda")
    norm_state = torch.zeros(5, *kernels.memory_norm_shape(H, d, e), device="cuda")
    state[1].fill_(7.0)
    norm_state[1].fill_(7.0)
    left = [[None] * H for _ in slots]
    for n, lengths in enumerate(steps):
        T = sum(lengths)
        proj, i_bias, f_bias = memory_inputs(H, d, e, T, 100 + n, gates)
        starts = starts_of(lengths)
        out = torch.full((T, H * e), float("nan"), device="cuda")
        chunks = None if way == "walk" else chunks_of(lengths, 64 if way == "chunks" else 37)
        kernels.matrix_memory_scan(proj.cuda(), out, state, norm_state, i32(starts), i32(slots), H * (2 * d + 2 * e),
                                   i_bias.cuda(), f_bias.cuda(), cap, len(slots), H, d, e, q_scale=d ** -0.5, chunks=chunks,
                                   scratch=scratch_memory())
        for j in range(len(slots)):
            want, left[j] = plain_memory(proj[starts[j]:starts[j + 1]], i_bias, f_bias, cap, H, d, e, left[j])
            close(out[starts[j]:starts[j + 1]], want, tolerance, f"step {n}, sequence {j}")
    for j, slot in enumerate(slots):
        for h, (S, nn, m) in enumerate(left[j]):
            close(state[slot, h], S, 3e-5, f"S of sequence {j}")
            for copy_ in norm_state[slot, h]:
                close(copy_[:d], nn, 3e-5, f"n of sequence {j}")
                assert abs(float(copy_[d]) - m) < 1e-5 * max(1.0, abs(m))
    assert bool((state[1] == 7.0).all()) and bool((norm_state[1] == 7.0).all()) and bool((state[3] == 0).all())


def test_a_memory_that_starts_low_stays_exact_over_many_chunks():
    """Strong forgetting: the sums of log gates grow to hundreds inside a chunk while only small differences count."""
    from tie_amd import kernels

    H, d, e, T = 1, 16, 16, 700
    proj, i_bias, f_bias = memory_inputs(H, d, e, T, 7, "forgetful")
    f_bias -= 30.0
    results = []
    for chunks in (None, chunks_of([T])):
        state, norm_state = torch.zeros(1, H, d, e, device="cuda"), torch.zeros(1, *kernels.memory_norm_shape(H, d, e), device="cuda")
        out = torch.empty(T, H * e, device="cuda")
        kernels.matrix_memory_scan(proj.cuda(), out, state, norm_state, i32([0, T]), i32([0]), H * (2 * d + 2 * e),
                                   i_bias.cuda(), f_bias.cuda(), 14.0, 1, H, d, e, q_scale=d ** -0.5, chunks=chunks,
                                   scratch=scratch_memory())
        results.append(out)
    want, _ = plain_memory(proj, i_bias, f_bias, 14.0, H, d, e, [None])
    for out, what in zip(results, ("walk", "chunks")):
        err = ((out.cpu().to(F64) - want).abs().amax(1) / want.abs().amax(1)).max()      # row by row: no row hides another
        assert float(err) < 2e-4, f"{what}: {float(err):.2e}"


@pytest.mark.parametrize("rot", [None, 2, 8, 1000])
@pytest.mark.parametrize("way", ["walk", "chunks", "ragged chunks"])
@pytest.mark.parametrize("H,d,e", [(3, 8, 12), (2, 64, 64), (1, 10, 5), (2, 128, 130), (1, 320, 36)])
def test_retention_rotated_and_scaled(H, d, e, way, rot):
    from tie_amd import kernels

    rot = None if rot is None else min(rot, d)
    decay = torch.tensor([0.99, 0.5, 1.0][:H])
    slots, steps = [1, 3], ([70, 1], [1, 131], [33, 64])
    state = torch.zeros(4, H, d, e, device="cuda")
    at, left = [0, 0], [[None] * H for _ in slots]
    inv_freq = (50.0 ** (-2.0 * torch.arange((rot or 2) // 2, dtype=F64) / (rot or 2))).float()
    for n, lengths in enumerate(steps):
        T, starts = sum(lengths), starts_of(lengths)
        proj = rnd(T, H * (2 * d + 2 * e) + 3, seed=200 + n)
        rotation = None
        if rot:
            positions = [p for j, c in enumerate(lengths) for p in range(at[j], at[j] + c)]
            angles = torch.empty(T, rot, device="cuda")
            kernels.rope_angles(i32(positions), inv_freq.cuda(), angles)
            rotation = (angles, rot)
        out = torch.full((T, H * e), float("nan"), device="cuda")
        chunks = None if way == "walk" else chunks_of(lengths, 64 if way == "chunks" else 29)
        kernels.decay_attention_scan(proj.clone().cuda(), out, state, i32(starts), i32(slots), decay.cuda(), len(slots), H, d, e,
                                     "none", chunks=chunks, scratch=scratch_memory(), q_scale=d ** -0.5, rotation=rotation)
        for j, c in enumerate(lengths):
            rows = proj[starts[j]:starts[j + 1]].to(F64)
            q, k = (rows[:, i * H * d:(i + 1) * H * d].view(c, H, d) for i in (0, 1))
            v = rows[:, 2 * H * d:2 * H * d + H * e].view(c, H, e)
            if rot:
                q, k = (plain.rotate(t, {"dims": rot, "base": 50.0}, at[j]) for t in (q, k))
            want = []
            for h in range(H):
                o, left[j][h] = plain.retention_scan(q[:, h], k[:, h] * d ** -0.5, v[:, h], float(decay[h]), left[j][h])
                want.append(o)
            close(out[starts[j]:starts[j + 1]], torch.cat(want, 1), 3e-5, f"step {n}, sequence {j}")
            at[j] += c


def test_heads_in_several_passes_where_the_chunks_memory_is_short(monkeypatch):
    from tie_amd import kernels

    H, d, e, lengths = 5, 24, 40, [150, 3, 70]
    T, starts = sum(lengths), starts_of(lengths)
    proj, i_bias, f_bias = memory_inputs(H, d, e, T, 11, "mixed")
    decay = torch.tensor([0.9, 0.99, 0.5, 1.0, 0.97]).cuda()
    results = []
    for limit in (1 << 30, 2 * 4 * (d * e + d) * chunks_of(lengths).count):
        monkeypatch.setattr(kernels, "CHUNK_STATE_SCRATCH_MAX", limit)
        state, norm_state = (rnd(3, *s, seed=5).cuda() for s in ((H, d, e), kernels.memory_norm_shape(H, d, e)))
        norm_state[:, :] = norm_state[:, :, :1]                     # copies that agree, as any step leaves them
        retained = rnd(3, H, d, e, seed=6).cuda()
        out, kept = torch.empty(T, H * e, device="cuda"), torch.empty(T, H * e, device="cuda")
        kernels.matrix_memory_scan(proj.cuda(), out, state, norm_state, i32(starts), i32([2, 0, 1]), H * (2 * d + 2 * e),
                                   i_bias.cuda(), f_bias.cuda(), 5.0, 3, H, d, e, chunks=chunks_of(lengths), scratch=scratch_memory())
        kernels.decay_attention_scan(proj.cuda(), kept, retained, i32(starts), i32([2, 0, 1]), decay, 3, H, d, e, "none",
                                     chunks=chunks_of(lengths), scratch=scratch_memory())
        results.append((out, state, norm_state, kept, retained))
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n", [30, 64, 101, 352, 2048, 5000, 9004])
def test_adding_normed_results_and_norming_the_sum(n):
    from tie_amd import kernels

    T = 7
    x, rows, planes = rnd(T, n, seed=n), rnd(T, n, seed=1, scale=3.0), rnd(5, T, n, seed=2)
    wa, wb, w = rnd(n, seed=3), rnd(n, seed=4), 1 + 0.2 * rnd(n, seed=5)
    eps = (1e-5, 0.3)

    def term(y, weight, e):
        return plain.over_rms(y.to(F64), e) * weight.to(F64)

    both = x.to(F64) + term(rows, wa, eps[0]) + term(planes.to(F64).sum(0), wb, eps[1])
    one = x.to(F64) + term(planes.to(F64).sum(0), wa, eps[1])
    for results, want in (([(rows.cuda(), wa.cuda(), eps[0]), (planes.cuda(), wb.cuda(), eps[1])], both),
                          ([(planes.cuda(), wa.cuda(), eps[1])], one)):
        xd = x.clone().cuda()
        kernels.add_normed_results(xd, results)
        close(xd, want, 2e-6, "the stream")
        for dtype, tolerance in ((torch.float32, 3e-6), (torch.bfloat16, 8e-3)):
            xd, out = x.clone().cuda(), torch.empty(T, n, dtype=dtype, device="cuda")
            kernels.add_normed_results(xd, results, norm=(w.cuda(), 1e-5, out))
            close(xd, want, 2e-6, "the stream beside a norm")
            close(out, plain.over_rms(want, 1e-5) * w.to(F64), tolerance, "the normed rows")


@pytest.mark.parametrize("n", [5, 64, 130, 2048])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gated_rows(n, dtype):
    from tie_amd import kernels

    rows, wide = rnd(9, n, seed=1).to(dtype), rnd(9, n + 7, seed=2, scale=4.0)
    got = rows.clone().cuda()
    kernels.gate_rows(got, wide.cuda()[:, 3:3 + n])
    close(got, rows.to(F64) * torch.sigmoid(wide[:, 3:3 + n].to(F64)), 1e-6 if dtype == torch.float32 else 8e-3)


@pytest.mark.parametrize("weights", ["a head", "all heads", None])
def test_the_gated_norm_of_every_head(weights):
    from tie_amd import kernels

    T, H, e, eps = 6, 3, 37, 0.2
    o, gate = rnd(T, H * e, seed=1, scale=2.0), rnd(T, H * e + 4, seed=2)
    w = {"a head": rnd(e, seed=3), "all heads": rnd(H * e, seed=3), None: None}[weights]
    full = torch.ones(H, e) if w is None else (w.expand(H, e) if w.numel() == e else w.view(H, e))
    for activation, f in (("sigmoid", torch.sigmoid), ("silu", torch.nn.functional.silu)):
        want = plain.over_rms(o.view(T, H, e).to(F64), eps) * full.to(F64) * f(gate[:, 4:].to(F64)).view(T, H, e)
        for dtype, tolerance in ((torch.float32, 2e-6), (torch.bfloat16, 8e-3)):
            out = torch.empty(T, H * e, dtype=dtype, device="cuda")
            kernels.grouped_gated_rms_norm(o.cuda(), w.cuda() if w is not None else None, eps, gate.cuda()[:, 4:], out, H,
                                           activation=activation)
            close(out, want.view(T, H * e), tolerance, f"{weights}, {activation}")


def test_gelu_in_both_forms():
    from tie_amd import kernels

    z = torch.cat([rnd(500, seed=1, scale=3.0), torch.tensor([-40.0, 40.0, 0.0])])
    for dtype, tolerance in ((torch.float32, 1e-6), (torch.bfloat16, 5e-3)):
        for form, f in (("tanh", plain.gelu_tanh), ("erf", torch.nn.functional.gelu)):
            out = torch.empty(z.numel(), dtype=dtype, device="cuda")
            kernels.gelu(z.cuda(), out, form=form)
            close(out, f(z.to(F64)), tolerance, form)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,E,top,F_,K,shared", [(3, 4, 2, 24, 64, 1), (70, 3, 2, 16, 40, 0), (300, 5, 1, 72, 96, 2), (700, 4, 3, 64, 128, 1),
                                                 (200, 2, 2, 9, 100, 3)])
def test_experts_weighted_on_their_input(T, E, top, F_, K, shared, dtype):
    """Routing by sigmoid scores with ungated shared experts behind the routed ones, then the experts' products."""
    from tie_amd import kernels

    h, z = rnd(T, K, seed=1).to(dtype), rnd(T, E, seed=9, scale=2.0)
    real = E + shared
    gate, up, down = (t.to(dtype) for t in (rnd(real, F_, K, seed=2, scale=0.3), rnd(real, F_, K, seed=3, scale=0.3),
                                            rnd(real, K, F_, seed=4, scale=0.3)))
    chosen, scores = plain.route(z.to(F64), top)
    want = torch.zeros(T, K, dtype=F64)
    for e in range(real):
        weight = (scores * (chosen == e)).sum(1, keepdim=True) if e < E else torch.ones(T, 1, dtype=F64)
        want += plain.expert(weight * h.to(F64), gate[e].to(F64), up[e].to(F64), down[e].to(F64))
    get, slots = scratch_memory(), top + shared
    tile = kernels.moe_tile_rows(dtype, dtype, K, F_, T * slots, real)
    ids, weights = get("ids", (T, slots), torch.int32), get("weights", (T, slots))
    rows = kernels.moe_route_align(z.cuda(), None, 1, 1, top, ids, weights, real, tile, get, scoring="sigmoid", shared=shared,
                                   shared_gated=False)
    close(weights, torch.cat([scores, torch.ones(T, shared, dtype=F64)], 1), 1e-6, "weights")
    act = get("act", (T * slots, F_), dtype)
    kernels.moe_gate_up(h.cuda(), gate.cuda(), up.cuda(), rows, act, slot_weights=weights)
    parts = get("parts", (T * slots, K))
    kernels.moe_down(act, down.cuda(), rows, parts)
    routed = kernels.RoutedParts(parts, rows.where, None, h.cuda())
    tolerance = 1e-5 if dtype == torch.float32 else 2e-2
    out = torch.zeros(T, K, device="cuda")
    kernels.moe_combine(routed, out)
    close(out, want, tolerance, "combined")
    x, w = rnd(T, K, seed=5), 1 + 0.1 * rnd(K, seed=6)
    xd, normed = x.clone().cuda(), torch.empty(T, K, device="cuda")
    kernels.add_results(xd, [routed], norm=("rms_norm", w.cuda(), 1e-5, normed))
    close(xd, x.to(F64) + want, tolerance, "added to the stream")
    close(normed, plain.over_rms(x.to(F64) + want, 1e-5) * w.to(F64), tolerance, "normed")
    xd = x.clone().cuda()
    kernels.norm_add_norm(routed, w.cuda(), 1e-5, xd)
    close(xd, x.to(F64) + plain.over_rms(want, 1e-5) * w.to(F64), tolerance, "normed on its way")


@pytest.mark.parametrize("tile", [16, 64, 128, 256])
@pytest.mark.parametrize("T,E,top,F_,K", [(3, 4, 2, 96, 128), (90, 3, 2, 128, 96), (600, 5, 1, 160, 224), (400, 40, 3, 96, 352)])
def test_packed_experts_weighted_on_their_input(T, E, top, F_, K, tile):
    from tie_amd import kernels

    bf = torch.bfloat16
    h, down = rnd(T, K, seed=1).to(bf), rnd(E, K, F_, seed=4, scale=0.2).to(bf)
    gate, up = rnd(E, F_, K, seed=2, scale=0.2).to(bf), rnd(E, F_, K, seed=3, scale=0.2).to(bf)
    g = torch.Generator().manual_seed(4)
    ids = torch.stack([torch.randperm(E - 1, generator=g)[:top] for _ in range(T)]).to(torch.int32)       # the last: nobody's
    weights = 0.2 + torch.rand(T, top, generator=g)
    want = torch.zeros(T, K, dtype=F64)
    for e in range(E):
        for slot in range(top):
            rows = torch.nonzero(ids[:, slot] == e).flatten()
            x = weights[rows, slot].to(F64)[:, None] * h[rows].to(F64)
            want.index_add_(0, rows, plain.expert(x, gate[e].to(F64), up[e].to(F64), down[e].to(F64)))
    up_packed, down_packed = kernels.pack_experts(gate.cuda(), up.cuda(), down.cuda())
    get = scratch_memory()
    rows = kernels.moe_align(ids.cuda(), E, tile, get)
    act = get("act", (T * top, F_), bf)
    kernels.moe_gate_up(h.cuda(), None, up_packed, rows, act, slot_weights=weights.cuda())
    parts = get("parts", (T * top, K))
    kernels.moe_down(act, down_packed, rows, parts)
    out = torch.zeros(T, K, device="cuda")
    kernels.moe_combine(kernels.RoutedParts(parts, rows.where, None, h.cuda()), out)
    close(out, want, 2e-2, f"packed experts in tiles of {tile}")


# ------------------------------------------------------------------------------------------- whole models
LENGTHS = {"A": [1, 23, 210, 37, 5], "B": [170, 2, 41, 90], "C": [33, 150, 8], "D": [12, 260, 3, 21, 9],
           "E": [150, 1, 66, 97], "F": [3, 140, 64, 20]}
TOLERANCE = {"float32": 6e-5, "bfloat16": 4e-2}        # of the largest logit; the queries are drawn wide
# A head's output is divided by its own size, so where a query meets the state at almost nothing the direction is rounding's:
# in bfloat16 a few positions of any request go there, and this share of them may lie above the tolerance, up to eight times.
LOOSE_SHARE = 0.06


@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    out = {}
    for name, config in CONFIGS.items():
        for dtype in ("float32", "bfloat16"):
            folder = tmp_path_factory.mktemp(f"vosurax_{name}_{dtype}")
            out[name, dtype] = write_model(folder, config, seed=41 + len(out), dtype=dtype)
    return out


def reference(folder, config, requests, streams=None):
    weights = load_plain(folder)
    out = {}
    for rid, toks in requests.items():
        logits, behind = plain.forward(config, weights, toks)
        out[rid] = logits.float()
        if streams is not None:
            streams[rid] = behind
    return out


def worst_error(got, want):
    worst = 0.0
    for rid, ref in want.items():
        mine = torch.stack([got[rid][p] for p in range(ref.shape[0])])
        worst = max(worst, float(((mine - ref).abs().amax(dim=1) / ref.abs().max()).max()))
    return worst


def check(got, want, tolerance, label):
    errors, where = [], []
    for rid, ref in want.items():
        rows = got[rid]
        assert sorted(rows) == list(range(ref.shape[0])), f"{label}: request {rid} misses positions"
        mine = torch.stack([rows[p] for p in range(ref.shape[0])])
        assert torch.isfinite(mine).all(), f"{label}: request {rid} has non-finite logits"
        errors.append((mine - ref).abs().amax(dim=1) / ref.abs().max())
        where += [(rid, p) for p in range(ref.shape[0])]
    err = torch.cat(errors)
    loose = tolerance >= 1e-2
    limit = 8 * tolerance if loose else tolerance
    bad = torch.nonzero(err > limit).flatten().tolist()
    assert not bad, (f"{label}: request {where[bad[0]][0]} first differs at position {where[bad[0]][1]} "
                     f"(relative error {float(err[bad[0]]):.3e}, allowed {limit:.0e}; {len(bad)} positions)")
    over = int((err > tolerance).sum())
    assert over <= max(1, LOOSE_SHARE * err.numel()), f"{label}: {over} of {err.numel()} positions above {tolerance:.0e}"
    print(f"[observed] {label}: {float(err.max()):.3e}, {over} of {err.numel()} above, median {float(err.median()):.1e}")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_every_way_of_cutting_the_work(folders, name, dtype):
    from tie_amd.engine.replay import TraceReplayer

    folder, config = folders[name, dtype], CONFIGS[name]
    requests = th.make_requests(config["vocab"], LENGTHS[name], seed=5)
    want = reference(folder, config, requests)
    bs = BLOCK_SIZE[name]
    biggest = max(th.round64(len(t)) for t in requests.values())

    def replayer(max_tokens):
        return TraceReplayer.from_folder(folder, dtype, max_tokens, block_size=bs, state_slots=4)

    results = {"whole": th.collect(replayer(biggest), th.whole(requests)),
               "prefill+decode": th.collect(replayer(biggest), th.prefill_then_decode(requests, tail=40)),
               "portions": th.collect(replayer(biggest), th.portions(requests)),
               "long portions": th.collect(replayer(biggest), th.portions(requests, sizes=(131, 2, 129))),
               "portions of two": th.collect(replayer(biggest), th.portions(requests, sizes=(2,))),
               "token by token": th.collect(replayer(biggest), th.portions(requests, sizes=(1,)))}
    for label, seed, sizes in (("mixed", 3, (13, 7, 2, 5, 3, 2, 9)), ("mixed, long portions", 4, (130, 2, 5))):
        steps, peak = th.mixed(requests, max_live=4, seed=seed, sizes=sizes)
        assert max(len(s["entries"]) for s in steps) >= 3
        rep = replayer(peak)
        results[label] = th.collect(rep, steps)
        assert rep.cache.all_free()                                   # every page and slot came back
    for label, got in results.items():
        check(got, want, TOLERANCE[dtype], f"{name}/{dtype}/{label}")
    if dtype == "float32":       # the ways of cutting agree with each other beyond what they owe the plain one
        for label in results:
            for rid in requests:
                a = torch.stack([results["whole"][rid][p] for p in range(len(requests[rid]))])
                b = torch.stack([results[label][rid][p] for p in range(len(requests[rid]))])
                assert float((a - b).abs().max() / a.abs().max()) < TOLERANCE["float32"], f"{name}: whole vs {label}, request {rid}"


def random_config(seed):
    """A model of random layers and sizes: every choice the reader knows is drawn, present or absent."""
    import random

    rng = random.Random(seed)
    pick = rng.choice
    width = pick([40, 64, 72, 96, 128])

    def mixer():
        if rng.random() < 0.4:
            d, heads = pick([4, 8, 16, 24, 48]), pick([1, 2, 3, 5])
            m = {"heads": heads, "dim": d, "decay": [pick([0.5, 0.9, 0.99, 1.0, 0.999]) for _ in range(heads)],
                 "rot": {"base": pick([50.0, 1000.0, 500000.0])}}
            if rng.random() < 0.7:
                m["vdim"] = pick([d, 8, 20, 64])
            if rng.random() < 0.7:
                m["rot"]["dims"] = pick([d, d // 2])
            return {"type": "retention", "mixer": m}
        kv, dim, mem = pick([1, 2, 3]), pick([8, 12, 16, 32, 48]), pick([8, 16, 20, 64])
        left = {"heads": kv * pick([1, 2, 4]), "kv_heads": kv, "dim": dim, "scale": rng.uniform(0.1, 0.4)}
        if rng.random() < 0.7:
            left["vdim"] = pick([dim, 8, 20, 64])
        if rng.random() < 0.8:
            left["mask"] = {"size": pick([5, 16, 40, 64, 100])}
        right = {"heads": pick([1, 2, 3]), "dim": mem, "vdim": pick([mem, 8, 24, 70]), "gate_cap": pick([1.0, 5.0, 15.0])}
        return {"type": "parallel", "mixer": {"left": left, "right": right}}

    def mlp():
        r = rng.random()
        if r < 0.2:
            return None
        if r < 0.5:
            return {"kind": "dense", "ff": pick([16, 40, 96, 33])}
        experts = pick([1, 2, 4, 7, 10])
        m = {"kind": "moe", "expert": {"ff": pick([8, 16, 24, 96, 9])},
             "router": {"experts": experts, "top": rng.randint(1, min(experts, 5))}}
        if rng.random() < 0.7:
            m["shared"] = {"ff": pick([8, 24, 50, 96])}
        return m

    n = rng.randint(1, 5)
    config = {"architecture": "Vosurax", "vocab": pick([50, 97, 200]), "width": width,
              "norm": {"eps": pick([1e-6, 1e-5, 1e-4])}, "layers": [{**mixer(), "mlp": mlp()} for _ in range(n)]}
    if rng.random() < 0.7:
        start = rng.randrange(n)
        config["loop"] = {"start": start, "stop": rng.randint(start + 1, n), "times": rng.randint(1, 3)}
    return config, pick([4, 8, 16, 32])


@pytest.mark.parametrize("dtype,seed", [("float32", s) for s in range(12)] + [("bfloat16", s) for s in (1, 4, 7, 10)])
def test_models_of_random_layers_and_sizes(tmp_path, seed, dtype):
    from tie_amd.engine.replay import TraceReplayer

    config, bs = random_config(seed)
    folder = write_model(tmp_path / "model", config, seed=100 + seed, dtype=dtype)
    requests = th.make_requests(config["vocab"], [155, 3, 41, 1, 58], seed=seed)
    want = reference(folder, config, requests)
    biggest = max(th.round64(len(t)) for t in requests.values())
    results = {"whole": th.collect(TraceReplayer.from_folder(folder, dtype, biggest, block_size=bs), th.whole(requests)),
               "prefill+decode": th.collect(TraceReplayer.from_folder(folder, dtype, biggest, block_size=bs),
                                            th.prefill_then_decode(requests, tail=35))}
    steps, peak = th.mixed(requests, max_live=4, seed=seed)
    rep = TraceReplayer.from_folder(folder, dtype, max(peak, bs), block_size=bs)
    results["mixed"] = th.collect(rep, steps)
    assert rep.cache.all_free()
    for label, got in results.items():
        check(got, want, TOLERANCE[dtype], f"random model {seed}/{dtype}/{label}: {json.dumps(config)}")


@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_the_stream_after_every_layer_run(folders, name):
    from tie_amd.engine.replay import TraceReplayer

    folder, config = folders[name, "float32"], CONFIGS[name]
    requests = th.make_requests(config["vocab"], [29], seed=8)
    streams = {}
    reference(folder, config, requests, streams)
    rep = TraceReplayer.from_folder(folder, "float32", 64, block_size=BLOCK_SIZE[name])
    seen = []
    rep.model.layer_hook = lambda index, x: seen.append(x.detach().double().cpu().clone())
    th.collect(rep, th.whole(requests))
    assert len(seen) == len(plain.run_order(config))
    for i, (mine, ref) in enumerate(zip(seen, streams["r0"])):
        close(mine, ref, 2e-5, f"{name}: the stream after run {i}")


@pytest.mark.parametrize("name,entries", [("D", 2), ("F", 2)])
def test_layers_of_one_shape_run_from_one_launch_list(folders, name, entries):
    """What a layer leaves for the next one's first pass carries over, and so does what stays inside a layer."""
    from tie_amd.engine.replay import TraceReplayer

    for dtype in ("float32", "bfloat16"):
        folder, config = folders[name, dtype], CONFIGS[name]
        requests = th.make_requests(config["vocab"], [150, 47], seed=18)
        want = reference(folder, config, requests)
        got = []
        for replay in (True, False):
            rep = TraceReplayer.from_folder(folder, dtype, 256, block_size=BLOCK_SIZE[name])
            rep.model.replay_layers = replay
            got.append(th.collect(rep, th.whole(requests)))
            assert rep.model.layers_replayed == (2 * entries if replay else 0)
            check(got[-1], want, TOLERANCE[dtype], f"launch lists {replay}")
        for rid, toks in requests.items():
            assert all(torch.equal(got[0][rid][p], got[1][rid][p]) for p in range(len(toks)))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("layers", [6, 7])
def test_norms_behind_two_mixers_keep_their_layers_weights(tmp_path, layers, dtype):
    """Layers of one shape without feed-forwards: what a layer leaves for the next one's first pass reads that layer's own
    norms, in steps of few rows and of many, the last layer's as well: the bits of a run of every layer's own code."""
    from tie_amd.engine.replay import TraceReplayer

    config = dict(CONFIGS["D"], layers=[dict(CONFIGS["D"]["layers"][0], mlp=None)] * layers)
    folder = write_model(tmp_path / "m", config, 23, dtype)
    requests = th.make_requests(config["vocab"], [5, 40], seed=24)
    want = reference(folder, config, requests)
    for rid, tokens in requests.items():
        got = []
        for replay in (True, False):
            rep = TraceReplayer.from_folder(folder, dtype, 256, block_size=16)
            rep.model.replay_layers = replay
            got.append(th.collect(rep, th.whole({rid: tokens})))
        check(got[0], {rid: want[rid]}, TOLERANCE[dtype], f"{layers} layers, {len(tokens)} rows")
        assert all(torch.equal(got[0][rid][p], got[1][rid][p]) for p in range(len(tokens)))


def test_a_fault_of_one_position_or_one_term_would_show(folders):
    """The engine agrees with the plain model, and the plain model with one mechanism slightly off does not agree
    with the engine by a wide margin."""
    from tie_amd.engine.replay import TraceReplayer

    folder, config = folders["A", "float32"], CONFIGS["A"]
    requests = th.make_requests(config["vocab"], [48, 71], seed=21)
    got = th.collect(TraceReplayer.from_folder(folder, "float32", 128, block_size=BLOCK_SIZE["A"]),
                     th.prefill_then_decode(requests, tail=20))
    weights = load_plain(folder)
    assert worst_error(got, reference(folder, config, requests)) < TOLERANCE["float32"]

    def off(label, config_change=None, weight_change=None):
        cfg, w = copy.deepcopy(config), dict(weights)
        if config_change:
            config_change(cfg)
        if weight_change:
            weight_change(w)
        err = worst_error(got, {rid: plain.forward(cfg, w, toks)[0].float() for rid, toks in requests.items()})
        print(f"[observed] {label}: {err:.3e}")
        assert err > 50 * TOLERANCE["float32"], f"{label} does not show in the logits ({err:.3e})"

    layer = lambda c, i: c["layers"][i]                                              # noqa: E731

    def drop(name, factor=0.0):
        return lambda w: w.__setitem__(name, w[name] * factor)

    def shift(name, dim=0):
        return lambda w: w.__setitem__(name, torch.roll(w[name], 1, dim))

    off("one pass fewer", lambda c: c["loop"].update(times=2))
    off("a loop one layer longer", lambda c: c["loop"].update(stop=4))
    off("the passes' vectors in another order", None, shift("loop.step"))
    off("no vector before the first pass", None,
        lambda w: w.__setitem__("loop.step", torch.cat([w["loop.step"][:1] * 0, w["loop.step"][1:]])))
    off("chunks one position longer", lambda c: layer(c, 0)["mixer"]["left"]["mask"].update(size=20))
    off("chunks one position shorter", lambda c: layer(c, 2)["mixer"]["left"]["mask"].update(size=32))
    off("no chunks", lambda c: layer(c, 3)["mixer"]["left"].pop("mask"))
    off("another scale", lambda c: layer(c, 0)["mixer"]["left"].update(scale=0.32))
    off("a gate cap", lambda c: layer(c, 0)["mixer"]["right"].update(gate_cap=4.5))
    off("a query without its bias", None, drop("l0.mix.left.q.b"))
    off("a key without its bias", None, drop("l0.mix.left.k.b"))
    off("a value without its bias", None, drop("l0.mix.left.v.b"))
    off("an attention gate of the wrong heads", None, shift("l0.mix.left.g"))
    off("a key norm off by one", None, shift("l0.mix.left.k.norm"))
    off("input gates of the wrong heads", None, shift("l0.mix.right.i"))
    off("a forget gate without its bias", None, drop("l2.mix.right.f.b"))
    off("an input gate without its bias", None, drop("l2.mix.right.i.b"))
    off("the memory's norm off by one", None, shift("l3.mix.right.norm"))
    off("the memory's gate of the wrong heads", None, shift("l3.mix.right.g"))
    off("the branches' norms swapped", None, lambda w: w.update(
        {"l2.mix.left.out": w["l2.mix.right.out"] + 0, "l2.mix.right.out": w["l2.mix.left.out"] + 0}))
    off("the whole head turned", lambda c: layer(c, 1)["mixer"]["rot"].update(dims=16))
    off("another base", lambda c: layer(c, 4)["mixer"]["rot"].update(base=50000.0))
    off("another decay", lambda c: layer(c, 1)["mixer"]["decay"].__setitem__(0, 0.91))
    off("decays of the wrong heads", lambda c: layer(c, 1)["mixer"]["decay"].reverse())
    off("retention gates of the wrong heads", None, shift("l1.mix.g"))
    off("one expert fewer", lambda c: layer(c, 1)["mlp"]["router"].update(top=1))
    off("one expert more", lambda c: layer(c, 3)["mlp"]["router"].update(top=4))
    off("no shared expert", lambda c: layer(c, 1)["mlp"].pop("shared"))
    off("a norm's weight", None, drop("l4.norm2", 2.0))
    off("no feed-forward", lambda c: layer(c, 4).update(mlp=None))


def far_model(tmp_path, chunk):
    """One layer whose attention, in chunks of ``chunk`` positions, lets token 49 in a prompt alone answer the query of
    token 48; the memory beside it is silent."""
    config = {"architecture": "Vosurax", "vocab": 50, "width": 32, "norm": {"eps": 1e-5},
              "layers": [{"type": "parallel", "mlp": None,
                          "mixer": {"left": {"heads": 2, "kv_heads": 1, "dim": 16, "vdim": 8, "scale": 3.0, "mask": {"size": chunk}},
                                    "right": {"heads": 1, "dim": 8, "vdim": 8, "gate_cap": 5.0}}}]}

    def point(tensors):
        w = {k: v.to(F64) for k, v in tensors.items()}
        for name in ("q.b", "k.b", "v.b"):
            tensors[f"l0.mix.left.{name}"].zero_()
        for name in ("q.norm", "k.norm"):
            tensors[f"l0.mix.left.{name}"].fill_(1.0)
        tensors["l0.mix.right.out"].zero_()
        rows = plain.stream_norm(w["embed"], w["l0.norm1"], 1e-5)
        key = w["l0.mix.left.k"] @ rows[49]
        q = key[:, None] * rows[48] / (rows[48] @ rows[48])
        tensors["l0.mix.left.q"] = torch.cat([q, q]).float()
        tensors["l0.mix.left.out"] *= 20.0

    folder = write_model(tmp_path / f"far{chunk}", config, seed=77, dtype="float32", change=point)
    return config, folder


@pytest.mark.parametrize("chunk", [400, 130, 64, 50])
def test_a_far_key_decides_a_token_inside_its_chunk_only(tmp_path, chunk):
    """The answering key at the first position, on both sides of pages' and chunks' borders, far back and just before the
    query; asked for by a decoded token, by the last token of a whole prompt and at the end and the start of a portion."""
    from tie_amd.engine.replay import TraceReplayer

    config, folder = far_model(tmp_path, chunk)
    weights = load_plain(folder)
    n = 397
    base = torch.randint(0, 48, (n,), generator=torch.Generator().manual_seed(3)).tolist()
    base[-1] = 48
    edge = (n - 1) // chunk * chunk                                       # the first position the last token sees
    without = plain.forward(config, weights, base)[0][-1].float()
    for place in sorted({0, 1, 15, 16, 47, 48, 255, 256, edge - 1, edge, edge + 1, n - 3, n - 2} - {-1}):
        tokens = list(base)
        tokens[place] = 49
        full = plain.forward(config, weights, tokens)[0][-1].float()
        decides = float((without - full).abs().max() / full.abs().max()) > 0.05
        assert decides == (place >= edge), f"the key at {place}"
        rep = TraceReplayer.from_folder(folder, "float32", 448, block_size=16)
        for cuts in ([n], [n - 1, n], [384, n], [100, n - 2, n], [16, 17, 300, n - 1, n], [edge + 1, n], [max(edge, 1), n]):
            steps, at = [], 0
            for cut in sorted(set(cuts)):
                steps.append({"step": len(steps), "entries": [{"id": "a", "tokens": tokens[at:cut],
                                                               "want": [cut - at - 1] if cut == n else []}],
                              "end": ["a"] if cut == n else []})
                at = cut
            for step in steps:
                logits = rep.run_step(step)
            err = float((logits.float().cpu()[0] - full).abs().max() / full.abs().max())
            assert err < TOLERANCE["float32"], f"key at {place}, cut at {cuts}: {err:.3e}"
        assert rep.cache.all_free()


@pytest.mark.parametrize("kind", ["parallel", "retention"])
def test_a_state_remembers_the_first_token_through_every_cut(tmp_path, kind):
    """One layer that hardly forgets: the last token's logits still know the first token, through long decoding and
    chunk borders; a state lost at any cut would show. Run twice in a row, so that two passes' states must stay apart."""
    from tie_amd.engine.replay import TraceReplayer

    mixer = {"heads": 2, "dim": 24, "vdim": 40, "decay": [1.0, 0.9999], "rot": {"base": 1e6, "dims": 2}} if kind == "retention" else \
        {"left": {"heads": 1, "kv_heads": 1, "dim": 8, "vdim": 8, "scale": 0.3, "mask": {"size": 3}},
         "right": {"heads": 2, "dim": 24, "vdim": 40, "gate_cap": 15.0}}
    config = {"architecture": "Vosurax", "vocab": 60, "width": 48, "norm": {"eps": 1e-5},
              "loop": {"start": 0, "stop": 1, "times": 2}, "layers": [{"type": kind, "mlp": None, "mixer": mixer}]}

    def remember(tensors):
        if kind == "parallel":
            tensors["l0.mix.right.f"].zero_()
            tensors["l0.mix.right.f.b"].fill_(14.0)
            tensors["l0.mix.left.out"].zero_()

    folder = write_model(tmp_path / "state", config, seed=5, dtype="float32", change=remember)
    weights = load_plain(folder)
    tokens = torch.randint(1, 60, (330,), generator=torch.Generator().manual_seed(8)).tolist()
    full = plain.forward(config, weights, tokens)[0].float()
    other = plain.forward(config, weights, [(tokens[0] + 7) % 60] + tokens[1:])[0].float()
    assert float((other[-1] - full[-1]).abs().max() / full.abs().max()) > 30 * TOLERANCE["float32"]
    want = {"a": full}
    for sizes in ((330,), (64,), (63, 1), (129, 2), (65, 130), (128, 1), (2, 150), (1,)):
        rep = TraceReplayer.from_folder(folder, "float32", 384, block_size=16)
        got = th.collect(rep, th.portions({"a": tokens}, sizes=sizes))
        check(got, want, TOLERANCE["float32"], f"portions of {sizes}")


def test_the_first_tokens_start_from_zeros(folders):
    """The memory's running maximum starts at 0 and the floor under its denominator counts at the start of a sequence."""
    from tie_amd.engine.replay import TraceReplayer

    for name in ("A", "C", "F"):
        folder, config = folders[name, "float32"], CONFIGS[name]
        requests = th.make_requests(config["vocab"], [1, 2, 3, 4], seed=50)
        want = reference(folder, config, requests)
        for steps in (th.whole(requests), th.portions(requests, sizes=(1,)), th.mixed(requests, tail=1, sizes=(2, 1))[0]):
            rep = TraceReplayer.from_folder(folder, "float32", 256, block_size=BLOCK_SIZE[name])
            check(th.collect(rep, steps), want, TOLERANCE["float32"], f"{name}: first tokens")


def test_long_decoding_with_pages_and_slots_used_again(folders):
    """Two requests decode 150 tokens each side by side, then others run in the pages and slots they left."""
    from tie_amd.engine.replay import TraceReplayer

    for dtype in ("float32", "bfloat16"):
        folder, config = folders["A", dtype], CONFIGS["A"]
        requests = th.make_requests(config["vocab"], [170, 165, 60, 140], seed=9)
        want = reference(folder, config, requests)
        steps = [{"step": 0, "entries": [{"id": r, "tokens": requests[r][:20 - i], "want": list(range(20 - i))}
                                        for i, r in enumerate(("r0", "r1"))], "end": []}]
        at = {"r0": 20, "r1": 19}
        while at:
            entries = [{"id": r, "tokens": [requests[r][p]], "want": [0]} for r, p in at.items()]
            at = {r: p + 1 for r, p in at.items()}
            ended = [r for r, p in at.items() if p == len(requests[r])]
            steps.append({"step": len(steps), "entries": entries, "end": ended})
            for r in ended:
                del at[r]
        for r in ("r2", "r3"):
            steps.append({"step": len(steps), "entries": [{"id": r, "tokens": requests[r], "want": list(range(len(requests[r])))}],
                          "end": [r]})
        rep = TraceReplayer.from_folder(folder, dtype, 384, block_size=4, state_slots=2)
        got = th.collect(rep, steps)
        assert rep.cache.all_free()
        check(got, want, TOLERANCE[dtype], f"long decoding, {dtype}")


def test_state_slots_are_cleared_when_they_are_used_again(folders):
    """Six requests through two state slots, one after another and side by side: every request starts from zeros,
    whatever the slot held."""
    from tie_amd.engine.replay import TraceReplayer

    for name in ("E", "F"):
        folder, config = folders[name, "float32"], CONFIGS[name]
        requests = th.make_requests(config["vocab"], [19, 30, 1, 135, 7, 22], seed=30)
        want = reference(folder, config, requests)
        steps, peak = th.mixed(requests, max_live=2, seed=6)
        rep = TraceReplayer.from_folder(folder, "float32", peak, block_size=BLOCK_SIZE[name], state_slots=2)
        got = th.collect(rep, steps)
        assert rep.cache.all_free()
        check(got, want, TOLERANCE["float32"], "slots used again")


def test_a_batch_gives_what_each_request_gives_alone(folders):
    """Unequal requests in one step, a long portion (its recurrences in chunks) beside single decoded tokens."""
    from tie_amd.engine.replay import TraceReplayer

    folder, config = folders["D", "float32"], CONFIGS["D"]
    requests = th.make_requests(config["vocab"], [200, 40, 3, 90], seed=33)
    want = reference(folder, config, requests)
    rep = TraceReplayer.from_folder(folder, "float32", 512, block_size=16)
    cuts = {"r0": [0, 20, 180, 199, 200], "r1": [0, 38, 39, 40, 40], "r2": [0, 1, 2, 3, 3], "r3": [0, 2, 3, 60, 90]}
    steps = []
    for i in range(4):
        entries = [{"id": r, "tokens": requests[r][c[i]:c[i + 1]], "want": list(range(c[i + 1] - c[i]))}
                   for r, c in cuts.items() if c[i + 1] > c[i]]
        steps.append({"step": i, "entries": entries, "end": [r for r, c in cuts.items()
                                                             if c[i] < len(requests[r]) == c[i + 1]]})
    check(th.collect(rep, steps), want, TOLERANCE["float32"], "a batch of unequal requests")
    assert rep.cache.all_free()


@pytest.mark.parametrize("name", ["A", "B", "D", "F"])
def test_decode_steps_replayed_from_recordings_give_the_eager_logits(folders, name):
    """bfloat16 decode-only steps are recorded into HIP graphs and replayed; every replay against the eager engine."""
    from tie_amd.engine.replay import TraceReplayer

    folder, config = folders[name, "bfloat16"], CONFIGS[name]
    requests = th.make_requests(config["vocab"], [50, 41, 47], seed=10)
    steps, peak = th.mixed(requests, max_live=3, seed=4, tail=30)
    eager = TraceReplayer.from_folder(folder, "bfloat16", peak, block_size=BLOCK_SIZE[name], use_graphs=False)
    recorded = TraceReplayer.from_folder(folder, "bfloat16", peak, block_size=BLOCK_SIZE[name])
    assert recorded.runner.use_graphs
    a, b = th.collect(eager, steps), th.collect(recorded, steps)
    assert recorded.runner.graph_replays > 10
    for rid, toks in requests.items():
        for p in range(len(toks)):
            assert torch.equal(a[rid][p], b[rid][p]), f"request {rid}, position {p}"


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["A", "B", "F"])
def test_greedy_generation_through_the_engine(folders, name, dtype):
    """The engine's own entry point and scheduler: several requests at once, prompts in portions, a small pool."""
    import tie_amd

    folder, config = folders[name, dtype], CONFIGS[name]
    weights = load_plain(folder)
    prompts = list(th.make_requests(config["vocab"], [7, 19, 3, 30], seed=12).values())
    new = 10
    engine = tie_amd.create_engine(folder, dtype=dtype, kv_blocks=64, block_size=BLOCK_SIZE[name], max_seqs=3,
                                   max_tokens_per_step=16, prefill_chunk=8)
    ids = [engine.add_request(p, tie_amd.SamplingParams(max_tokens=new)) for p in prompts]
    while engine.has_work():
        engine.step()
    for sid, prompt in zip(ids, prompts):
        generated = list(engine.sequence(sid).generated)
        assert len(generated) == new
        tokens = list(prompt)
        for i, token in enumerate(generated):       # every generated token is the plain model's best, or ties it
            logits = plain.forward(config, weights, tokens)[0][-1]
            best = float(logits.max())
            margin = 1e-4 * float(logits.abs().max()) if dtype == "float32" else 0.05 * float(logits.abs().max())
            assert float(logits[token]) >= best - margin, f"request {sid}: token {i} is not the plain model's choice"
            tokens.append(token)


def test_the_command_line_generates_the_plain_models_tokens(folders):
    from conftest import ROOT

    folder, config = folders["A", "float32"], CONFIGS["A"]
    weights = load_plain(folder)
    prompt = list(th.make_requests(config["vocab"], [11], seed=14).values())[0]
    tokens = list(prompt)
    for _ in range(6):
        tokens.append(int(plain.forward(config, weights, tokens)[0][-1].argmax()))
    proc = subprocess.run([sys.executable, str(ROOT / "bin" / "tie"), "generate", "-m", folder, "-p",
                           ",".join(map(str, prompt)), "--temp", "0", "--max-tokens", "6", "--dtype", "float32",
                           "--kv-mem", "16M"], capture_output=True, text=True, timeout=600)
    assert proc.returncode == 0, proc.stderr[-2000:]
    assert [int(t) for t in proc.stdout.split()] == tokens[len(prompt):]


def test_the_trace_program_runs_the_design(folders, tmp_path):
    """JSON lines in, .f32 files and 'done' lines out; four slots, pages used again."""
    from conftest import ROOT

    folder, config = folders["B", "float32"], CONFIGS["B"]
    requests = th.make_requests(config["vocab"], [23, 140, 9, 31, 17], seed=2)
    steps, peak = th.mixed(requests, max_live=4, seed=1)
    out = tmp_path / "out"
    proc = subprocess.run([sys.executable, str(ROOT / "bin" / "trace_run"), "--model", folder, "--dtype", "float32",
                           "--out", str(out), "--max-tokens", str(peak)],
                          input="".join(json.dumps(s) + "\n" for s in steps), capture_output=True, text=True, timeout=600)
    assert proc.returncode == 0, proc.stderr[-2000:]
    assert [line for line in proc.stdout.splitlines() if line.startswith("done")] == [f"done {s['step']}" for s in steps]
    want = reference(folder, config, requests)
    position = {}
    for s in steps:
        data = np.fromfile(out / f"{s['step']}.f32", dtype="<f4").reshape(-1, config["vocab"])
        r = 0
        for e in s["entries"]:
            start = position.get(e["id"], 0)
            for w in e["want"]:
                ref = want[e["id"]][start + w]
                assert float(np.abs(data[r] - ref.numpy()).max() / ref.abs().max()) < TOLERANCE["float32"]
                r += 1
            position[e["id"]] = start + len(e["tokens"])
        assert r == data.shape[0]
