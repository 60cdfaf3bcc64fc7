"""GPU parity of the grouped GEMMs' row tiles at their edges.

Experts get exact row counts around the tile heights (32, 64, 128 and 256
rows) at averages on both sides of the rules that choose a launch: 256-row
tiles with 128-row remainders, or tiles of at most 128 rows alone (forward:
weight-streaming tiles). Each case asserts the launch that it is meant for. Bounds: the layer
bound of test_gpu_layer.py forward, the per-gradient bounds of test_gpu_backward.py
for training (the oracle rounds at the same points, so only fp32 sums in
another order and their bf16 roundings differ).
"""

import numpy as np
import pytest
import torch

from mirai_amd import _native as nat
from mirai_amd import workloads as wl
from oracle import codec
from oracle import layer as olayer

from helpers import (assert_layer_close, build_module, mixed_rank_factors, oracle_loras,
                     oracle_weights)

pytestmark = pytest.mark.gpu


def exact_routes(counts, seed):
    """Top-1 routes giving expert e exactly counts[e] rows, in a shuffled order."""
    rng = np.random.default_rng(seed)
    idx = rng.permutation(np.repeat(np.arange(len(counts)), counts)).reshape(-1, 1)
    scores = (rng.random(idx.shape) + 0.5).astype(np.float32)
    return torch.from_numpy(idx), torch.from_numpy(scores)


def workload(fmt, counts, d=256, f=384, r=16):
    return wl.Workload(f"rows_{fmt}", 12, int(sum(counts)), d, f, len(counts), 1, r, 16.0, fmt,
                       torch.bfloat16)


FORMATS = {"nf4": nat.FMT_NF4, "int8": nat.FMT_INT8, "bf16": nat.FMT_BF16}


def launches(fmt, counts, *ks, backward=False):
    """The launches of GEMMs over K = each of ks with these rows per expert."""
    lib = nat.load_library()
    return {lib.mx_gemm_launch(FORMATS[fmt], int(backward), k, sum(counts), len(counts))
            for k in ks}


# Averages of 147, 33 and 31.
COUNTS = {
    "tall": (1, 127, 128, 129, 255, 256, 257, 20),
    "few": (0, 0, 129, 1, 2, 0, 128, 4),
    "below": (0, 0, 129, 0, 0, 0, 119, 0),
}
# Forward, averages on the line and just below it: 48 (NF4, INT8), 112 (bf16), and
# 256 where K is at most 512.
LINES = {
    48: (129, 1, 2, 128, 4, 120, 0, 0),
    112: (257, 129, 128, 1, 255, 126, 0, 0),
    256: (513, 257, 129, 385, 256, 255, 128, 125),
}


def _forward_case(fmt, counts, d, f):
    w = workload(fmt, counts, d=d, f=f)
    idx, scores = exact_routes(counts, 5)
    dense, lora, x = wl.dense_weights(w), wl.lora_factors(w), wl.tokens(w)
    m = build_module(w, dense, lora)
    with torch.no_grad():
        out = m.run_direct_routed(x.cuda(), scores.cuda(), idx.cuda())
    ref = olayer.layer_forward(x, scores, idx, oracle_weights(w, dense), oracle_loras(w, lora),
                               w.experts)
    assert_layer_close(out.cpu(), ref)


@pytest.mark.parametrize("fmt", list(FORMATS))
@pytest.mark.parametrize("case", list(COUNTS))
def test_rows_around_the_tile_heights(case, fmt):
    counts = COUNTS[case]
    kind = nat.LAUNCH_DUAL if case == "tall" else nat.LAUNCH_STREAM
    assert launches(fmt, counts, 640, 768) == {kind}
    _forward_case(fmt, counts, 640, 768)


@pytest.mark.parametrize("fmt,line,d,f", [
    ("nf4", 48, 640, 768), ("int8", 48, 640, 768), ("bf16", 112, 640, 768),
    ("nf4", 256, 256, 384), ("int8", 256, 256, 384), ("bf16", 256, 256, 384)])
@pytest.mark.parametrize("fewer", [0, 1])
def test_rows_around_the_forward_lines(fmt, line, d, f, fewer):
    counts = (LINES[line][0] - fewer,) + LINES[line][1:]
    assert sum(LINES[line]) == line * len(counts)
    kind = nat.LAUNCH_STREAM if fewer else nat.LAUNCH_DUAL
    assert launches(fmt, counts, d, f) == {kind}
    _forward_case(fmt, counts, d, f)


@pytest.mark.parametrize("case", list(COUNTS))
def test_rows_around_the_tile_heights_backward(case):
    from test_gpu_backward import _close, _gpu_grads, _oracle_grads

    counts = COUNTS[case]
    kind = nat.LAUNCH_128 if case == "below" else nat.LAUNCH_DUAL
    assert launches("int8", counts, 256, 384, backward=True) == {kind}
    w = workload("int8", counts)
    idx, scores = exact_routes(counts, 6)
    dense, lora, x, dy = (wl.dense_weights(w), wl.lora_factors(w), wl.tokens(w),
                          wl.upstream_grad(w))
    _, g = _gpu_grads(build_module(w, dense, lora), x, scores, idx, dy)
    _, ref = _oracle_grads(w, dense, lora, x, scores, idx, dy, torch.arange(w.tokens))
    for name, e in ref.items():
        _close(name, g[name], e)


# Streaming tiles: one, two and four row blocks of 32, each at its edges; 640
# and 384 K columns take the rules of long and of short K, 192 is no multiple
# of a streaming step (128) and keeps the tiles that stage decoded weights.
STREAM_COUNTS = (1, 31, 32, 33, 0, 64, 65, 97, 128, 2, 0, 0)


@pytest.mark.parametrize("rank", [0, 16, 40])
@pytest.mark.parametrize("d,f", [(640, 384), (128, 320), (192, 256)])
@pytest.mark.parametrize("fmt", ["nf4", "int8", "bf16"])
def test_streaming_tiles(fmt, d, f, rank):
    kind = nat.LAUNCH_DUAL if d == 192 else nat.LAUNCH_STREAM  # 38 rows per expert
    assert launches(fmt, STREAM_COUNTS, d) == {kind}
    w = workload(fmt, STREAM_COUNTS, d=d, f=f, r=max(rank, 1))
    idx, scores = exact_routes(STREAM_COUNTS, 7)
    dense, x = wl.dense_weights(w), wl.tokens(w)
    lora = wl.lora_factors(w) if rank else None
    m = build_module(w, dense, lora)
    with torch.no_grad():
        out = m.run_direct_routed(x.cuda(), scores.cuda(), idx.cuda())
    ref = olayer.layer_forward(x, scores, idx, oracle_weights(w, dense), oracle_loras(w, lora),
                               w.experts)
    assert_layer_close(out.cpu(), ref)


# Low-rank columns staged for the up-projection: 64 of each adapter of gate/up
# and 128 of down at four row blocks, all 256 at one; further ones
# are read in the epilogue. Adapters of unequal rank and an absent one too.
@pytest.mark.parametrize("ranks", [(64, 64, 64), (72, 136, 128), (8, 64, 136), (256, 200, 256),
                                   (0, 40, 16), (72, 0, 0)])
@pytest.mark.parametrize("fmt", ["nf4", "bf16"])
def test_streaming_tiles_of_many_ranks(fmt, ranks):
    w = workload(fmt, STREAM_COUNTS, d=256, f=384)
    idx, scores = exact_routes(STREAM_COUNTS, 9)
    dense, x = wl.dense_weights(w), wl.tokens(w)
    lora = mixed_rank_factors(w, dict(zip(("w1", "w3", "w2"), (max(r, 1) for r in ranks))))
    lora = {key: t for (key, t), r in zip(lora.items(), ranks) if r}
    m = build_module(w, dense, lora)
    with torch.no_grad():
        out = m.run_direct_routed(x.cuda(), scores.cuda(), idx.cuda())
    ref = olayer.layer_forward(x, scores, idx, oracle_weights(w, dense), oracle_loras(w, lora),
                               w.experts)
    assert_layer_close(out.cpu(), ref)


@pytest.mark.parametrize("heavy", [0, 900])
@pytest.mark.parametrize("rank", [0, 16])
@pytest.mark.parametrize("d,f", [(640, 384), (256, 640)])
def test_streaming_tiles_of_ingested_nf4(d, f, rank, heavy):
    """fp32 and two-level absmax: every row count of STREAM_COUNTS, K above and
    below 512, rows whose blocks lie in two nested-scale groups (256 blocks are no
    multiple of a row's); with a heavy expert the same tiles are remainders of the
    launch with 256-row tiles where K is above 512. The two give the same bits,
    within the layer bound of the oracle."""
    from test_gpu_codec import _bnb_state

    from mirai_amd import CompressedGroupedExperts

    counts = (*STREAM_COUNTS[:-1], heavy)
    E = len(counts)
    for fmt in (nat.FMT_NF4_F32, nat.FMT_NF4_DQ):
        for K in (d, f):
            kind = nat.LAUNCH_DUAL if heavy and K > 512 else nat.LAUNCH_STREAM
            assert nat.load_library().mx_gemm_launch(fmt, 0, K, sum(counts), E) == kind
    state, dense, shapes = _bnb_state(E, d, f, 90)
    w = workload("nf4", counts, d=d, f=f, r=max(rank, 1))
    lora = wl.lora_factors(w) if rank else None
    idx, scores = exact_routes(counts, 11)
    x, outs = wl.tokens(w), []
    for two_level in (False, True):
        m = CompressedGroupedExperts.from_empty(num_experts=E, quant_format="nf4",
                                                expert_weight_access="fused_kernel")
        m.load_bnb_state_dict(state, shapes, two_level=two_level)
        for key, (a, b) in (lora or {}).items():
            ad = m.attach_expert_lora(tensor_name=key, adapter_name="test", rank=rank, alpha=w.alpha)
            with torch.no_grad():
                ad.lora_a.copy_(a.cuda())
                ad.lora_b.copy_(b.cuda())
        with torch.no_grad():
            outs.append(m.run_direct_routed(x.cuda(), scores.cuda(), idx.cuda()))
    assert torch.equal(outs[0], outs[1])
    ref = olayer.layer_forward(x, scores, idx, dense, oracle_loras(w, lora), E)
    assert_layer_close(outs[0].cpu(), ref)


@pytest.mark.parametrize("fmt", ["nf4", "int8", "bf16"])
def test_a_rows_bits_do_not_depend_on_the_launch(fmt):
    # The same rows of experts 0 .. 10 alone (streaming launch) and beside a
    # heavy expert 11 (the launch with 256-row tiles), and the heavy expert's
    # rows in 300s (256 + 44) and in 100s: tiles of more than 32 rows sum K in one
    # order, smaller ones in theirs in either launch.
    w = workload(fmt, STREAM_COUNTS, d=640, f=768)
    assert launches(fmt, STREAM_COUNTS, 640, 768) == {nat.LAUNCH_STREAM}
    assert launches(fmt, (*STREAM_COUNTS[:-1], 900), 640, 768) == {nat.LAUNCH_DUAL}
    m = build_module(w, wl.dense_weights(w), wl.lora_factors(w))
    x = wl.tokens(w.with_tokens(w.tokens + 900)).cuda()
    idx = torch.full((x.shape[0], 1), 11, dtype=torch.int64)
    idx[:w.tokens] = exact_routes(STREAM_COUNTS, 7)[0]
    idx, ones = idx.cuda(), torch.ones(x.shape[0], 1, device="cuda")

    def run(a, b):
        with torch.no_grad():
            return m.run_direct_routed(x[a:b], ones[a:b], idx[a:b])

    whole = run(0, x.shape[0])
    assert torch.equal(whole[:w.tokens], run(0, w.tokens))
    for step in (100, 300):
        for a in range(w.tokens, x.shape[0], step):
            assert torch.equal(whole[a:a + step], run(a, a + step))


def _blockwise(K):
    """Positions of the columns 64 h + 8 s + j of each 128-block after the order
    16 s + 8 h + j."""
    k = torch.arange(K).view(K // 128, 2, 8, 8)
    return k.permute(0, 2, 1, 3).reshape(K)


@pytest.mark.parametrize("heavy", [0, 300])
@pytest.mark.parametrize("m", [1, 31, 32])
@pytest.mark.parametrize("d,f", [(256, 384), (640, 768), (2048, 640), (2176, 640)])
def test_few_rows_sum_k_blockwise(d, f, m, heavy):
    """NF4 tiles of at most 32 rows and 2048 columns of K sum K as half-waves
    read it (columns 8 s .. + 7 of both 64-blocks of a step together); tiles of
    more rows or columns take 16 columns in a row. So m rows alone give the
    bits that they give beside another 33 rows of their expert once K's
    columns are reordered; every block has one absmax, so reordering does not
    change what the weights stand for. ``heavy`` rows of the other expert bring
    the launch with 256-row tiles (K above 512) or leave it out."""
    g = torch.Generator().manual_seed(31 * d + m)
    w = wl.Workload("blockwise", 13, m, d, f, 2, 1, 1, 1.0, "nf4", torch.bfloat16)
    levels = torch.from_numpy(codec.NF4_LEVELS).to(torch.bfloat16)

    def weight(o, i):
        t = levels[torch.randint(0, 16, (2, o, i), generator=g)]
        t[:, :, ::8] = 1.0  # every 64-block's absmax, before and after the reordering
        return t / 32

    dense = {"w1": weight(f, d), "w3": weight(f, d), "w2": weight(d, f)}
    x = torch.randn((m + 33 + heavy, d), generator=g).to(torch.bfloat16)
    pd = _blockwise(d) if d <= 2048 else torch.arange(d)
    pf = _blockwise(f)
    moved = {"w1": dense["w1"][:, pf][:, :, pd], "w3": dense["w3"][:, pf][:, :, pd],
             "w2": dense["w2"][:, :, pf]}

    def run(weights, x, n):
        idx = torch.zeros(n + heavy, 1, dtype=torch.int64)
        idx[n:] = 1
        rows = torch.cat([x[:n], x[m + 33:]])
        with torch.no_grad():
            return build_module(w, weights, None).run_direct_routed(
                rows.cuda(), torch.ones(n + heavy, 1, device="cuda"), idx.cuda())[:m]

    few = run(dense, x, m)
    assert float(few.float().abs().max()) > 0
    assert torch.equal(few, run(moved, x[:, pd], m + 33))
