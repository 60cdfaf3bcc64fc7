"""GPU parity of the grouped GEMMs' row tiles at their edges.

Experts get exact row counts around the tile heights (32, 64, 128 and 256
rows) at averages on both sides of the rules that choose a launch: 256-row
tiles with 128-row remainders, or 128-row tiles alone. Bounds: the layer bound
of test_gpu_layer.py forward, the per-gradient bounds of test_gpu_backward.py
for training (the oracle rounds at the same points, so only fp32 sums in
another order and their bf16 roundings differ).
"""

import numpy as np
import pytest
import torch

from mirai_amd import workloads as wl
from oracle import layer as olayer

from helpers import assert_layer_close, build_module, oracle_loras, oracle_weights

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


# Averages of 147, 33 (both the launch with 256-row tiles) and 31 (128-row tiles only).
COUNTS = {
    "tall": (1, 127, 128, 129, 255, 256, 257, 20),
    "few": (0, 0, 129, 1, 2, 0, 128, 4),
    "below": (0, 0, 129, 0, 0, 0, 119, 0),
}


@pytest.mark.parametrize("fmt", ["nf4", "int8", "bf16"])
@pytest.mark.parametrize("case", list(COUNTS))
def test_rows_around_the_tile_heights(case, fmt):
    counts = COUNTS[case]
    w = workload(fmt, counts)
    idx, scores = exact_routes(counts, 5)
    dense, lora, x = wl.dense_weights(w), wl.lora_factors(w), wl.tokens(w)
    m = build_module(w, dense, lora)
    with torch.no_grad():
        out = m.run_direct_routed(x.cuda(), scores.cuda(), idx.cuda())
    ref = olayer.layer_forward(x, scores, idx, oracle_weights(w, dense), oracle_loras(w, lora),
                               w.experts)
    assert_layer_close(out.cpu(), ref)


@pytest.mark.parametrize("case", list(COUNTS))
def test_rows_around_the_tile_heights_backward(case):
    from test_gpu_backward import _close, _gpu_grads, _oracle_grads

    counts = COUNTS[case]
    w = workload("int8", counts)
    idx, scores = exact_routes(counts, 6)
    dense, lora, x, dy = (wl.dense_weights(w), wl.lora_factors(w), wl.tokens(w),
                          wl.upstream_grad(w))
    _, g = _gpu_grads(build_module(w, dense, lora), x, scores, idx, dy)
    _, ref = _oracle_grads(w, dense, lora, x, scores, idx, dy, torch.arange(w.tokens))
    for name, e in ref.items():
        _close(name, g[name], e)
